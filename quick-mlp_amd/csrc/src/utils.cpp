#include <qmlp/utils.h>

#include <qmlp/errors.h>
#include <qmlp/fused_network.h>
#include <qmlp/qmlp.h>

#include "qmlp_hip.h"

#include <algorithm>
#include <mutex>
#include <vector>

QUICKMLP_NAMESPACE_BEGIN

namespace {

const char* scalarName(Tensor::Precision p)
{
    if (p == Tensor::FLOAT) return "float";
    if (p == Tensor::DOUBLE) return "double";
    throw std::runtime_error("fractionalPullpush works on float or double tensors");
}

// Kernels on one line share a code object.
const std::vector<std::vector<const char*>> KERNEL_NAMES = {
    {"PullPushDownKernel<$T>", "PullPushDownTreeKernel<$T>"},
    {"PullPushUpKernel<$T>", "PullPushUpTreeKernel<$T>"},
    {"PullPushTailKernel<$T>"},
    {"PullPushGradientUpKernel<$T>", "PullPushGradientUpTreeKernel<$T>"},
    {"PullPushGradientKernel<$T, false>", "PullPushGradientTreeKernel<$T>"},
    {"PullPushGradientKernel<$T, true>"},
    {"PullPushGradientTailKernel<$T, false>"},
    {"PullPushGradientTailKernel<$T, true>"},
    {"PullPushAddKernel<$T, 4>"},
    {"PullPushCopyKernel<$T, 4>"}};
constexpr int SECOND = 16;   // the second kernel of a line
enum KernelIndex { DOWN, UP, TAIL, GRADIENT_UP, GRADIENT, GRADIENT_ADD, GRADIENT_TAIL, GRADIENT_TAIL_ADD, ADD_4, COPY_4,
                   DOWN_TREE = DOWN + SECOND, GRADIENT_UP_TREE = GRADIENT_UP + SECOND, UP_TREE = UP + SECOND, GRADIENT_TREE = GRADIENT + SECOND };

// as in kernels/pullpush.h
constexpr int TAIL_BLOCK = 1024, TILE_W = 32, TILE_H = 8, BLOCK = 256, UP_TILE_W = 14, UP_TILE_H = 14, UP_THREADS = 256;
// What the kernel of the coarse levels keeps in LDS beside them for step A, four rows at least: all of 32 x 32 pixels of 4
// channels of floats with a border.
constexpr size_t TAIL_FILL_BYTES = 24 * 1024;

/** \param wide for images whose planes span 2^32 entries or more, or run backwards (see the header) */
std::string pullpushSource(bool wide)
{
    return (wide ? "#define PULLPUSH_WIDE_PLANES\n" : "") + KernelLoader::MainFile("qmlp/kernels/pullpush.h");
}

std::vector<std::string> kernelNames(size_t line, const std::string& scalar)
{
    std::vector<std::string> names;
    for (std::string name : KERNEL_NAMES[line]) {
        name.replace(name.find("$T"), 2, scalar);
        names.push_back("qmlp::kernel::" + name);
    }
    return names;
}

/** The compiled kernels stay loaded for the life of the process, like the reference's static kernels. */
template <typename T>
KernelFunction& pullpushKernel(KernelIndex index, bool wide = false)
{
    static std::mutex mutex;
    static std::vector<KernelFunction> kernels[2][SECOND];
    std::lock_guard<std::mutex> lock(mutex);
    auto& line = kernels[wide ? 1 : 0][index % SECOND];
    if (line.empty())
        line = QuickMLP::Instance().kernelLoader()->getKernels(kernelNames(index % SECOND, sizeof(T) == 4 ? "float" : "double"), pullpushSource(wide),
                                                               QuickMLP::Instance().getCompileFlags());
    return line.at(index / SECOND);
}

/** PullPushView of kernels/pullpush.h */
template <typename T>
struct View
{
    T* p = nullptr;
    long long b = 0, c = 0;
    unsigned y = 0, x = 0;   // (the bits of a PullPushStride)
};
/** PullPushLevel of kernels/pullpush.h */
template <typename T>
struct Level
{
    int H, W;
    View<T> maskPre, dataPre, maskPost, dataPost, maskSum, gradMaskPost, gradDataPost, gradMaskPre, gradDataPre;
};
template <typename T>
View<T> viewOf(const Tensor& t)
{
    View<T> v;
    v.p = static_cast<T*>(const_cast<void*>(t.rawPtr()));
    const int n = t.ndim();
    v.b = t.stride(0);
    v.c = n == 4 ? t.stride(1) : 0;
    v.y = static_cast<unsigned>(t.stride(n - 2));
    v.x = static_cast<unsigned>(t.stride(n - 1));
    return v;
}
/** Whether an entry of a plane of some of these images has no 32-bit offset from the first. */
bool anyWide(std::initializer_list<const Tensor*> images)
{
    for (const Tensor* t : images) {
        const int n = t->ndim();
        if (t->stride(n - 2) < 0 || t->stride(n - 1) < 0
            || (t->size(n - 2) - 1ll) * t->stride(n - 2) + (t->size(n - 1) - 1ll) * t->stride(n - 1) >= (1ll << 32))
            return true;
    }
    return false;
}

bool isCoarsest(int H, int W) { return H <= 1 || W <= 1; }

/** Hands out the image stacks of a workspace one after the other; rows start at even entries, stacks at multiples of 16. */
template <typename T>
struct Workspace
{
    T* base;
    size_t entries = 0;
    View<T> take(int B, int C, int H, int W)
    {
        View<T> v;
        v.p = base ? base + entries : nullptr;
        v.x = 1;
        v.y = static_cast<unsigned>(roundUp(W, 2));
        v.c = static_cast<long long>(H) * v.y;
        v.b = C * v.c;
        entries += roundUp(static_cast<size_t>(B) * static_cast<size_t>(v.b), size_t(16));
        return v;
    }
};

/** PullPushTail of kernels/pullpush.h */
struct Tail
{
    int numLevels;
    int offsets[31];
};

/** Where the kernel of the coarse levels keeps, in entries, what is read of the level above them and the fills of step A. */
struct TailLds
{
    int topOffset, fillOffset, fillEntries;
};

/** LDS bytes of the kernel that takes over the coarse levels below an (H, W) level: with the gradients, which need more. */
template <typename T>
size_t tailLdsBytes(int C, int H, int W, bool gradients, Tail* tail = nullptr, TailLds* lds = nullptr)
{
    size_t entries = 0;
    int level = 0;
    const size_t top = static_cast<size_t>(C + 1) * (gradients ? 2 : 1) * static_cast<size_t>(H) * roundUp(W, 2);
    const size_t fill = std::max(TAIL_FILL_BYTES / sizeof(T), static_cast<size_t>(C + 1) * 4 * (static_cast<size_t>(W) + 2));
    while (!isCoarsest(H, W)) {
        H /= 2;
        W /= 2;
        ++level;
        if (tail) tail->offsets[level] = static_cast<int>(entries);
        const size_t plane = static_cast<size_t>(H) * roundUp(W, 2);
        const bool coarsest = isCoarsest(H, W);
        entries += plane * (coarsest ? 2 + C : 3 + 2 * C);
        if (gradients) entries += plane * (coarsest ? 1 + C : 2 + 2 * C);
    }
    if (tail) tail->numLevels = level + 1;
    if (lds) *lds = {static_cast<int>(entries), static_cast<int>(entries + top), static_cast<int>(fill)};
    return (entries + top + (gradients ? fill : 0)) * sizeof(T);
}

/**
 * The levels of the pyramid of a (B, C, H, W) image that have kernel launches of their own, finest first, with the views of
 * the low-res ones in the given workspaces (null: only the sizes are wanted, in 'bytes' and 'gradientBytes'). The levels
 * below the last one (their copy behind the forward pass: keptTail) are left to the kernels that keep them in LDS: from there on where all of them fit (1 x 4 float:
 * from 32 x 32 pixels on), as a step inside such a workgroup takes less than the 3 us of a launch.
 */
template <typename T>
std::vector<Level<T>> layout(int B, int C, int H, int W, void* pyramid, void* gradients, T*& keptTail, size_t* bytes = nullptr,
                             size_t* gradientBytes = nullptr)
{
    std::vector<Level<T>> levels(1);
    levels[0] = {};
    levels[0].H = H;
    levels[0].W = W;
    Workspace<T> forward{static_cast<T*>(pyramid)}, adjoint{static_cast<T*>(gradients)};
    const size_t lds = FusedNetwork::MaxSharedMemoryBytes();
    while (!isCoarsest(H, W) && tailLdsBytes<T>(C, H, W, true) > lds) {
        H /= 2;
        W /= 2;
        Level<T> l = {};
        l.H = H;
        l.W = W;
        l.maskPre = forward.take(B, 1, H, W);
        l.dataPre = forward.take(B, C, H, W);
        l.maskSum = forward.take(B, 1, H, W);
        l.gradMaskPost = adjoint.take(B, 1, H, W);
        l.gradDataPost = adjoint.take(B, C, H, W);
        if (isCoarsest(H, W)) {   // its own inpainting: nothing changes from before to after
            l.maskPost = l.maskPre;
            l.dataPost = l.dataPre;
            l.gradMaskPre = l.gradMaskPost;
            l.gradDataPre = l.gradDataPost;
        } else {
            l.maskPost = forward.take(B, 1, H, W);
            l.dataPost = forward.take(B, C, H, W);
            l.gradMaskPre = adjoint.take(B, 1, H, W);
            l.gradDataPre = adjoint.take(B, C, H, W);
        }
        levels.push_back(l);
    }
    keptTail = forward.base ? forward.base + forward.entries : nullptr;
    TailLds tail = {};
    (void)tailLdsBytes<T>(C, H, W, false, nullptr, &tail);
    forward.entries += static_cast<size_t>(B) * tail.topOffset;
    if (bytes) *bytes = forward.entries * sizeof(T);
    if (gradientBytes) *gradientBytes = adjoint.entries * sizeof(T);
    return levels;
}

/** The levels below the last one with launches of its own, one workgroup per image. */
template <typename T>
void launchTail(KernelIndex kernel, bool wide, int B, int C, Level<T> finest, bool gradients, T* kept, stream_t stream)
{
    if (isCoarsest(finest.H, finest.W)) return;
    Tail tail = {}, keptTail = {};
    TailLds places = {}, keptPlaces = {};
    const size_t lds = tailLdsBytes<T>(C, finest.H, finest.W, gradients, &tail, &places);
    (void)tailLdsBytes<T>(C, finest.H, finest.W, false, &keptTail, &keptPlaces);
    int keptEntries = keptPlaces.topOffset;   // the levels alone
    std::vector<void*> args = {&finest, &C, &tail, &kept, &keptEntries};
    if (gradients) args.push_back(&keptTail);
    args.push_back(&places.topOffset);
    if (gradients) args.insert(args.end(), {&places.fillOffset, &places.fillEntries});
    pullpushKernel<T>(kernel, wide).launch(static_cast<unsigned>(B), TAIL_BLOCK, static_cast<unsigned>(lds), stream, args.data());
}

/** Whether the pixels (y, 2k) and (y, 2k + 1) of all images of a level can be moved as one aligned pair. */
template <typename T>
bool movesPairs(const Level<T>& level, bool padded)
{
    for (const View<T>* v : {&level.maskPre, &level.dataPre, &level.maskPost, &level.dataPost, &level.gradMaskPost, &level.gradDataPost,
                             &level.gradMaskPre, &level.gradDataPre})
        if (v->p && !(v->x == 1 && v->y % 2 == 0 && v->b % 2 == 0 && v->c % 2 == 0 && reinterpret_cast<uintptr_t>(v->p) % (2 * sizeof(T)) == 0))
            return false;
    return padded || level.W % 2 == 0;   // the rows of the workspaces end at even entries, the caller's where they end
}

/** One launch for one level: a workgroup per tile of 32 x 8 items, for step A of 14 x 14. */
template <typename T>
void launchLevel(KernelIndex kernel, bool wide, int B, int C, int height, int width, const std::vector<Level<T>>& levels, int l, stream_t stream)
{
    Level<T> high = levels[l], low = levels[l + 1];
    int pairs = movesPairs(high, l > 0) ? 1 : 0;
    const bool up = kernel == GRADIENT_UP;
    const long long grid = static_cast<long long>(B) * divUp(height, up ? UP_TILE_H : TILE_H) * divUp(width, up ? UP_TILE_W : TILE_W);
    void* args[] = {&high, &low, &C, &pairs};
    pullpushKernel<T>(kernel, wide).launch(static_cast<unsigned>(grid), up ? UP_THREADS : BLOCK, 0, stream, args);
}

// The finest levels that trees take, counted from the image. Forward and adjoint of one image of 4 channels of floats, with steps B, A and the
// way up from level 1 | 2 | 3 on in trees: 512 x 512 117 | 128 | 145 us, 1024 x 1024 164 | 169 | 182, 777 x 1001 247 | 189 | 188, 2048 x 2048
// 374 | 353 | 357, 4096 x 4096 1250 | 1081 | 1025; 8 images of 3 x 256 x 256 126 | 122 | 121. A large level with a launch of its own is better
// off (1024 x 1024 pixels, step B 18 us, within a tree 27), a small one costs 5 to 11 us, and odd sizes, whose tiles need borders, suffer
// most from large trees: level 2 never loses much.
constexpr int DOWN_TREE_FINEST = 1, UP_TREE_FINEST = 2, GRADIENT_UP_TREE_FINEST = 2, GRADIENT_TREE_FINEST = 2;

constexpr size_t TREE_LDS_BYTES = 72 * 1024;
constexpr int GRADIENT_UP_TREE_LEVELS = 3;   // a border grows by a pixel per level
/** PullPushTree of kernels/pullpush.h */
template <typename T>
struct Tree
{
    static constexpr int LEVELS = 6, BORDER = 5;
    int count, tile;
    Level<T> levels[LEVELS];
};

/**
 * The steps from the level below levels[from] up to levels[to], several levels per launch. A launch for one of these levels
 * takes 5 to 11 us whatever its size; of a tree a step takes 2.
 */
template <typename T>
void launchTrees(KernelIndex kernel, int B, int C, const std::vector<Level<T>>& levels, int from, int to, stream_t stream)
{
    while (from >= to) {
        Tree<T> tree = {};
        const int finest = std::max(to, from + 1 - (Tree<T>::LEVELS - 1));
        tree.count = from + 1 - finest + 1;
        for (int k = 0; k < tree.count; ++k) tree.levels[k] = levels[finest + k];
        auto ldsBytes = [&] {
            size_t entries = 0;
            for (int k = 1; k < tree.count - 1; ++k) entries += static_cast<size_t>(C + 1) * ((tree.tile >> k) + Tree<T>::BORDER) * ((tree.tile >> k) + Tree<T>::BORDER);
            return entries * sizeof(T);
        };
        auto workgroups = [&] { return static_cast<long long>(B) * divUp(levels[finest].H, tree.tile) * divUp(levels[finest].W, tree.tile); };
        // a workgroup on every compute unit, and room for two
        tree.tile = 64;
        while (tree.tile > 16 && (workgroups() < KernelFunction::computeUnits() || ldsBytes() > TREE_LDS_BYTES)) tree.tile /= 2;
        void* args[] = {&tree, &C};
        pullpushKernel<T>(kernel).launch(static_cast<unsigned>(workgroups()), TAIL_BLOCK, static_cast<unsigned>(ldsBytes()), stream, args);
        from = finest - 1;
    }
}

/**
 * The steps from levels[from] down to levels[to], several levels per launch.
 * \param border pixels that a region of a level grows by on its way to the next finer one (2 n + border)
 */
template <typename T>
void launchTreesDown(KernelIndex kernel, int B, int C, const std::vector<Level<T>>& levels, int from, int to, int most, int border, stream_t stream)
{
    while (from < to) {
        Tree<T> tree = {};
        const bool fills = kernel == GRADIENT_UP_TREE;
        int last = std::min(to - from, most - 1);
        auto ldsEntries = [&] {
            size_t entries = 0;
            for (int k = 1; k < last; ++k) {
                const size_t size = (tree.tile >> k) + border * ((1 << (last - k)) - 1);
                entries += (C + 1) * size * size;
            }
            return entries;
        };
        auto fillBytes = [&] {   // at least four rows
            const size_t size = (tree.tile >> 1) + border * ((1 << (last - 1)) - 1);
            return fills ? std::max(TAIL_FILL_BYTES, static_cast<size_t>(C + 1) * 4 * (2 * size + 2) * sizeof(T)) : size_t(0);
        };
        auto workgroups = [&] {
            const int tile = tree.tile >> last;
            return static_cast<long long>(B) * divUp(levels[from + last].H, tile) * divUp(levels[from + last].W, tile);
        };
        // a workgroup on every compute unit and room for two; of many channels fewer levels
        for (;; --last) {
            const int smallest = 1 << (last + 1);   // 2 x 2 pixels of the coarsest level
            tree.tile = 64;
            while (tree.tile > smallest && (workgroups() < KernelFunction::computeUnits() || ldsEntries() * sizeof(T) + fillBytes() > TREE_LDS_BYTES)) tree.tile /= 2;
            if (last == 1 || ldsEntries() * sizeof(T) + fillBytes() <= TREE_LDS_BYTES) break;
        }
        const int coarsest = from + last;
        tree.count = last + 1;
        for (int k = 0; k <= last; ++k) tree.levels[k] = levels[from + k];
        int fillOffset = static_cast<int>(ldsEntries()), fillEntries = static_cast<int>(fillBytes() / sizeof(T));
        void* args[] = {&tree, &C, &fillOffset, &fillEntries};   // (the last two for step A)
        pullpushKernel<T>(kernel).launch(static_cast<unsigned>(workgroups()), TAIL_BLOCK, static_cast<unsigned>(ldsEntries() * sizeof(T) + fillBytes()), stream, args);
        from = coarsest;
    }
}

/** The pyramid down to the coarsest level and the inpainted levels up to levels[1]; with 'finest' up to levels[0]. */
template <typename T>
void runForward(const std::vector<Level<T>>& levels, bool wide, int B, int C, bool finest, T* keptTail, stream_t stream)
{
    const int last = static_cast<int>(levels.size()) - 1;
    const int single = wide ? last : std::min(last, DOWN_TREE_FINEST);   // levels of a launch each
    for (int k = 0; k < single; ++k) launchLevel(DOWN, wide, B, C, levels[k + 1].H, levels[k + 1].W, levels, k, stream);
    launchTreesDown(DOWN_TREE, B, C, levels, single, last, Tree<T>::LEVELS, 1, stream);
    launchTail(TAIL, wide, B, C, levels[last], false, keptTail, stream);
    int l = last - 1;
    if (!wide) {
        launchTrees(UP_TREE, B, C, levels, l, UP_TREE_FINEST, stream);
        l = std::min(l, UP_TREE_FINEST - 1);
    }
    for (; l >= (finest ? 0 : 1); --l)
        launchLevel(UP, wide, B, C, divUp(levels[l].H, 2), divUp(levels[l].W, 2), levels, l, stream);
}

template <typename T>
void runAdjoint(const std::vector<Level<T>>& levels, bool wide, int B, int C, bool accumulate, T* keptTail, stream_t stream)
{
    const int last = static_cast<int>(levels.size()) - 1;
    const int single = wide ? last : std::min(last, GRADIENT_UP_TREE_FINEST);
    for (int k = 0; k < single; ++k) launchLevel(GRADIENT_UP, wide, B, C, levels[k + 1].H, levels[k + 1].W, levels, k, stream);
    launchTreesDown(GRADIENT_UP_TREE, B, C, levels, single, last, GRADIENT_UP_TREE_LEVELS, 2, stream);
    launchTail(last == 0 && accumulate ? GRADIENT_TAIL_ADD : GRADIENT_TAIL, wide, B, C, levels[last], true, keptTail, stream);
    int l = last - 1;
    if (!wide) {
        launchTrees(GRADIENT_TREE, B, C, levels, l, GRADIENT_TREE_FINEST, stream);
        l = std::min(l, GRADIENT_TREE_FINEST - 1);
    }
    for (; l >= 0; --l)
        launchLevel(l == 0 && accumulate ? GRADIENT_ADD : GRADIENT, wide, B, C, divUp(levels[l].H, 2), divUp(levels[l].W, 2), levels, l, stream);
}

/** dst = src or dst += src for image stacks of any strides; without src: zero. */
template <typename T>
void elementwise(KernelIndex kernel, const Tensor& dst, const Tensor* src, stream_t stream)
{
    auto accessor = [](const Tensor& t) {   // a mask is an image of one channel
        kernel::TensorAccessor<T, 4> a;
        const bool mask = t.ndim() == 3;
        a.data_ = static_cast<T*>(const_cast<void*>(t.rawPtr()));
        for (int d = 0; d < 4; ++d) {
            a.sizes_[d] = mask && d == 1 ? 1 : t.size(mask && d > 1 ? d - 1 : d);
            a.strides_[d] = mask && d == 1 ? 0 : t.stride(mask && d > 1 ? d - 1 : d);
        }
        return a;
    };
    long long numel = dst.numel();
    auto d = accessor(dst);
    kernel::TensorAccessor<T, 4> s = {};
    if (src) s = accessor(*src);
    void* args[] = {&numel, &d, &s};
    pullpushKernel<T>(kernel).launch(static_cast<unsigned>(std::min<long long>(divUp<long long>(numel, BLOCK), 1 << 16)), BLOCK, 0, stream, args);
}

template <typename T>
void forward(const Tensor& mask, const Tensor& data, Tensor& output, void* pyramid, stream_t stream)
{
    const int B = data.size(0), C = data.size(1), H = data.size(2), W = data.size(3);
    if (isCoarsest(H, W)) {   // nothing coarser to fill from
        elementwise<T>(COPY_4, output, &data, stream);
        return;
    }
    T* keptTail = nullptr;
    auto levels = layout<T>(B, C, H, W, pyramid, nullptr, keptTail);
    levels[0].maskPre = viewOf<T>(mask);
    levels[0].dataPre = viewOf<T>(data);
    levels[0].dataPost = viewOf<T>(output);
    runForward(levels, anyWide({&mask, &data, &output}), B, C, true, keptTail, stream);
}

template <typename T>
void adjoint(const Tensor& mask, const Tensor& data, const Tensor& adjOutput, Tensor& adjMask, Tensor& adjData, bool accumulate,
             void* pyramid, bool pyramidReady, void* gradients, stream_t stream)
{
    const int B = data.size(0), C = data.size(1), H = data.size(2), W = data.size(3);
    if (isCoarsest(H, W)) {
        elementwise<T>(accumulate ? ADD_4 : COPY_4, adjData, &adjOutput, stream);
        if (!accumulate) elementwise<T>(COPY_4, adjMask, nullptr, stream);   // the mask of a row or a column has no influence
        return;
    }
    T* keptTail = nullptr;
    auto levels = layout<T>(B, C, H, W, pyramid, gradients, keptTail);
    levels[0].maskPre = viewOf<T>(mask);
    levels[0].dataPre = viewOf<T>(data);
    const bool wide = anyWide({&mask, &data, &adjOutput, &adjMask, &adjData});
    if (!pyramidReady) runForward(levels, wide, B, C, false, keptTail, stream);
    levels[0].gradDataPost = viewOf<T>(adjOutput);
    levels[0].gradMaskPre = viewOf<T>(adjMask);
    levels[0].gradDataPre = viewOf<T>(adjData);
    runAdjoint(levels, wide, B, C, accumulate, keptTail, stream);
}

void checkShapes(const Tensor& mask, const Tensor& data)
{
    CHECK_DIM(mask, 3);
    CHECK_DIM(data, 4);
    CHECK_SIZE(mask, 0, data.size(0));
    CHECK_SIZE(mask, 1, data.size(2));
    CHECK_SIZE(mask, 2, data.size(3));
    CHECK_DTYPE(mask, data.precision());
    CHECK_ERROR(data.precision() == Tensor::FLOAT || data.precision() == Tensor::DOUBLE,
                "fractionalPullpush works on float or double tensors");
    CHECK_ERROR(data.size(1) < 16, "fractionalPullpush only supports up to 16 channels, but got ", data.size(1));
}

void checkLike(const Tensor& x, const Tensor& like, const char* what)
{
    CHECK_ERROR(x.ndim() == like.ndim(), what, " has the wrong number of dimensions");
    for (int d = 0; d < like.ndim(); ++d) CHECK_ERROR(x.size(d) == like.size(d), what, " has the wrong size at dimension ", d);
    CHECK_DTYPE(x, like.precision());
}

/** Device memory of one call, in the order of the stream. */
struct CallMemory
{
    void* p = nullptr;
    stream_t stream;
    CallMemory(size_t bytes, stream_t s) : stream(s) { if (bytes > 0) QMLP_HIP_CALL(qmlp_hip_malloc_async(&p, bytes, s)); }
    ~CallMemory() { if (p) qmlp_hip_free_async(p, stream); }
    CallMemory(const CallMemory&) = delete;
    CallMemory& operator=(const CallMemory&) = delete;
};

} // namespace

void Utils::precompile(Tensor::Precision precision)
{
    const std::string t = scalarName(precision);
    auto kl = QuickMLP::Instance().kernelLoader();
    const int flags = QuickMLP::Instance().getCompileFlags() | KernelLoader::CompileOnly;
    for (size_t i = 0; i < KERNEL_NAMES.size(); ++i) kl->getKernels(kernelNames(i, t), pullpushSource(false), flags);
}

void Utils::pullpushMemory(const Tensor& data, size_t& pyramidBytes, size_t& gradientBytes)
{
    CHECK_DIM(data, 4);
    pyramidBytes = gradientBytes = 0;
    if (data.numel() == 0) return;
    const int B = data.size(0), C = data.size(1), H = data.size(2), W = data.size(3);
    if (data.precision() == Tensor::FLOAT) {
        float* keptTail = nullptr;
        layout<float>(B, C, H, W, nullptr, nullptr, keptTail, &pyramidBytes, &gradientBytes);
    } else {
        double* keptTail = nullptr;
        layout<double>(B, C, H, W, nullptr, nullptr, keptTail, &pyramidBytes, &gradientBytes);
    }
}

void Utils::fractionalPullpush(const Tensor& mask, const Tensor& data, Tensor& output, stream_t stream)
{
    checkShapes(mask, data);
    checkLike(output, data, "output");
    size_t pyramidBytes = 0, gradientBytes = 0;
    pullpushMemory(data, pyramidBytes, gradientBytes);
    CallMemory pyramid(pyramidBytes, stream);
    fractionalPullpush(mask, data, output, pyramid.p, stream);
}

void Utils::fractionalPullpush(const Tensor& mask, const Tensor& data, Tensor& output, void* pyramid, stream_t stream)
{
    checkShapes(mask, data);
    checkLike(output, data, "output");
    if (data.numel() == 0) return;
    if (data.precision() == Tensor::FLOAT) forward<float>(mask, data, output, pyramid, stream);
    else forward<double>(mask, data, output, pyramid, stream);
}

void Utils::adjointFractionalPullpush(const Tensor& mask, const Tensor& data, const Tensor& adjOutput, Tensor& adjMask,
                                      Tensor& adjData, stream_t stream)
{
    checkShapes(mask, data);
    checkLike(adjOutput, data, "adjOutput");
    checkLike(adjData, data, "adjData");
    checkLike(adjMask, mask, "adjMask");
    size_t pyramidBytes = 0, gradientBytes = 0;
    pullpushMemory(data, pyramidBytes, gradientBytes);
    CallMemory pyramid(pyramidBytes, stream), gradients(gradientBytes, stream);
    adjointFractionalPullpush(mask, data, adjOutput, adjMask, adjData, true, pyramid.p, false, gradients.p, stream);
}

void Utils::adjointFractionalPullpush(const Tensor& mask, const Tensor& data, const Tensor& adjOutput, Tensor& adjMask, Tensor& adjData,
                                      bool accumulate, void* pyramid, bool pyramidReady, void* gradients, stream_t stream)
{
    checkShapes(mask, data);
    checkLike(adjOutput, data, "adjOutput");
    checkLike(adjData, data, "adjData");
    checkLike(adjMask, mask, "adjMask");
    if (data.numel() == 0) {
        if (accumulate || mask.numel() == 0) return;   // images of no channels: their mask has no influence
        if (mask.precision() == Tensor::FLOAT) elementwise<float>(COPY_4, adjMask, nullptr, stream);
        else elementwise<double>(COPY_4, adjMask, nullptr, stream);
        return;
    }
    if (data.precision() == Tensor::FLOAT)
        adjoint<float>(mask, data, adjOutput, adjMask, adjData, accumulate, pyramid, pyramidReady, gradients, stream);
    else
        adjoint<double>(mask, data, adjOutput, adjMask, adjData, accumulate, pyramid, pyramidReady, gradients, stream);
}

QUICKMLP_NAMESPACE_END
