#pragma once
// Differentiable pull-push inpainting on an image pyramid (fractional masks).
//
//   down:  low-res pixel = mask-weighted mean of its window of high-res pixels, low-res mask =
//          maximum of the window (windows as in adaptive pooling, [floor(i*H/oH), ceil((i+1)*H/oH))
//          with oH = H/2: rows 2i, 2i+1 of an even height, 2i .. 2i+2 of an odd one, where
//          neighbouring windows share a row)
//   up:    high-res pixel = m*data + (1-m)*(bilinear mix of the 4 nearest low-res pixels,
//          weights 9/16, 3/16, 3/16, 1/16, renormalised by the low-res masks)
//
// The coarsest level (a row or a column of pixels) is its own inpainting. Every step is bound by HBM traffic
// on the fine levels and by latency on the coarse ones (a launch for a level of 64 x 64 pixels takes 5 to 10 us). Hence one
// launch per level while a level is large, one for several levels below, and one with a workgroup per image for the coarsest, which
// fit into LDS (4 channels of float: below 32 x 32).
//
// The unit of work is the quad: the 2 x 2 high-res pixels of one low-res pixel. Its pixels are moved in pairs
// (8 or 16 bytes per lane) and share their 3 x 3 low-res neighbours (9 loads instead of 16).
//
// The adjoint walks the pyramid twice and keeps no per-pixel intermediates:
//   A, fine to coarse: the gradient of the inpainted low-res level from that of the inpainted high-res level
//      (adjoint of up with respect to the low-res level; the terms that high-res pixels pass down stay in LDS)
//   B, coarse to fine: the gradient of a level before inpainting = adjoint of up with respect to the high-res
//      level + adjoint of down, both formed per quad by gathering, without atomics
// so the finest level of C channels moves C+1 + (2C+2)/4 planes in A and 3C+2 + (3C+4)/4 in B (a coarser one, whose mask has a
// gradient, one more in each), C+1 + (C+2)/4 in down and 2C+1 + (C+1)/4 in up.
// 1 x 4 x 2048 x 2048 floats, finest level: down 21, up 36, A 45, B 70 us (5.2, 4.8, 2.8, 4.3 TB/s of the planes above; a
// large copy reaches 4.8), 172 of the 352 us of a forward and adjoint call; 1024 x 1024 takes 50, the levels below it, which take several
// steps per launch (the trees below) or live in one workgroup's LDS, the rest: a step is a chain of 1.5 to 2 us. (A launch per level: 446 us.
// Coarse levels formed again by the adjoint: 10 us more; four passes per level through memory, atomics for odd sizes, and memory allocated and
// released by every call: 9.4 ms.) A and B are held to 128 registers for floats, four wavefronts per SIMD.
//
// Follows src_cpp/include/qmlp/kernels/pullpush.cuh:22-303 of the reference. Differences on
// purpose: no per-thread channel arrays, no atomics (the reference scatters the adjoint of up with atomics and adds
// the adjoint of down without them, a race between overlapping windows), window limits in integers (the reference's
// fp32 quotient is exact only while the products stay below 2^24), the pyramid of the forward pass is kept for the
// adjoint pass.

#include <qmlp/kernels/common.h>

QUICKMLP_KERNEL_NAMESPACE_BEGIN

// The entries of a plane lie within 2^32 of each other and behind the first: the same plane for a whole workgroup (scalar
// registers) and one 32-bit offset per lane. For other images the host (src/utils.cpp) defines PULLPUSH_WIDE_PLANES.
#ifdef PULLPUSH_WIDE_PLANES
typedef int PullPushStride;
typedef long long PullPushOffset;
#else
typedef unsigned PullPushStride;
typedef unsigned PullPushOffset;
#endif

/** A stack of images: entry (b, c, y, x); p == nullptr: absent. */
template <typename T>
struct PullPushView
{
    T* p;
    long long b, c;   // strides in entries
    PullPushStride y, x;
};

/** One level of the pyramid. The views of the coarsest level alias (post = pre, its gradients too). */
template <typename T>
struct PullPushLevel
{
    int H, W;
    PullPushView<T> maskPre, dataPre;     // before inpainting
    PullPushView<T> maskPost, dataPost;   // inpainted; the mask of the finest level is absent
    PullPushView<T> maskSum;              // sum of the masks of the window of this pixel in the finer level
    PullPushView<T> gradMaskPost, gradDataPost, gradMaskPre, gradDataPre;   // adjoint; the first is absent on the finest level (zero)
};

constexpr int PULLPUSH_TAIL_BLOCK = 1024;
/** The levels that the kernels for all coarse levels keep in LDS: levels[0] is the one above them. */
struct PullPushTail
{
    int numLevels;
    int offsets[31];   // of level k in entries
};
/** Consecutive levels, finest first, that one launch walks through, with the tile of the finest that a workgroup takes. */
constexpr int PULLPUSH_TREE_LEVELS = 6;
template <typename T>
struct PullPushTree
{
    int count, tile;
    PullPushLevel<T> levels[PULLPUSH_TREE_LEVELS];
};
/** Channels that are in flight together: their loads are issued before the first of them is used. */
template <typename T> constexpr int pullpushChunk() { return sizeof(T) == 4 ? 4 : 2; }

namespace pullpush
{
template <typename T> struct Pair;
template <> struct Pair<float> { typedef float type __attribute__((ext_vector_type(2))); };
template <> struct Pair<double> { typedef double type __attribute__((ext_vector_type(2))); };

template <typename T>
__device__ __forceinline__ T* at(const PullPushView<T>& v, int b, int c, int y, int x)
{
    return v.p + (b * v.b + c * v.c) + (static_cast<PullPushOffset>(y) * v.y + static_cast<PullPushOffset>(x) * v.x);
}

/**
 * Two neighbours in a row. PAIRS: the host found the images aligned for it, they are moved as one, and what lies behind
 * an odd row is padding that belongs to the image. Otherwise the second is only touched if it exists (v[1] stays as it is).
 */
template <bool PAIRS, typename T>
__device__ __forceinline__ void loadPair(const T* p, PullPushStride stride, bool second, T (&v)[2])
{
    if constexpr (PAIRS) {
        const typename Pair<T>::type w = *reinterpret_cast<const typename Pair<T>::type*>(p);
        v[0] = w[0];
        v[1] = w[1];
    } else {
        v[0] = p[0];
        if (second) v[1] = p[stride];
    }
}
template <bool PAIRS, typename T>
__device__ __forceinline__ void storePair(T* p, PullPushStride stride, bool second, const T (&v)[2])
{
    if constexpr (PAIRS) {
        typename Pair<T>::type w;
        w[0] = v[0];
        w[1] = v[1];
        *reinterpret_cast<typename Pair<T>::type*>(p) = w;
    } else {
        p[0] = v[0];
        if (second) p[stride] = v[1];
    }
}

/** d / n for a sum of masks n, and zero where nothing is known, whatever d is then (NaN or infinite data times a mask of zero). */
template <typename T>
__device__ __forceinline__ T quotient(T d, T n)
{
    return n > 0 ? d / n : T(0);
}

/**
 * The same as a multiplication, for several quotients by one sum in the adjoint, whose terms are products of several factors
 * anyway. Scaled, as the reciprocal of a sum below 3e-39 has no float.
 */
template <typename T>
struct Reciprocal
{
    static constexpr T SCALE = sizeof(T) == 4 ? T(1 << 22) : T(1ll << 52);
    T inverse;
    __device__ __forceinline__ Reciprocal() : inverse(0) {}
    __device__ __forceinline__ explicit Reciprocal(T n) : inverse(n > 0 ? T(1) / (n * SCALE) : T(0)) {}
    __device__ __forceinline__ T operator()(T d) const { return inverse > 0 ? d * inverse * SCALE : T(0); }
};

/** down for the low-res pixel (a, e). */
template <bool PAIRS, typename T>
__device__ __forceinline__ void downPixel(const PullPushLevel<T>& high, const PullPushLevel<T>& low, int C, int b, int a, int e)
{
    const int rows = 2 + (high.H & 1), columns = 2 + (high.W & 1);
    T m[3][3];
    T sum = 0, most = 0;
    auto window = [&](const PullPushView<T>& v, int c, T (&out)[3][3]) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            out[i][0] = out[i][1] = out[i][2] = T(0);
            if (i >= rows) continue;
            const T* p = at(v, b, c, 2 * a + i, 2 * e);
            T pair[2];
            loadPair<PAIRS>(p, v.x, true, pair);
            out[i][0] = pair[0];
            out[i][1] = pair[1];
            if (columns > 2) out[i][2] = p[static_cast<PullPushOffset>(2) * v.x];
        }
    };
    window(high.maskPre, 0, m);
    // column by column, as the sums of the whole pyramid have always been taken
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            sum += m[i][j];             // (entries beyond the window are zero)
            most = max(most, m[i][j]);
        }
    *at(low.maskPre, b, 0, a, e) = most;
    *at(low.maskSum, b, 0, a, e) = sum;
    constexpr int CHUNK = pullpushChunk<T>();
    for (int c0 = 0; c0 < C; c0 += CHUNK) {
        T d[CHUNK];
#pragma unroll
        for (int k = 0; k < CHUNK; ++k) {
            T v[3][3];
            d[k] = T(0);
            if (c0 + k >= C) continue;
            window(high.dataPre, c0 + k, v);
#pragma unroll
            for (int j = 0; j < 3; ++j)
#pragma unroll
                for (int i = 0; i < 3; ++i)
                    if (i < rows && j < columns) d[k] += m[i][j] * v[i][j];
        }
#pragma unroll
        for (int k = 0; k < CHUNK; ++k)
            if (c0 + k < C) *at(low.dataPre, b, c0 + k, a, e) = quotient(d[k], sum);
    }
}

/**
 * The low-res neighbourhood of a quad (a, e): rows a-1 .. a+1, columns e-1 .. e+1; validity as factors of the bilinear weights.
 * \tparam INTERIOR all of it lies in the image
 */
template <bool INTERIOR = false>
struct Neighbourhood
{
    float rowIn[3], columnIn[3];
    __device__ __forceinline__ Neighbourhood(int a, int e, int oH, int oW)
    {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const int y = a - 1 + k, x = e - 1 + k;
            rowIn[k] = INTERIOR || (y >= 0 && y < oH) ? 1.f : 0.f;
            columnIn[k] = INTERIOR || (x >= 0 && x < oW) ? 1.f : 0.f;
        }
    }
    /** Weights of the own cell, the neighbour in the other row, in the other column, and the diagonal one, for pixel (di, dj) of the quad. */
    __device__ __forceinline__ void weights(int di, int dj, float (&w)[4]) const
    {
        const float own = 0.75f * rowIn[1], other = 0.25f * rowIn[2 * di];
        const float ownColumn = 0.75f * columnIn[1], otherColumn = 0.25f * columnIn[2 * dj];
        w[0] = own * ownColumn;
        w[1] = other * ownColumn;
        w[2] = own * otherColumn;
        w[3] = other * otherColumn;
    }
    template <typename T>
    __device__ __forceinline__ static void pick(const T (&v)[3][3], int di, int dj, T (&out)[4])
    {
        out[0] = v[1][1];
        out[1] = v[2 * di][1];
        out[2] = v[1][2 * dj];
        out[3] = v[2 * di][2 * dj];
    }
};

/** Masks and weights of the low-res neighbours of the four pixels of a quad: wm[k] = weight * mask, their sum n. */
template <typename T>
struct QuadMix
{
    T wm[2][2][4], n[2][2], weight[2][2];
    Reciprocal<T> inverse[2][2];
    template <typename Neighbours>
    __device__ __forceinline__ QuadMix(const Neighbours& nb, const T (&maskLow)[3][3])
    {
#pragma unroll
        for (int di = 0; di < 2; ++di)
#pragma unroll
            for (int dj = 0; dj < 2; ++dj) {
                float w[4];
                T ml[4];
                nb.weights(di, dj, w);
                nb.pick(maskLow, di, dj, ml);
                weight[di][dj] = 0;
                n[di][dj] = 0;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    wm[di][dj][k] = w[k] * ml[k];
                    weight[di][dj] += w[k];
                    n[di][dj] += wm[di][dj][k];
                }
                inverse[di][dj] = Reciprocal<T>(n[di][dj]);
            }
    }
    /** The weighted sum of a channel for pixel (di, dj). */
    __device__ __forceinline__ T sum(const T (&low)[3][3], int di, int dj) const
    {
        T v[4];
        Neighbourhood<>::pick(low, di, dj, v);
        T d = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) d += wm[di][dj][k] * v[k];
        return d;
    }
};

/**
 * The low-res pixels that the quads of a workgroup interpolate from, in LDS: QW x QH quads from (a0, e0) on and one more on every
 * side, clamped into the image. A thread that loads the nine of its quad itself asks the memory pipeline for 45 values (4 channels), at 16
 * cycles per instruction of a wavefront, and holds their addresses: 2048 x 2048 floats, the way up 39 us in 222 registers, from LDS 36 in
 * 96, step B 73 and 70.
 */
template <typename T, int QW, int QH>
struct LowTile
{
    static constexpr int PITCH = QW + 2, ENTRIES = PITCH * (QH + 2), PLANES = pullpushChunk<T>() + 1;
    typedef T Memory[PLANES][ENTRIES];

    /** All threads of the workgroup; up to CHUNK channels from c0 on, and with the first of them the mask into the last plane. */
    __device__ __forceinline__ static void stage(Memory& s, const PullPushLevel<T>& low, int C, int b, int c0, int a0, int e0)
    {
#pragma unroll 2
        for (int i = threadIdx.x; i < ENTRIES; i += blockDim.x) {
            const int a = min(max(a0 - 1 + i / PITCH, 0), low.H - 1), e = min(max(e0 - 1 + i % PITCH, 0), low.W - 1);
            T v[PLANES];
#pragma unroll
            for (int k = 0; k + 1 < PLANES; ++k)
                if (c0 + k < C) v[k] = *at(low.dataPost, b, c0 + k, a, e);
            if (c0 == 0) v[PLANES - 1] = *at(low.maskPost, b, 0, a, e);
#pragma unroll
            for (int k = 0; k + 1 < PLANES; ++k)
                if (c0 + k < C) s[k][i] = v[k];
            if (c0 == 0) s[PLANES - 1][i] = v[PLANES - 1];
        }
    }
    /** The neighbours of quad (la, le) of the tile. */
    __device__ __forceinline__ static void load(const T (&plane)[ENTRIES], int la, int le, T (&out)[3][3])
    {
        const T* p = plane + (la * PITCH + le);
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) out[i][j] = p[i * PITCH + j];
    }
};

/** up for the QW x QH quads from (a0, e0) on, a thread each (all threads of the workgroup call this). */
template <bool PAIRS, int QW, int QH, typename T>
__device__ __forceinline__ void upQuads(const PullPushLevel<T>& high, const PullPushLevel<T>& low, int C, int b, int a0, int e0,
                                        typename LowTile<T, QW, QH>::Memory& sLow)
{
    typedef LowTile<T, QW, QH> Low;
    constexpr int CHUNK = pullpushChunk<T>();
    const int la = threadIdx.x / QW, le = threadIdx.x % QW, a = a0 + la, e = e0 + le;
    const bool mine = 2 * a < high.H && 2 * e < high.W, second = 2 * e + 1 < high.W;
    T m[2][2];
    for (int c0 = 0; c0 < C; c0 += CHUNK) {
        T v[CHUNK][2][2];
#pragma unroll
        for (int di = 0; di < 2; ++di) {
            if (!mine || 2 * a + di >= high.H) continue;
            if (c0 == 0) {
                m[di][0] = m[di][1] = T(0);
                loadPair<PAIRS>(at(high.maskPre, b, 0, 2 * a + di, 2 * e), high.maskPre.x, second, m[di]);
            }
#pragma unroll
            for (int k = 0; k < CHUNK; ++k)
                if (c0 + k < C) loadPair<PAIRS>(at(high.dataPre, b, c0 + k, 2 * a + di, 2 * e), high.dataPre.x, second, v[k][di]);
        }
        if (c0 > 0) __syncthreads();   // the channels in front of these have been read
        Low::stage(sLow, low, C, b, c0, a0, e0);
        __syncthreads();
        if (!mine) continue;
        const Neighbourhood<> nb(a, e, low.H, low.W);
        T lowMask[3][3];
        Low::load(sLow[Low::PLANES - 1], la, le, lowMask);
        const QuadMix<T> mix(nb, lowMask);
#pragma unroll
        for (int di = 0; di < 2; ++di) {
            if (2 * a + di >= high.H || c0 > 0 || !high.maskPost.p) continue;
            T out[2];
#pragma unroll
            for (int dj = 0; dj < 2; ++dj)
                out[dj] = m[di][dj] + (mix.n[di][dj] > 0 ? (1 - m[di][dj]) * (mix.n[di][dj] / mix.weight[di][dj]) : T(0));
            storePair<PAIRS>(at(high.maskPost, b, 0, 2 * a + di, 2 * e), high.maskPost.x, second, out);
        }
#pragma unroll
        for (int k = 0; k < CHUNK; ++k) {
            if (c0 + k >= C) continue;
            T lowData[3][3];
            Low::load(sLow[k], la, le, lowData);
#pragma unroll
            for (int di = 0; di < 2; ++di) {
                if (2 * a + di >= high.H) continue;
                T out[2];
#pragma unroll
                for (int dj = 0; dj < 2; ++dj)
                    out[dj] = m[di][dj] * v[k][di][dj] + (1 - m[di][dj]) * quotient(mix.sum(lowData, di, dj), mix.n[di][dj]);
                storePair<PAIRS>(at(high.dataPost, b, c0 + k, 2 * a + di, 2 * e), high.dataPost.x, second, out);
            }
        }
    }
}

/** The value of the lane in front (STEP = -1) or behind (1) in a row of 16 lanes; zero where there is none. All lanes of the wavefront. */
template <int STEP, typename T>
__device__ __forceinline__ T besides(T v)
{
    constexpr int CONTROL = STEP < 0 ? 0x111 : 0x101;   // row_shr:1, row_shl:1
    int words[sizeof(T) / 4];
    __builtin_memcpy(words, &v, sizeof(T));
#pragma unroll
    for (int i = 0; i < static_cast<int>(sizeof(T) / 4); ++i) words[i] = __builtin_amdgcn_update_dpp(0, words[i], CONTROL, 0xf, 0xf, true);
    __builtin_memcpy(&v, words, sizeof(T));
    return v;
}

/**
 * Step A for the TW x TH low-res pixels from (a0, e0) on, by a workgroup of a thread per quad of the tile and a border of one quad (all
 * of them call this; a row of quads is a row of 16 lanes):
 *   gradDataPost_c of the low-res pixel = mask * sum over the 4 x 4 high-res pixels p that interpolate from it of w_p fill_c(p)
 *   gradMaskPost                        = sum of w_p (fillN(p) + sum_c fill_c(p) data_c)
 * with fill_c(p) the gradient of the weighted low-res sum d_c of p and fillN(p) that of its mask sum n. The weights are
 * products of 1/4, 3/4, 3/4, 1/4 in both directions: a thread forms the terms of its quad's four pixels and adds up those of
 * a row with the quads besides it, and what remains of the rows above and below comes through LDS, two values per quad and channel. (All
 * terms through LDS and 16 of them read per low-res pixel and channel: two per bank and instruction, the same time on 2048 x 2048
 * floats with the tests for the border taken out of the interior. Bound by its vector instructions, about 700 per quad: 33 of 45 us.)
 */
template <bool PAIRS, bool INTERIOR, int TW, int TH, typename T>
__device__ __forceinline__ void gradientUpTile(const PullPushLevel<T>& high, const PullPushLevel<T>& low, int C, int b, int a0, int e0,
                                               T (&sRows)[pullpushChunk<T>() + 1][2][(TW + 2) * (TH + 2)],
                                               typename LowTile<T, TW + 2, TH + 2>::Memory& sLow)
{
    typedef LowTile<T, TW + 2, TH + 2> Low;
    constexpr int QW = TW + 2, CHUNK = pullpushChunk<T>();
    static_assert(QW == 16, "a row of quads is a row of 16 lanes");
    const int tid = threadIdx.x, la = tid / QW, le = tid % QW;
    const int qa = a0 - 1 + la, qe = e0 - 1 + le;   // the quad, and the low-res pixel that it lies in
    const bool inside = INTERIOR || (qa >= 0 && qe >= 0 && 2 * qa < high.H && 2 * qe < high.W);
    const bool mine = la >= 1 && la <= TH && le >= 1 && le <= TW && (INTERIOR || (qa < low.H && qe < low.W));
    const bool second = INTERIOR || 2 * qe + 1 < high.W;
    bool in[2][2];   // outside: passes nothing down
#pragma unroll
    for (int i = 0; i < 4; ++i) in[i >> 1][i & 1] = INTERIOR || (inside && 2 * qa + (i >> 1) < high.H && ((i & 1) == 0 || second));
    T fillN[2][2], m[2][2], gradMask = 0;
    // the sum along the rows of the terms of a quad and of those besides it
    auto along = [&](const T (&f)[2][2], T (&rows)[2]) {
#pragma unroll
        for (int di = 0; di < 2; ++di) rows[di] = 0.75f * (f[di][0] + f[di][1]) + 0.25f * (besides<-1>(f[di][1]) + besides<1>(f[di][0]));
    };
    auto down = [&](const T (&rows)[2], const T (&other)[2][(TW + 2) * (TH + 2)]) {
        return 0.75f * (rows[0] + rows[1]) + 0.25f * (other[1][tid - QW] + other[0][tid + QW]);
    };
    for (int c0 = 0; c0 < C; c0 += CHUNK) {
        if (c0 > 0) ldsBarrier();   // what the channels in front of these left has been read
        Low::stage(sLow, low, C, b, c0, a0 - 1, e0 - 1);
        ldsBarrier();
        T fill[CHUNK][2][2], gm[2][2];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            gm[i >> 1][i & 1] = T(0);
#pragma unroll
            for (int k = 0; k < CHUNK; ++k) fill[k][i >> 1][i & 1] = T(0);
        }
        if (inside) {
#pragma unroll
            for (int di = 0; di < 2; ++di) {
                if (!INTERIOR && 2 * qa + di >= high.H) continue;
                if (c0 == 0) {
                    m[di][0] = m[di][1] = T(0);
                    loadPair<PAIRS>(at(high.maskPre, b, 0, 2 * qa + di, 2 * qe), high.maskPre.x, second, m[di]);
                    if (high.gradMaskPost.p)
                        loadPair<PAIRS>(at(high.gradMaskPost, b, 0, 2 * qa + di, 2 * qe), high.gradMaskPost.x, second, gm[di]);
                }
#pragma unroll
                for (int k = 0; k < CHUNK; ++k)   // (the gradient: turned into the fill below)
                    if (c0 + k < C) loadPair<PAIRS>(at(high.gradDataPost, b, c0 + k, 2 * qa + di, 2 * qe), high.gradDataPost.x, second, fill[k][di]);
            }
        }
        {
            const Neighbourhood<INTERIOR> nb(qa, qe, low.H, low.W);
            T masks[3][3];
            Low::load(sLow[CHUNK], la, le, masks);
            const QuadMix<T> mix(nb, masks);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int di = i >> 1, dj = i & 1;
                if (c0 == 0) fillN[di][dj] = high.gradMaskPost.p && in[di][dj] ? gm[di][dj] * ((1 - m[di][dj]) / mix.weight[di][dj]) : T(0);
            }
#pragma unroll
            for (int k = 0; k < CHUNK; ++k) {
                if (c0 + k >= C) continue;
                T lowData[3][3];
                Low::load(sLow[k], la, le, lowData);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int di = i >> 1, dj = i & 1;
                    const T f = mix.inverse[di][dj](fill[k][di][dj] * (1 - m[di][dj]));
                    fill[k][di][dj] = in[di][dj] ? f : T(0);
                    if (in[di][dj]) fillN[di][dj] -= f * mix.inverse[di][dj](mix.sum(lowData, di, dj));
                }
            }
        }
        T rows[CHUNK + 1][2];
#pragma unroll
        for (int k = 0; k < CHUNK; ++k) {
            if (c0 + k >= C) continue;
            along(fill[k], rows[k]);
            sRows[k][0][tid] = rows[k][0];
            sRows[k][1][tid] = rows[k][1];
        }
        const bool last = c0 + CHUNK >= C;
        if (last) {
            along(fillN, rows[CHUNK]);
            sRows[CHUNK][0][tid] = rows[CHUNK][0];
            sRows[CHUNK][1][tid] = rows[CHUNK][1];
        }
        ldsBarrier();
        if (!mine) continue;
        const int own = (la + 1) * Low::PITCH + le + 1;
        const T lowMask = sLow[CHUNK][own];
#pragma unroll
        for (int k = 0; k < CHUNK; ++k) {
            if (c0 + k >= C) continue;
            const T sum = down(rows[k], sRows[k]);
            gradMask += sum * sLow[k][own];
            *at(low.gradDataPost, b, c0 + k, qa, qe) = sum * lowMask;
        }
        if (last) *at(low.gradMaskPost, b, 0, qa, qe) = gradMask + down(rows[CHUNK], sRows[CHUNK]);
    }
}

/**
 * Step B for the QW x QH quads from (a0, e0) on: the gradients of their pixels before inpainting, a thread per quad (all threads of
 * the workgroup call this).
 * \tparam ACCUMULATE add to what is there
 */
template <bool PAIRS, bool ACCUMULATE, int QW, int QH, typename T>
__device__ __forceinline__ void gradientQuads(const PullPushLevel<T>& high, const PullPushLevel<T>& low, int C, int b, int a0, int e0,
                                              typename LowTile<T, QW, QH>::Memory& sLow)
{
    typedef LowTile<T, QW, QH> Low;
    constexpr int STAGED = pullpushChunk<T>();
    const int la = threadIdx.x / QW, le = threadIdx.x % QW, a = a0 + la, e = e0 + le;
    const bool mine = 2 * a < high.H && 2 * e < high.W;
    Low::stage(sLow, low, C, b, 0, a0, e0);
    __syncthreads();
    const Neighbourhood<> nb(a, e, low.H, low.W);
    T lowMask[3][3];
    Low::load(sLow[STAGED], la, le, lowMask);
    const QuadMix<T> mix(nb, lowMask);
    const bool second = 2 * e + 1 < high.W;
    // the low-res windows the pixels lie in: (a, e), and of odd sizes also those of the row above and the column to the
    // left, which reach into the first row and column of the quad
    const bool oddH = high.H & 1, oddW = high.W & 1;
    bool in[2][2];
    T most[2][2], gradMost[2][2];
    Reciprocal<T> sums[2][2];
#pragma unroll
    for (int wa = 0; wa < 2; ++wa)
#pragma unroll
        for (int we = 0; we < 2; ++we) {
            const int y = a - wa, x = e - we;
            in[wa][we] = mine && (wa == 0 || oddH) && (we == 0 || oddW) && y >= 0 && x >= 0 && y < low.H && x < low.W;
            most[wa][we] = gradMost[wa][we] = T(0);
            if (!in[wa][we]) continue;
            sums[wa][we] = Reciprocal<T>(*at(low.maskSum, b, 0, y, x));
            most[wa][we] = *at(low.maskPre, b, 0, y, x);
            gradMost[wa][we] = *at(low.gradMaskPre, b, 0, y, x);
        }
    T m[2][2], gradMask[2][2];
#pragma unroll
    for (int di = 0; di < 2; ++di) {
        m[di][0] = m[di][1] = gradMask[di][0] = gradMask[di][1] = T(0);
        if (!mine || 2 * a + di >= high.H) continue;
        loadPair<PAIRS>(at(high.maskPre, b, 0, 2 * a + di, 2 * e), high.maskPre.x, second, m[di]);
        T gm[2] = {T(0), T(0)};
        if (high.gradMaskPost.p)
            loadPair<PAIRS>(at(high.gradMaskPost, b, 0, 2 * a + di, 2 * e), high.gradMaskPost.x, second, gm);
#pragma unroll
        for (int dj = 0; dj < 2; ++dj) {
            if (dj == 1 && !second) continue;
            // maskHigh = m + (n > 0 ? (1 - m) * n / weight : 0)
            gradMask[di][dj] = high.gradMaskPost.p ? gm[dj] * (1 - mix.n[di][dj] / mix.weight[di][dj]) : T(0);
            // the maximum of a window passes its gradient to every pixel that attains it
#pragma unroll
            for (int wa = 0; wa <= 1 - di; ++wa)
#pragma unroll
                for (int we = 0; we <= 1 - dj; ++we)
                    if (in[wa][we] && most[wa][we] == m[di][dj]) gradMask[di][dj] += gradMost[wa][we];
        }
    }
    constexpr int CHUNK = 1;   // (more of them in flight cost more wavefronts than they hide: 2048 x 2048 floats 70 us with one, 98 us with two)
    for (int c0 = 0; c0 < C; c0 += CHUNK) {
        if (c0 > 0 && c0 % STAGED == 0) {
            __syncthreads();   // the channels in front of these have been read
            Low::stage(sLow, low, C, b, c0, a0, e0);
            __syncthreads();
        }
        if (!mine) continue;
        T lowData[CHUNK][3][3], v[CHUNK][2][2], g[CHUNK][2][2], before[CHUNK][2][2];
        T mean[CHUNK][2][2], grad[CHUNK][2][2];   // of the windows
#pragma unroll
        for (int k = 0; k < CHUNK; ++k) {
            if (c0 + k >= C) continue;
            Low::load(sLow[(c0 + k) % STAGED], la, le, lowData[k]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int wa = i >> 1, we = i & 1;
                mean[k][wa][we] = grad[k][wa][we] = T(0);
                if (!in[wa][we]) continue;
                mean[k][wa][we] = *at(low.dataPre, b, c0 + k, a - wa, e - we);
                grad[k][wa][we] = sums[wa][we](*at(low.gradDataPre, b, c0 + k, a - wa, e - we));
            }
#pragma unroll
            for (int di = 0; di < 2; ++di) {
                before[k][di][0] = before[k][di][1] = T(0);
                if (2 * a + di >= high.H) continue;
                loadPair<PAIRS>(at(high.dataPre, b, c0 + k, 2 * a + di, 2 * e), high.dataPre.x, second, v[k][di]);
                loadPair<PAIRS>(at(high.gradDataPost, b, c0 + k, 2 * a + di, 2 * e), high.gradDataPost.x, second, g[k][di]);
                if (ACCUMULATE) loadPair<PAIRS>(at(high.gradDataPre, b, c0 + k, 2 * a + di, 2 * e), high.gradDataPre.x, second, before[k][di]);
            }
        }
#pragma unroll
        for (int k = 0; k < CHUNK; ++k) {
            if (c0 + k >= C) continue;
#pragma unroll
            for (int di = 0; di < 2; ++di) {
                if (2 * a + di >= high.H) continue;
                T out[2];
#pragma unroll
                for (int dj = 0; dj < 2; ++dj) {
                    // dataHigh = m * data + (1 - m) * (n > 0 ? d / n : 0)
                    gradMask[di][dj] += g[k][di][dj] * (v[k][di][dj] - mix.inverse[di][dj](mix.sum(lowData[k], di, dj)));
                    T sum = g[k][di][dj];
#pragma unroll
                    for (int wa = 0; wa <= 1 - di; ++wa)
#pragma unroll
                        for (int we = 0; we <= 1 - dj; ++we) {
                            // dataLow = sum m * data / sum m
                            if (!in[wa][we]) continue;
                            sum += grad[k][wa][we];
                            gradMask[di][dj] += grad[k][wa][we] * (v[k][di][dj] - mean[k][wa][we]);
                        }
                    out[dj] = before[k][di][dj] + m[di][dj] * sum;
                }
                storePair<PAIRS>(at(high.gradDataPre, b, c0 + k, 2 * a + di, 2 * e), high.gradDataPre.x, second, out);
            }
        }
    }
    if (!mine) return;
#pragma unroll
    for (int di = 0; di < 2; ++di) {
        if (2 * a + di >= high.H) continue;
        T* target = at(high.gradMaskPre, b, 0, 2 * a + di, 2 * e);
        if (ACCUMULATE) {
            T before[2];
            loadPair<PAIRS>(target, high.gradMaskPre.x, second, before);
            gradMask[di][0] += before[0];
            gradMask[di][1] += before[1];
        }
        storePair<PAIRS>(target, high.gradMaskPre.x, second, gradMask[di]);
    }
}

constexpr int TILE_W = 32, TILE_H = 8;   // of the kernels with a launch per level: 256 threads
// ... and of step A: with their border the quads of a tile are as many as there are threads, in rows of 16 lanes (32 x 8 pixels by 256
// threads were 340 quads, two rounds with the second a third full; 2048 x 2048 floats 51 us, now 45)
constexpr int UP_TILE_W = 14, UP_TILE_H = 14, UP_THREADS = (UP_TILE_W + 2) * (UP_TILE_H + 2);

/**
 * Tile of this workgroup: a stack of B images of width x height items in tiles of TILE_W x TILE_H. Workgroups go to the 8 XCDs
 * in turn; every XCD gets a run of consecutive tiles, whose borders then meet in its own L2.
 */
template <int TW = TILE_W, int TH = TILE_H>
__device__ __forceinline__ void tileOf(int width, int height, int& b, int& a0, int& e0)
{
    constexpr unsigned XCDS = 8;
    const unsigned xcd = blockIdx.x % XCDS, perXcd = gridDim.x / XCDS, more = gridDim.x % XCDS;
    const unsigned tile = xcd * perXcd + min(xcd, more) + blockIdx.x / XCDS;
    const unsigned tilesX = (width + TW - 1) / TW, tilesY = (height + TH - 1) / TH;
    const unsigned row = tile / tilesX;
    e0 = static_cast<int>(tile - row * tilesX) * TW;
    b = static_cast<int>(row / tilesY);
    a0 = static_cast<int>(row - b * tilesY) * TH;
}

/**
 * Level k (> 0) of the coarse levels that one workgroup keeps in LDS, below a level of H x W pixels (sizes are halved, rounding
 * down, and rows start at even entries). Read and written as LDS and not through addresses that may lie anywhere.
 */
template <typename T>
struct LdsLevel
{
    typedef __attribute__((address_space(3))) T entry;
    int H, W, pitch, plane;
    entry *maskPreP, *dataPreP, *maskSumP, *maskPostP, *dataPostP, *gradMaskPostP, *gradDataPostP, *gradMaskPreP, *gradDataPreP;

    /** \param gradients the gradients of a level lie behind it */
    __device__ __forceinline__ LdsLevel(entry* levels, const PullPushTail& tail, int finestH, int finestW, int C, int k, bool gradients)
    {
        entry* next = levels + tail.offsets[k];
        H = finestH >> k;
        W = finestW >> k;
        pitch = (W + 1) & ~1;
        plane = H * pitch;
        auto take = [&](int channels) {
            entry* p = next;
            next += channels * plane;
            return p;
        };
        maskPreP = take(1);
        dataPreP = take(C);
        maskSumP = take(1);
        const bool coarsest = k == tail.numLevels - 1;   // its own inpainting: nothing changes from before to after
        maskPostP = coarsest ? maskPreP : take(1);
        dataPostP = coarsest ? dataPreP : take(C);
        gradMaskPostP = gradDataPostP = gradMaskPreP = gradDataPreP = next;
        if (gradients) {
            gradMaskPostP = take(1);
            gradDataPostP = take(C);
            gradMaskPreP = coarsest ? gradMaskPostP : take(1);
            gradDataPreP = coarsest ? gradDataPostP : take(C);
        }
    }
    __device__ __forceinline__ entry& at(entry* p, int c, int y, int x) const { return p[c * plane + y * pitch + x]; }
    __device__ __forceinline__ bool hasMaskPost() const { return true; }
    __device__ __forceinline__ bool hasGradMaskPost() const { return true; }
    __device__ __forceinline__ entry& maskPre(int y, int x) const { return at(maskPreP, 0, y, x); }
    __device__ __forceinline__ entry& dataPre(int c, int y, int x) const { return at(dataPreP, c, y, x); }
    __device__ __forceinline__ entry& maskSum(int y, int x) const { return at(maskSumP, 0, y, x); }
    __device__ __forceinline__ entry& maskPost(int y, int x) const { return at(maskPostP, 0, y, x); }
    __device__ __forceinline__ entry& dataPost(int c, int y, int x) const { return at(dataPostP, c, y, x); }
    __device__ __forceinline__ void setGradMaskPost(int y, int x, T v) const { gradMaskPost(y, x) = v; }
    __device__ __forceinline__ void setGradDataPost(int c, int y, int x, T v) const { gradDataPost(c, y, x) = v; }
    __device__ __forceinline__ entry& gradMaskPost(int y, int x) const { return at(gradMaskPostP, 0, y, x); }
    __device__ __forceinline__ entry& gradDataPost(int c, int y, int x) const { return at(gradDataPostP, c, y, x); }
    __device__ __forceinline__ entry& gradMaskPre(int y, int x) const { return at(gradMaskPreP, 0, y, x); }
    __device__ __forceinline__ entry& gradDataPre(int c, int y, int x) const { return at(gradDataPreP, c, y, x); }
};

/**
 * The level above them, in global memory: what the steps read of it is copied into LDS first, as it is read several
 * times and by few lanes (a global load in every round of a step's loop: 64 x 64 pixels 103 us), what they write goes to global memory.
 */
template <typename T>
struct TopLevel
{
    typedef typename LdsLevel<T>::entry entry;
    const PullPushLevel<T>& l;
    int b, H, W, pitch, plane;
    entry *maskPreP, *dataPreP, *gradMaskPostP, *gradDataPostP;

    __device__ __forceinline__ static void copy(entry* to, const PullPushView<T>& from, int b, int C, int H, int W, int pitch)
    {
        const float inverse = 1.f / static_cast<float>(W);
        for (int c = 0; c < C; ++c)
#pragma unroll 4
            for (int i = threadIdx.x; i < H * W; i += PULLPUSH_TAIL_BLOCK) {
                const int y = static_cast<int>((static_cast<float>(i) + 0.5f) * inverse);
                to[(c * H + y) * pitch + (i - y * W)] = *at(from, b, c, y, i - y * W);
            }
    }
    /** All lanes of the workgroup; a barrier is up to the caller. */
    __device__ __forceinline__ TopLevel(const PullPushLevel<T>& level, int image, entry* top, int C, bool gradients)
        : l(level), b(image), H(level.H), W(level.W)
    {
        pitch = (W + 1) & ~1;
        plane = H * pitch;
        maskPreP = top;
        dataPreP = maskPreP + plane;
        gradMaskPostP = dataPreP + C * plane;
        gradDataPostP = gradMaskPostP + plane;
        copy(maskPreP, l.maskPre, b, 1, H, W, pitch);
        copy(dataPreP, l.dataPre, b, C, H, W, pitch);
        if (!gradients) return;
        if (l.gradMaskPost.p) copy(gradMaskPostP, l.gradMaskPost, b, 1, H, W, pitch);
        copy(gradDataPostP, l.gradDataPost, b, C, H, W, pitch);
    }
    __device__ __forceinline__ bool hasMaskPost() const { return l.maskPost.p != nullptr; }
    __device__ __forceinline__ bool hasGradMaskPost() const { return l.gradMaskPost.p != nullptr; }
    __device__ __forceinline__ T maskPre(int y, int x) const { return maskPreP[y * pitch + x]; }
    __device__ __forceinline__ T dataPre(int c, int y, int x) const { return dataPreP[c * plane + y * pitch + x]; }
    __device__ __forceinline__ T gradMaskPost(int y, int x) const { return gradMaskPostP[y * pitch + x]; }
    __device__ __forceinline__ T gradDataPost(int c, int y, int x) const { return gradDataPostP[c * plane + y * pitch + x]; }
    __device__ __forceinline__ T& maskPost(int y, int x) const { return *at(l.maskPost, b, 0, y, x); }
    __device__ __forceinline__ T& dataPost(int c, int y, int x) const { return *at(l.dataPost, b, c, y, x); }
    __device__ __forceinline__ T& gradMaskPre(int y, int x) const { return *at(l.gradMaskPre, b, 0, y, x); }
    __device__ __forceinline__ T& gradDataPre(int c, int y, int x) const { return *at(l.gradDataPre, b, c, y, x); }
};

/** What the steps read of a low-res level in global memory, all planes of which have the same pitch (the workspaces'). */
template <typename T>
struct GlobalLow
{
    int H, W, pitch;
    long long plane;
    const T *maskPreP, *dataPreP, *maskSumP, *maskPostP, *dataPostP, *gradMaskPreP, *gradDataPreP;
    __device__ __forceinline__ GlobalLow(const PullPushLevel<T>& l, int b)
        : H(l.H), W(l.W), pitch(static_cast<int>(l.maskPre.y)), plane(l.dataPre.c), maskPreP(l.maskPre.p + b * l.maskPre.b),
          dataPreP(l.dataPre.p + b * l.dataPre.b), maskSumP(l.maskSum.p + b * l.maskSum.b), maskPostP(l.maskPost.p + b * l.maskPost.b),
          dataPostP(l.dataPost.p + b * l.dataPost.b), gradMaskPreP(l.gradMaskPre.p + b * l.gradMaskPre.b),
          gradDataPreP(l.gradDataPre.p + b * l.gradDataPre.b)
    {
    }
    __device__ __forceinline__ T gradMaskPre(int a, int e) const { return gradMaskPreP[a * pitch + e]; }
    __device__ __forceinline__ T gradDataPre(int c, int a, int e) const { return gradDataPreP[c * plane + a * pitch + e]; }
};

/** Rows and columns of a level that a workgroup works on. */
struct PullPushRegion
{
    int y0, y1, x0, x1;
    __device__ __forceinline__ int rows() const { return y1 - y0; }
    __device__ __forceinline__ int columns() const { return x1 - x0; }
};

/** C + 1 planes of a region in LDS: of a mask, and of the channels. Zero bytes behind the entries of the region before it. */
template <typename T>
struct LdsTile
{
    typedef typename LdsLevel<T>::entry entry;
    entry* p;
    int y0, x0, pitch, plane;
    __device__ __forceinline__ LdsTile(entry* memory, const PullPushRegion& r)
        : p(memory), y0(r.y0), x0(r.x0), pitch(r.columns()), plane(r.rows() * r.columns()) {}
    __device__ __forceinline__ entry& mask(int y, int x) const { return p[(y - y0) * pitch + (x - x0)]; }
    __device__ __forceinline__ entry& data(int c, int y, int x) const { return p[(c + 1) * plane + (y - y0) * pitch + (x - x0)]; }
};

/** What the steps read and write of a high-res level in global memory. */
template <typename T>
struct GlobalHigh
{
    const PullPushLevel<T>& l;
    int b, H, W;
    __device__ __forceinline__ GlobalHigh(const PullPushLevel<T>& level, int image) : l(level), b(image), H(level.H), W(level.W) {}
    __device__ __forceinline__ bool hasMaskPost() const { return l.maskPost.p != nullptr; }
    __device__ __forceinline__ bool hasGradMaskPost() const { return l.gradMaskPost.p != nullptr; }
    __device__ __forceinline__ T maskPre(int y, int x) const { return *at(l.maskPre, b, 0, y, x); }
    __device__ __forceinline__ T dataPre(int c, int y, int x) const { return *at(l.dataPre, b, c, y, x); }
    __device__ __forceinline__ T gradMaskPost(int y, int x) const { return *at(l.gradMaskPost, b, 0, y, x); }
    __device__ __forceinline__ T gradDataPost(int c, int y, int x) const { return *at(l.gradDataPost, b, c, y, x); }
    __device__ __forceinline__ T& maskPost(int y, int x) const { return *at(l.maskPost, b, 0, y, x); }
    __device__ __forceinline__ T& dataPost(int c, int y, int x) const { return *at(l.dataPost, b, c, y, x); }
    __device__ __forceinline__ T& gradMaskPre(int y, int x) const { return *at(l.gradMaskPre, b, 0, y, x); }
    __device__ __forceinline__ T& gradDataPre(int c, int y, int x) const { return *at(l.gradDataPre, b, c, y, x); }
};
/** ... whose gradients before inpainting stay in LDS, and a low-res level with its own there. */
template <typename T>
struct GradientTileHigh : GlobalHigh<T>
{
    LdsTile<T> tile;
    __device__ __forceinline__ GradientTileHigh(const PullPushLevel<T>& level, int image, const LdsTile<T>& t) : GlobalHigh<T>(level, image), tile(t) {}
    __device__ __forceinline__ typename LdsTile<T>::entry& gradMaskPre(int y, int x) const { return tile.mask(y, x); }
    __device__ __forceinline__ typename LdsTile<T>::entry& gradDataPre(int c, int y, int x) const { return tile.data(c, y, x); }
};
template <typename T>
struct GradientTileLow : GlobalLow<T>
{
    LdsTile<T> tile;
    __device__ __forceinline__ GradientTileLow(const PullPushLevel<T>& level, int image, const LdsTile<T>& t) : GlobalLow<T>(level, image), tile(t) {}
    __device__ __forceinline__ T gradMaskPre(int a, int e) const { return tile.mask(a, e); }
    __device__ __forceinline__ T gradDataPre(int c, int a, int e) const { return tile.data(c, a, e); }
};

/** An inpainted low-res level in LDS, and a high-res level that is inpainted into LDS, into global memory where it is owned, or both. */
template <typename T>
struct InpaintedTileLow
{
    int H, W, pitch, plane;
    typename LdsTile<T>::entry *maskPostP, *dataPostP;
    __device__ __forceinline__ InpaintedTileLow(const PullPushLevel<T>& l, const LdsTile<T>& t)
        : H(l.H), W(l.W), pitch(t.pitch), plane(t.plane), maskPostP(t.p - (t.y0 * t.pitch + t.x0)), dataPostP(maskPostP + t.plane) {}
};

/**
 * Where workgroups of PULLPUSH_TAIL_BLOCK lanes take tiles of the finest of several levels and what the coarser ones below have to
 * do with them. Sizes in LDS: a region of level k has at most (tile >> k) + TREE_BORDER rows and columns.
 */
constexpr int TREE_BORDER = 5;
__device__ __forceinline__ PullPushRegion treeTile(int H, int W, int tile, int& b)
{
    constexpr unsigned XCDS = 8;
    const unsigned xcd = blockIdx.x % XCDS, perXcd = gridDim.x / XCDS, more = gridDim.x % XCDS;
    const unsigned index = xcd * perXcd + min(xcd, more) + blockIdx.x / XCDS;
    const unsigned tilesX = (W + tile - 1) / tile, tilesY = (H + tile - 1) / tile;
    const unsigned row = index / tilesX;
    b = static_cast<int>(row / tilesY);
    const int x0 = static_cast<int>(index - row * tilesX) * tile, y0 = static_cast<int>(row - b * tilesY) * tile;
    return {y0, min(y0 + tile, H), x0, min(x0 + tile, W)};
}
template <typename T>
__device__ __forceinline__ typename LdsLevel<T>::entry* treeMemory(typename LdsLevel<T>::entry* memory, const PullPushTree<T>& tree, int C, int k)
{
    for (int i = 1; i < k; ++i) memory += (C + 1) * ((tree.tile >> i) + TREE_BORDER) * ((tree.tile >> i) + TREE_BORDER);
    return memory;
}

/** A high-res level with its pixels before inpainting in LDS. */
template <typename T>
struct DownTileHigh
{
    int H, W;
    LdsTile<T> tile;
    __device__ __forceinline__ DownTileHigh(const PullPushLevel<T>& l, const LdsTile<T>& t) : H(l.H), W(l.W), tile(t) {}
    __device__ __forceinline__ T maskPre(int y, int x) const { return tile.mask(y, x); }
    __device__ __forceinline__ T dataPre(int c, int y, int x) const { return tile.data(c, y, x); }
};
/** A high-res level with the gradients of its inpainted pixels in LDS, and a low-res one that receives its own there, in global memory where it is owned, or both. */
template <typename T>
struct UpTileHigh : GlobalHigh<T>
{
    LdsTile<T> tile;
    __device__ __forceinline__ UpTileHigh(const PullPushLevel<T>& level, int image, const LdsTile<T>& t) : GlobalHigh<T>(level, image), tile(t) {}
    __device__ __forceinline__ T gradMaskPost(int y, int x) const { return tile.mask(y, x); }
    __device__ __forceinline__ T gradDataPost(int c, int y, int x) const { return tile.data(c, y, x); }
};
template <typename T>
struct UpTileLow : GlobalLow<T>
{
    const PullPushLevel<T>& l;
    int b;
    PullPushRegion owned;
    bool keep;
    LdsTile<T> tile;
    __device__ __forceinline__ UpTileLow(const PullPushLevel<T>& level, int image, const PullPushRegion& own, bool keepTile, const LdsTile<T>& t)
        : GlobalLow<T>(level, image), l(level), b(image), owned(own), keep(keepTile), tile(t) {}
    __device__ __forceinline__ bool own(int a, int e) const { return a >= owned.y0 && a < owned.y1 && e >= owned.x0 && e < owned.x1; }
    __device__ __forceinline__ void setGradDataPost(int c, int a, int e, T v) const
    {
        if (own(a, e)) *at(l.gradDataPost, b, c, a, e) = v;
        if (keep) tile.data(c, a, e) = v;
    }
    __device__ __forceinline__ void setGradMaskPost(int a, int e, T v) const
    {
        if (own(a, e)) *at(l.gradMaskPost, b, 0, a, e) = v;
        if (keep) tile.mask(a, e) = v;
    }
    __device__ __forceinline__ T maskPost(int a, int e) const { return this->maskPostP[a * this->pitch + e]; }
    __device__ __forceinline__ T dataPost(int c, int a, int e) const { return this->dataPostP[c * this->plane + a * this->pitch + e]; }
};
/** Rows (and columns) at most of a region of level k in LDS, of a tree that ends at level 'last' with (tile >> last) of them. */
__device__ __forceinline__ int treeDownSize(int tile, int last, int k) { return (tile >> k) + (1 << (last - k)) - 1; }
__device__ __forceinline__ int treeUpSize(int tile, int last, int k) { return (tile >> k) + 2 * ((1 << (last - k)) - 1); }

/**
 * The steps of the coarse levels, by one compute unit: a chain of a few dependent loads and a division per step, and on the larger
 * levels vector instructions. An item is a pixel with all its channels where that fills the workgroup, on smaller levels 2^n neighbouring
 * lanes share the channels of a pixel, look the masks up each for itself, and add up what the mask's gradient takes
 * from all channels with shuffles. (A lane per channel on every level: 39
 * instead of 32 us for the adjoint of 32 x 32 x 4 floats and below, of which a step of 2 x 2 pixels takes 2 us, one of 32 x 32 up to 5.)
 */
template <typename T>
struct TailSteps
{
    typedef typename LdsLevel<T>::entry entry;
    int C;
    __device__ __forceinline__ explicit TailSteps(int channels) : C(channels) {}

    /** Lanes per pixel (their logarithm) for so many pixels and channels. */
    __device__ __forceinline__ static int lanesLog2(int pixels, int channels)
    {
        int log2 = 0;
        while ((1 << log2) < channels && (pixels << (log2 + 1)) <= PULLPUSH_TAIL_BLOCK) ++log2;
        return log2;
    }
    /** Calls item(y, x, lane of the pixel) for rows x W pixels from (y0, x0) on, all lanes of a pixel at the same time. */
    template <typename Item>
    __device__ __forceinline__ static void forEach(int y0, int x0, int rows, int W, int log2, const Item& item)
    {
        const int items = (rows * W) << log2;
        const float inverse = 1.f / static_cast<float>(W);
        for (int i = threadIdx.x; i < items; i += PULLPUSH_TAIL_BLOCK) {
            const int pixel = i >> log2;
            const int y = static_cast<int>((static_cast<float>(pixel) + 0.5f) * inverse);   // exact: LDS holds fewer than 2^20 pixels
            item(y0 + y, x0 + pixel - y * W, i & ((1 << log2) - 1));
        }
    }
    __device__ __forceinline__ static T sumOver(T v, int log2)
    {
        for (int d = 1; d < (1 << log2); d *= 2) v += __shfl_xor(v, d, 64);
        return v;
    }

    /** down for a region of the low-res level: store(c, a, e, value), storeMask(a, e, mask, sum of masks). */
    template <typename High, typename Store, typename StoreMask>
    __device__ __forceinline__ void downTo(const High& high, const PullPushRegion& r, const Store& store, const StoreMask& storeMask) const
    {
        if ((high.H | high.W) & 1) downTo<true>(high, r, store, storeMask);
        else downTo<false>(high, r, store, storeMask);
    }
    /** \tparam ODD some size is odd: windows of three rows or columns */
    template <bool ODD, typename High, typename Store, typename StoreMask>
    __device__ __forceinline__ void downTo(const High& high, const PullPushRegion& r, const Store& store, const StoreMask& storeMask) const
    {
        constexpr int MOST = ODD ? 3 : 2;
        const int rows = ODD ? 2 + (high.H & 1) : 2, columns = ODD ? 2 + (high.W & 1) : 2;
        const int log2 = lanesLog2(r.rows() * r.columns(), C);
        forEach(r.y0, r.x0, r.rows(), r.columns(), log2, [&](int a, int e, int lane) {
            T m[MOST][MOST];
            T sum = 0, most = 0;
#pragma unroll
            for (int j = 0; j < MOST; ++j)
#pragma unroll
                for (int i = 0; i < MOST; ++i) {
                    m[i][j] = T(0);
                    if (i >= rows || j >= columns) continue;
                    m[i][j] = high.maskPre(2 * a + i, 2 * e + j);
                    sum += m[i][j];
                    most = max(most, m[i][j]);
                }
            for (int c = lane; c < C; c += 1 << log2) {
                T d = 0;
#pragma unroll
                for (int j = 0; j < MOST; ++j)
#pragma unroll
                    for (int i = 0; i < MOST; ++i)
                        if (i < rows && j < columns) d += m[i][j] * high.dataPre(c, 2 * a + i, 2 * e + j);
                store(c, a, e, quotient(d, sum));
            }
            if (lane == 0) storeMask(a, e, most, sum);
        });
    }
    template <typename High>
    __device__ __forceinline__ void down(const High& high, const LdsLevel<T>& low) const
    {
        downTo(high, PullPushRegion{0, low.H, 0, low.W}, [&](int c, int a, int e, T v) { low.dataPre(c, a, e) = v; },
               [&](int a, int e, T most, T sum) {
                   low.maskPre(a, e) = most;
                   low.maskSum(a, e) = sum;
               });
    }
    /** ... into global memory what is owned, all of it into a tile as well. */
    template <typename High>
    __device__ __forceinline__ void downRegion(const High& high, const GlobalHigh<T>& low, const PullPushRegion& r, const PullPushRegion& owned, bool keep,
                                               const LdsTile<T>& tile) const
    {
        auto own = [&](int a, int e) { return a >= owned.y0 && a < owned.y1 && e >= owned.x0 && e < owned.x1; };
        downTo(high, r,
               [&](int c, int a, int e, T v) {
                   if (own(a, e)) *at(low.l.dataPre, low.b, c, a, e) = v;
                   if (keep) tile.data(c, a, e) = v;
               },
               [&](int a, int e, T most, T sum) {
                   if (own(a, e)) {
                       *at(low.l.maskPre, low.b, 0, a, e) = most;
                       *at(low.l.maskSum, low.b, 0, a, e) = sum;
                   }
                   if (keep) tile.mask(a, e) = most;
               });
    }

    /** The low-res neighbours of high-res pixel (y, x): the own cell, the one in the other row, in the other column, the diagonal one. */
    struct Mix
    {
        int at[4];
        T wm[4], n, weight;
        template <typename Low>
        __device__ __forceinline__ Mix(int y, int x, const Low& low)
        {
            const int row = y >> 1, column = x >> 1;
            const int otherRow = row - 1 + 2 * (y & 1), otherColumn = column - 1 + 2 * (x & 1);
            const float own = row < low.H ? 0.75f : 0.f, other = otherRow >= 0 && otherRow < low.H ? 0.25f : 0.f;
            const float ownColumn = column < low.W ? 0.75f : 0.f, otherC = otherColumn >= 0 && otherColumn < low.W ? 0.25f : 0.f;
            const int a[2] = {min(row, low.H - 1) * low.pitch, min(max(otherRow, 0), low.H - 1) * low.pitch};
            const int e[2] = {min(column, low.W - 1), min(max(otherColumn, 0), low.W - 1)};
            const float w[4] = {own * ownColumn, other * ownColumn, own * otherC, other * otherC};
            n = weight = 0;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                at[k] = a[k & 1] + e[k >> 1];
                wm[k] = w[k] * low.maskPostP[at[k]];
                weight += w[k];
                n += wm[k];
            }
        }
        template <typename Low>
        __device__ __forceinline__ T sum(const Low& low, int c) const
        {
            const auto* data = low.dataPostP + c * low.plane;
            T d = 0;
#pragma unroll
            for (int k = 0; k < 4; ++k) d += wm[k] * data[at[k]];
            return d;
        }
    };

    template <typename High>
    __device__ __forceinline__ void up(const High& high, const LdsLevel<T>& low) const
    {
        const int log2 = lanesLog2(high.H * high.W, C);
        forEach(0, 0, high.H, high.W, log2, [&](int y, int x, int lane) {
            const T m = high.maskPre(y, x);
            const Mix mix(y, x, low);
            for (int c = lane; c < C; c += 1 << log2)
                high.dataPost(c, y, x) = m * high.dataPre(c, y, x) + (1 - m) * quotient(mix.sum(low, c), mix.n);
            if (lane == 0 && high.hasMaskPost()) high.maskPost(y, x) = m + (mix.n > 0 ? (1 - m) * (mix.n / mix.weight) : T(0));
        });
    }

    /** The way up for a region of the high-res level: into global memory what is owned, all of it into a tile as well. */
    template <typename High, typename Low>
    __device__ __forceinline__ void upRegion(const High& high, const Low& low, const PullPushRegion& r, const PullPushRegion& owned, bool keep,
                                             const LdsTile<T>& tile) const
    {
        const int log2 = lanesLog2(r.rows() * r.columns(), C);
        forEach(r.y0, r.x0, r.rows(), r.columns(), log2, [&](int y, int x, int lane) {
            const bool own = y >= owned.y0 && y < owned.y1 && x >= owned.x0 && x < owned.x1;
            const T m = high.maskPre(y, x);
            const Mix mix(y, x, low);
            for (int c = lane; c < C; c += 1 << log2) {
                const T v = m * high.dataPre(c, y, x) + (1 - m) * quotient(mix.sum(low, c), mix.n);
                if (own) high.dataPost(c, y, x) = v;
                if (keep) tile.data(c, y, x) = v;
            }
            if (lane == 0) {
                const T v = m + (mix.n > 0 ? (1 - m) * (mix.n / mix.weight) : T(0));
                if (own && high.hasMaskPost()) high.maskPost(y, x) = v;
                if (keep) tile.mask(y, x) = v;
            }
        });
    }

    /**
     * Step A (see gradientUpTile) for a region of the low-res level. fill: room for fillEntries entries, at least (C + 1) x 4 rows of the
     * high-res pixels that it reaches. Ends with a barrier.
     */
    template <typename High, typename Low>
    __device__ __forceinline__ void gradientUp(const High& high, const Low& low, const PullPushRegion& r, entry* fill, int fillEntries) const
    {
        const int x0 = 2 * r.x0 - 1, pitch = 2 * r.columns() + 2;
        const int stripe = max(1, (fillEntries / ((C + 1) * pitch) - 2) / 2);   // low-res rows that are gathered together
        for (int a0 = r.y0; a0 < r.y1; a0 += stripe) {
            const int a1 = min(a0 + stripe, r.y1);
            const int y0 = 2 * a0 - 1, rows = 2 * (a1 - a0) + 2;   // (what lies outside of the image passes nothing down)
            const int plane = rows * pitch;
            const int fillLog2 = lanesLog2(plane, C);
            forEach(y0, x0, rows, pitch, fillLog2, [&](int y, int x, int lane) {
                entry* to = fill + ((y - y0) * pitch + x - x0);
                const bool inside = y >= 0 && y < high.H && x >= 0 && x < high.W;
                if (!inside) {
                    for (int c = lane; c <= C; c += 1 << fillLog2) to[c * plane] = T(0);
                    return;
                }
                const T m = high.maskPre(y, x);
                const Mix mix(y, x, low);
                const Reciprocal<T> inverse(mix.n);
                T fromMask = 0;
                for (int c = lane; c < C; c += 1 << fillLog2) {
                    const T f = inverse(high.gradDataPost(c, y, x) * (1 - m));
                    to[c * plane] = f;
                    fromMask += f * inverse(mix.sum(low, c));
                }
                fromMask = sumOver(fromMask, fillLog2);
                if (lane == 0) to[C * plane] = (high.hasGradMaskPost() ? high.gradMaskPost(y, x) * ((1 - m) / mix.weight) : T(0)) - fromMask;
            });
            ldsBarrier();
            const int gatherLog2 = lanesLog2((a1 - a0) * r.columns(), C + 1);
            forEach(a0, r.x0, a1 - a0, r.columns(), gatherLog2, [&](int a, int e, int lane) {
                T gradMask = 0;
                const T mask = low.maskPost(a, e);
                for (int c = lane; c <= C; c += 1 << gatherLog2) {
                    const entry* from = fill + (c * plane + 2 * (a - a0) * pitch + 2 * (e - r.x0));
                    T sum = 0;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float wr = (i == 1 || i == 2) ? 0.75f : 0.25f;
#pragma unroll
                        for (int j = 0; j < 4; ++j) sum += (wr * ((j == 1 || j == 2) ? 0.75f : 0.25f)) * from[i * pitch + j];
                    }
                    if (c == C) {
                        gradMask += sum;
                    } else {
                        gradMask += sum * low.dataPost(c, a, e);
                        low.setGradDataPost(c, a, e, sum * mask);
                    }
                }
                gradMask = sumOver(gradMask, gatherLog2);
                if (lane == 0) low.setGradMaskPost(a, e, gradMask);
            });
            ldsBarrier();
        }
    }

    /** Step B (see gradientQuads) for a region of the high-res level. \tparam ACCUMULATE add to what is there */
    template <bool ACCUMULATE, typename High, typename Low>
    __device__ __forceinline__ void gradient(const High& high, const Low& low, const PullPushRegion& r) const
    {
        if ((high.H | high.W) & 1) gradient<ACCUMULATE, true>(high, low, r);
        else gradient<ACCUMULATE, false>(high, low, r);
    }
    /** \tparam ODD some size is odd: a pixel may lie in several windows */
    template <bool ACCUMULATE, bool ODD, typename High, typename Low>
    __device__ __forceinline__ void gradient(const High& high, const Low& low, const PullPushRegion& r) const
    {
        constexpr int MOST = ODD ? 2 : 1;
        const bool oddH = high.H & 1, oddW = high.W & 1;
        const int log2 = lanesLog2(r.rows() * r.columns(), C);
        forEach(r.y0, r.x0, r.rows(), r.columns(), log2, [&](int y, int x, int lane) {
            const T m = high.maskPre(y, x);
            const Mix mix(y, x, low);
            const Reciprocal<T> inverse(mix.n);
            // the windows that the pixel lies in: of the own cell, and of odd sizes those of the row above and of the column to the left
            Reciprocal<T> sums[MOST][MOST];
            int window[MOST][MOST];
            bool in[MOST][MOST];
            T gradMask = 0;
#pragma unroll
            for (int wa = 0; wa < MOST; ++wa)
#pragma unroll
                for (int we = 0; we < MOST; ++we) {
                    const int a = (y >> 1) - wa, e = (x >> 1) - we;
                    in[wa][we] = (wa == 0 || (oddH && !(y & 1))) && (we == 0 || (oddW && !(x & 1))) && (!ODD || (a >= 0 && e >= 0 && a < low.H && e < low.W));
                    window[wa][we] = 0;
                    if (!in[wa][we]) continue;
                    window[wa][we] = a * low.pitch + e;
                    sums[wa][we] = Reciprocal<T>(low.maskSumP[window[wa][we]]);
                    // the maximum of a window passes its gradient to every pixel that attains it
                    if (lane == 0 && low.maskPreP[window[wa][we]] == m) gradMask += low.gradMaskPre(a, e);
                }
            for (int c = lane; c < C; c += 1 << log2) {
                const T v = high.dataPre(c, y, x), g = high.gradDataPost(c, y, x);
                T sum = g;
                gradMask += g * (v - inverse(mix.sum(low, c)));
#pragma unroll
                for (int wa = 0; wa < MOST; ++wa)
#pragma unroll
                    for (int we = 0; we < MOST; ++we) {
                        if (!in[wa][we]) continue;
                        const T grad = sums[wa][we](low.gradDataPre(c, (y >> 1) - wa, (x >> 1) - we));
                        sum += grad;
                        gradMask += grad * (v - low.dataPreP[c * low.plane + window[wa][we]]);
                    }
                const T out = m * sum;
                high.gradDataPre(c, y, x) = ACCUMULATE ? high.gradDataPre(c, y, x) + out : out;
            }
            gradMask = sumOver(gradMask, log2);
            if (lane == 0) {
                if (high.hasGradMaskPost()) gradMask += high.gradMaskPost(y, x) * (1 - mix.n / mix.weight);
                high.gradMaskPre(y, x) = ACCUMULATE ? high.gradMaskPre(y, x) + gradMask : gradMask;
            }
        });
    }
};
} // namespace pullpush

template <typename T>
__global__ void __launch_bounds__(256) PullPushDownKernel(const PullPushLevel<T> high, const PullPushLevel<T> low, int C, int pairs)
{
    using namespace pullpush;
    int b, a, e;
    tileOf(low.W, low.H, b, a, e);
    a += threadIdx.x / TILE_W;
    e += threadIdx.x % TILE_W;
    if (a >= low.H || e >= low.W) return;
    if (pairs) downPixel<true>(high, low, C, b, a, e);
    else downPixel<false>(high, low, C, b, a, e);
}

template <typename T>
__global__ void __launch_bounds__(256) PullPushUpKernel(const PullPushLevel<T> high, const PullPushLevel<T> low, int C, int pairs)
{
    using namespace pullpush;
    __shared__ typename LowTile<T, TILE_W, TILE_H>::Memory sLow;
    int b, a0, e0;
    tileOf((high.W + 1) / 2, (high.H + 1) / 2, b, a0, e0);
    if (pairs) upQuads<true, TILE_W, TILE_H>(high, low, C, b, a0, e0, sLow);
    else upQuads<false, TILE_W, TILE_H>(high, low, C, b, a0, e0, sLow);
}

template <typename T>
__global__ void __launch_bounds__(pullpush::UP_THREADS) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 4 : 2))) PullPushGradientUpKernel(const PullPushLevel<T> high, const PullPushLevel<T> low, int C, int pairs)
{
    using namespace pullpush;
    __shared__ T sRows[pullpushChunk<T>() + 1][2][UP_THREADS];
    __shared__ typename LowTile<T, UP_TILE_W + 2, UP_TILE_H + 2>::Memory sLow;
    int b, a0, e0;
    tileOf<UP_TILE_W, UP_TILE_H>(low.W, low.H, b, a0, e0);
    // all quads of the tile and its border, and their neighbours, lie in the image
    const bool interior = a0 >= 2 && e0 >= 2 && a0 + UP_TILE_H + 1 < low.H && e0 + UP_TILE_W + 1 < low.W;
    if (pairs && interior) gradientUpTile<true, true, UP_TILE_W, UP_TILE_H>(high, low, C, b, a0, e0, sRows, sLow);
    else if (pairs) gradientUpTile<true, false, UP_TILE_W, UP_TILE_H>(high, low, C, b, a0, e0, sRows, sLow);
    else gradientUpTile<false, false, UP_TILE_W, UP_TILE_H>(high, low, C, b, a0, e0, sRows, sLow);
}

template <typename T, bool ACCUMULATE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 && !ACCUMULATE ? 4 : 1))) PullPushGradientKernel(const PullPushLevel<T> high, const PullPushLevel<T> low, int C, int pairs)
{
    using namespace pullpush;
    __shared__ typename LowTile<T, TILE_W, TILE_H>::Memory sLow;
    int b, a0, e0;
    tileOf((high.W + 1) / 2, (high.H + 1) / 2, b, a0, e0);
    if (pairs) gradientQuads<true, ACCUMULATE, TILE_W, TILE_H>(high, low, C, b, a0, e0, sLow);
    else gradientQuads<false, ACCUMULATE, TILE_W, TILE_H>(high, low, C, b, a0, e0, sLow);
}

/**
 * All coarse levels, one workgroup per image: from 'finest' down to the coarsest level and up again (without an output
 * for 'finest' up to the level below it). The levels below 'finest' live in LDS (dynamic, sized by the host); a copy goes
 * to kept, keptEntries per image, for the adjoint. 32 x 32 x 4 floats: 12 us, the adjoint 32; with a quad of pixels per
 * lane and addresses that may lie anywhere 26 and 58.
 */
template <typename T>
__global__ void __launch_bounds__(PULLPUSH_TAIL_BLOCK) PullPushTailKernel(const PullPushLevel<T> finest, int C, const PullPushTail tail,
                                                                           T* __restrict__ kept, int keptEntries, int topOffset)
{
    using namespace pullpush;
    extern __shared__ __align__(16) unsigned char sMemory[];
    auto* sLevels = (typename LdsLevel<T>::entry*)sMemory;
    const int b = blockIdx.x;
    const TailSteps<T> steps(C);
    const TopLevel<T> top(finest, b, sLevels + topOffset, C, false);
    auto level = [&](int k) { return LdsLevel<T>(sLevels, tail, finest.H, finest.W, C, k, false); };
    ldsBarrier();
    steps.down(top, level(1));
    ldsBarrier();
    for (int k = 1; k + 1 < tail.numLevels; ++k) {
        steps.down(level(k), level(k + 1));
        ldsBarrier();
    }
    for (int k = tail.numLevels - 2; k >= 1; --k) {
        steps.up(level(k), level(k + 1));
        ldsBarrier();
    }
    if (finest.dataPost.p) steps.up(top, level(1));
    for (int i = threadIdx.x; i < keptEntries; i += PULLPUSH_TAIL_BLOCK) kept[static_cast<long long>(b) * keptEntries + i] = sLevels[i];
}

/**
 * The adjoint of all coarse levels, one workgroup per image. ACCUMULATE: 'finest' is the image itself and its gradients are
 * added to. Behind the levels lie what is read of 'finest' and the fills of step A, fillEntries of them.
 */
template <typename T, bool ACCUMULATE>
__global__ void __launch_bounds__(PULLPUSH_TAIL_BLOCK) PullPushGradientTailKernel(const PullPushLevel<T> finest, int C, const PullPushTail tail,
                                                                                   const T* __restrict__ kept, int keptEntries,
                                                                                   const PullPushTail keptTail, int topOffset, int fillOffset, int fillEntries)
{
    using namespace pullpush;
    extern __shared__ __align__(16) unsigned char sMemory[];
    auto* sLevels = (typename LdsLevel<T>::entry*)sMemory;
    auto* sFill = sLevels + fillOffset;
    const int b = blockIdx.x;
    const TailSteps<T> steps(C);
    const TopLevel<T> top(finest, b, sLevels + topOffset, C, true);
    auto level = [&](int k) { return LdsLevel<T>(sLevels, tail, finest.H, finest.W, C, k, true); };
    // the levels of the forward pass; here the gradients of a level follow behind it
    for (int k = 1; k < tail.numLevels; ++k) {
        const T* from = kept + (static_cast<long long>(b) * keptEntries + keptTail.offsets[k]);
        const int entries = (k + 1 < tail.numLevels ? keptTail.offsets[k + 1] : keptEntries) - keptTail.offsets[k];
#pragma unroll 4
        for (int i = threadIdx.x; i < entries; i += PULLPUSH_TAIL_BLOCK) sLevels[tail.offsets[k] + i] = from[i];
    }
    ldsBarrier();
    auto whole = [](const auto& l) { return PullPushRegion{0, l.H, 0, l.W}; };
    steps.gradientUp(top, level(1), whole(level(1)), sFill, fillEntries);
    for (int k = 1; k + 1 < tail.numLevels; ++k) steps.gradientUp(level(k), level(k + 1), whole(level(k + 1)), sFill, fillEntries);
    for (int k = tail.numLevels - 2; k >= 1; --k) {
        steps.template gradient<false>(level(k), level(k + 1), whole(level(k)));
        ldsBarrier();
    }
    steps.template gradient<ACCUMULATE>(top, level(1), whole(top));
}

/**
 * Step B for all levels of a tree but the coarsest, which has its gradients already, in one launch: a workgroup walks from the
 * coarsest to a tile of the finest level, the gradients of the levels in between stay in its LDS (where sizes are odd, a tile needs a
 * pixel more of the next coarser level, which neighbours form twice). 64 x 64 to 512 x 512 pixels of 4 floats: 22 us, with a launch
 * each 45. Bound by the chain of a step, 1.5 to 2 us whatever the size; a level of 1024 x 1024 is better off with a launch of its own (18 us, within the
 * tree 27).
 */
template <typename T>
__global__ void __launch_bounds__(PULLPUSH_TAIL_BLOCK) PullPushGradientTreeKernel(const PullPushTree<T> tree, int C)
{
    using namespace pullpush;
    extern __shared__ __align__(16) unsigned char sMemory[];
    auto* sTiles = (typename LdsLevel<T>::entry*)sMemory;
    const TailSteps<T> steps(C);
    int b;
    const int H = tree.levels[0].H, W = tree.levels[0].W;   // halved from level to level, rounding down
    const PullPushRegion finest = treeTile(H, W, tree.tile, b);
    auto region = [&](int k) {   // of level k: the windows that the pixels of the level above lie in
        PullPushRegion r = finest;
        for (int i = 0; i < k; ++i)
            r = {max((r.y0 >> 1) - ((H >> i) & 1), 0), min(((r.y1 - 1) >> 1) + 1, H >> (i + 1)), max((r.x0 >> 1) - ((W >> i) & 1), 0),
                 min(((r.x1 - 1) >> 1) + 1, W >> (i + 1))};
        return r;
    };
    auto tile = [&](int k) { return LdsTile<T>(treeMemory(sTiles, tree, C, k), region(k)); };
    const int last = tree.count - 2;
    if (last == 0) {
        steps.template gradient<false>(GlobalHigh<T>(tree.levels[0], b), GlobalLow<T>(tree.levels[1], b), finest);
        return;
    }
    steps.template gradient<false>(GradientTileHigh<T>(tree.levels[last], b, tile(last)), GlobalLow<T>(tree.levels[last + 1], b), region(last));
    for (int k = last - 1; k >= 1; --k) {
        ldsBarrier();
        steps.template gradient<false>(GradientTileHigh<T>(tree.levels[k], b, tile(k)), GradientTileLow<T>(tree.levels[k + 1], b, tile(k + 1)), region(k));
    }
    ldsBarrier();
    steps.template gradient<false>(GlobalHigh<T>(tree.levels[0], b), GradientTileLow<T>(tree.levels[1], b, tile(1)), finest);
}

/**
 * The way up for all levels of a tree but the coarsest, which is inpainted already, in one launch: as above; a tile needs the
 * neighbours of its pixels on every coarser level, a border that neighbours form twice. 64 x 64 to 512 x 512 pixels of 4 floats: 15 us,
 * with a launch each 23.
 */
template <typename T>
__global__ void __launch_bounds__(PULLPUSH_TAIL_BLOCK) PullPushUpTreeKernel(const PullPushTree<T> tree, int C)
{
    using namespace pullpush;
    extern __shared__ __align__(16) unsigned char sMemory[];
    auto* sTiles = (typename LdsLevel<T>::entry*)sMemory;
    const TailSteps<T> steps(C);
    int b;
    const int H = tree.levels[0].H, W = tree.levels[0].W;   // halved from level to level, rounding down
    const PullPushRegion finest = treeTile(H, W, tree.tile, b);
    auto region = [&](int k) {
        PullPushRegion r = finest;
        for (int i = 0; i < k; ++i)
            r = {max((r.y0 >> 1) - 1, 0), min(((r.y1 - 1) >> 1) + 2, H >> (i + 1)), max((r.x0 >> 1) - 1, 0), min(((r.x1 - 1) >> 1) + 2, W >> (i + 1))};
        return r;
    };
    auto tile = [&](int k) { return LdsTile<T>(treeMemory(sTiles, tree, C, k), region(k)); };
    // (what is owned of level k: sizes are halved rounding down, so the tiles cover all of it)
    auto owned = [&](int k) {
        return PullPushRegion{finest.y0 >> k, (finest.y0 + tree.tile) >> k, finest.x0 >> k, (finest.x0 + tree.tile) >> k};
    };
    const int last = tree.count - 2;
    for (int k = last; k >= 0; --k) {
        const bool keep = k > 0;
        if (k == last) steps.upRegion(GlobalHigh<T>(tree.levels[k], b), GlobalLow<T>(tree.levels[k + 1], b), region(k), owned(k), keep, tile(max(k, 1)));
        else steps.upRegion(GlobalHigh<T>(tree.levels[k], b), InpaintedTileLow<T>(tree.levels[k + 1], tile(k + 1)), region(k), owned(k), keep, tile(max(k, 1)));
        ldsBarrier();
    }
}

/**
 * The way down for all levels of a tree but the finest, which is there already, in one launch: a workgroup forms a tile of the
 * coarsest level and all that it needs of the finer ones (where sizes are odd, windows overlap, and neighbours form a border twice). The
 * tile is counted in pixels of the finest level. 1024 x 1024 to 32 x 32 pixels of 4 floats: 17 us, with a launch each 24.
 */
template <typename T>
__global__ void __launch_bounds__(PULLPUSH_TAIL_BLOCK) PullPushDownTreeKernel(const PullPushTree<T> tree, int C)
{
    using namespace pullpush;
    extern __shared__ __align__(16) unsigned char sMemory[];
    auto* sTiles = (typename LdsLevel<T>::entry*)sMemory;
    const TailSteps<T> steps(C);
    const int last = tree.count - 1;
    int b;
    const int H = tree.levels[0].H, W = tree.levels[0].W;   // halved from level to level, rounding down
    const PullPushRegion coarsest = treeTile(H >> last, W >> last, tree.tile >> last, b);
    auto region = [&](int k) {   // of level k: what the windows of the level below cover
        PullPushRegion r = coarsest;
        for (int i = last - 1; i >= k; --i)
            r = {2 * r.y0, min(2 * r.y1 + ((H >> i) & 1), H >> i), 2 * r.x0, min(2 * r.x1 + ((W >> i) & 1), W >> i)};
        return r;
    };
    auto tile = [&](int k) {
        auto* memory = sTiles;
        for (int i = 1; i < k; ++i) memory += (C + 1) * treeDownSize(tree.tile, last, i) * treeDownSize(tree.tile, last, i);
        return LdsTile<T>(memory, region(k));
    };
    auto owned = [&](int k) {   // the last tile has what is left over
        return PullPushRegion{coarsest.y0 << (last - k), coarsest.y1 == H >> last ? H >> k : coarsest.y1 << (last - k), coarsest.x0 << (last - k),
                              coarsest.x1 == W >> last ? W >> k : coarsest.x1 << (last - k)};
    };
    for (int k = 1; k <= last; ++k) {
        const bool keep = k < last;
        if (k == 1) steps.downRegion(GlobalHigh<T>(tree.levels[0], b), GlobalHigh<T>(tree.levels[1], b), region(1), owned(1), keep, tile(1));
        else steps.downRegion(DownTileHigh<T>(tree.levels[k - 1], tile(k - 1)), GlobalHigh<T>(tree.levels[k], b), region(k), owned(k), keep, tile(min(k, last - 1)));
        ldsBarrier();
    }
}

/**
 * Step A for all levels of a tree but the finest, in one launch: as the way down, where a tile needs a border of one pixel more of the next
 * finer level. fillOffset: where the fills lie in LDS, behind the tiles. 512 x 512 to 32 x 32 pixels of 4 floats in two
 * launches of two steps: 23 us, with a launch each 32.
 */
template <typename T>
__global__ void __launch_bounds__(PULLPUSH_TAIL_BLOCK) PullPushGradientUpTreeKernel(const PullPushTree<T> tree, int C, int fillOffset, int fillEntries)
{
    using namespace pullpush;
    extern __shared__ __align__(16) unsigned char sMemory[];
    auto* sTiles = (typename LdsLevel<T>::entry*)sMemory;
    const TailSteps<T> steps(C);
    const int last = tree.count - 1;
    int b;
    const int H = tree.levels[0].H, W = tree.levels[0].W;   // halved from level to level, rounding down
    const PullPushRegion coarsest = treeTile(H >> last, W >> last, tree.tile >> last, b);
    auto region = [&](int k) {   // of level k: what the gathers of the level below reach
        PullPushRegion r = coarsest;
        for (int i = last - 1; i >= k; --i)
            r = {max(2 * r.y0 - 1, 0), min(2 * r.y1 + 1, H >> i), max(2 * r.x0 - 1, 0), min(2 * r.x1 + 1, W >> i)};
        return r;
    };
    auto tile = [&](int k) {
        auto* memory = sTiles;
        for (int i = 1; i < k; ++i) memory += (C + 1) * treeUpSize(tree.tile, last, i) * treeUpSize(tree.tile, last, i);
        return LdsTile<T>(memory, region(k));
    };
    auto owned = [&](int k) {
        return PullPushRegion{coarsest.y0 << (last - k), coarsest.y1 == H >> last ? H >> k : coarsest.y1 << (last - k), coarsest.x0 << (last - k),
                              coarsest.x1 == W >> last ? W >> k : coarsest.x1 << (last - k)};
    };
    for (int k = 1; k <= last; ++k) {
        const UpTileLow<T> low(tree.levels[k], b, owned(k), k < last, tile(max(min(k, last - 1), 1)));
        if (k == 1) steps.gradientUp(GlobalHigh<T>(tree.levels[0], b), low, region(1), sTiles + fillOffset, fillEntries);
        else steps.gradientUp(UpTileHigh<T>(tree.levels[k - 1], b, tile(k - 1)), low, region(k), sTiles + fillOffset, fillEntries);
    }
}

namespace pullpush
{
/** Offsets of the idx-th entry (row-major over dst's sizes) in dst and src. */
template <typename D, typename S, int N>
__device__ __forceinline__ void offsetsOf(long long idx, const TensorAccessor<D, N>& dst, const TensorAccessor<S, N>& src,
                                          long long& od, long long& os)
{
    od = 0;
    os = 0;
#pragma unroll
    for (int k = N - 1; k >= 0; --k) {
        const long long c = idx % dst.sizes_[k];
        idx /= dst.sizes_[k];
        od += c * dst.strides_[k];
        os += c * src.strides_[k];
    }
}
} // namespace pullpush

/** dst += src for tensors of 3 or 4 dimensions (the coarsest pyramid level passes its gradients through). */
template <typename T, int N>
__global__ void __launch_bounds__(256) PullPushAddKernel(long long numel, TensorAccessor<T, N> dst, const TensorAccessor<const T, N> src)
{
    for (long long idx = blockIdx.x * static_cast<long long>(blockDim.x) + threadIdx.x; idx < numel;
         idx += static_cast<long long>(blockDim.x) * gridDim.x)
    {
        long long od, os;
        pullpush::offsetsOf(idx, dst, src, od, os);
        dst.data_[od] += src.data_[os];
    }
}

/** dst = src (zero if src has no data) for tensors of any strides (an image of one row or column is its own inpainting). */
template <typename T, int N>
__global__ void __launch_bounds__(256) PullPushCopyKernel(long long numel, TensorAccessor<T, N> dst, const TensorAccessor<const T, N> src)
{
    for (long long idx = blockIdx.x * static_cast<long long>(blockDim.x) + threadIdx.x; idx < numel;
         idx += static_cast<long long>(blockDim.x) * gridDim.x)
    {
        long long od, os;
        pullpush::offsetsOf(idx, dst, src, od, os);
        dst.data_[od] = src.data_ ? src.data_[os] : T(0);
    }
}

QUICKMLP_KERNEL_NAMESPACE_END
