// Parameter gradients of a dense single-level grid for a batch that is sorted by grid slab (point_order.h):
// no records at all. The nodes of the grid are shared out by the two sorted coordinates: owner (o0, o1) holds
// the nodes whose first two indices lie in [o0 * CPS, (o0 + 1) * CPS) x [o1 * CPS, (o1 + 1) * CPS) (CPS: cells
// per slab and coordinate) and every index of the other coordinates -- a "column" of the table whose sums fit
// the LDS (a 4-D grid of 32 nodes per coordinate with 8 features, CPS = 1: 32 x 32 x 8 sums of 8 bytes = 64 KiB).
// A point of slab (a0, a1) touches nodes of the owners (a0 | a0 + 1, a1 | a1 + 1) only, so the workgroup of
// an owner walks the points of the up to four slabs (o0 - 1 | o0, o1 - 1 | o1) -- two runs of the sorted batch --
// and adds, of every point, the corners that it owns: 64-bit fixed-point sums in LDS as in the slice kernel
// (grid_gradient.h), added to the gradient tensor once at the end (atomics of 16 neighbouring floats per request,
// 0.5 M requests for the grid above). Every point is read by four workgroups (32 bytes from the L2 each time); in
// return the 2^(D-1) records of 16 + 2 F bytes per point are neither written nor read, nor sorted into buckets.
//   GridGradientColumnsPlan    one workgroup: slab totals of the sort -> slab starts; per owner the number of
//                              points it visits and from it the work items (an owner whose slabs hold more than
//                              PART_POINTS points is split over several workgroups, which then add their sums
//                              with atomics: a batch that crowds into few slabs still uses the whole device);
//   GridGradientColumnsKernel  one workgroup per work item, as above. The workgroup whose owner indices equal
//                              the slab of a point (its home) also adds the grid's share of the gradient with
//                              respect to the input, from a gather of all corners as in the records kernel, and
//                              adds all corners of points that do not fit the scheme with atomics on the
//                              gradient tensor: points outside the box (extrapolated with weights beyond one,
//                              NaN coordinates; the fixed-point scale counts on weights of at most one), points
//                              whose adjoint is not finite, and points whose cell lies in another slab than
//                              the sort's slab arithmetic put them (a coordinate within rounding of a slab
//                              boundary, or on the upper border).
// Measured on the dense 4-D grid above, 2^21 points: 150 + 7 us where the records and slice kernels take 281 + 154 us.
// The loop over the points is short of two things at once: vector instructions (73 % of the time before the last of the steps
// below) and 268 M additions in LDS, of which ds_add_u64 takes 6.4 lanes per clock and compute unit (entries at random,
// features rotated; 4.5 with all addresses at random, 7.7 side by side): 68 us. The input gradients take 32, writing the
// sums back 8. Hence few instructions per addition: a term is one v_fma_f64 (GridGradientSlices::toFixed) and a subtraction, the corners
// along the unsorted coordinates lie at constant distances (the address of one serves all), features change places two to a
// register, and a lane's rows are found by adding to a pointer, instead of integer products, an address per addition and a
// choice among all features: 168 -> 150 us, together with adjoints scanned 8 points per load, and the input gradients' loads
// one point ahead and as rows of four floats. (Half of the workgroups starting with the input gradients, so that two of a
// compute unit want different things: no gain.)
//
// Replaces, for such batches, the atomicAdd of src_cpp/include/qmlp/kernels/encoding_hashgrid.cuh:117-166,345-369
// of the reference.

#include <qmlp/kernels/common.h>
#include <qmlp/kernels/encoding_hashgrid.h>
#include <qmlp/kernels/grid_gradient.h>
#include <qmlp/kernels/point_order_key.h>

QUICKMLP_KERNEL_NAMESPACE_BEGIN

/** One workgroup of GridGradientColumnsKernel: part `part` of `parts` of the points that owner (owner0, owner1) visits. */
struct GridGradientColumnItem
{
    int owner0;
    int owner1;
    int part;
    int parts;
};

constexpr int GRID_GRADIENT_COLUMNS_MAX_SLABS = 1024;   // as POINT_ORDER_MAX_SLABS
/** Points per work item from which an owner is split (four average slabs of 2^21 points in 31 x 31 slabs: 8.7 K). */
constexpr int GRID_GRADIENT_COLUMNS_PART_POINTS = 24 * 1024;

template <typename Cfg, int CPS>
struct GridGradientColumns
{
    typedef EncodingHashGrid<Cfg> Grid;
    typedef typename Grid::param_t param_t;
    static constexpr int D = Grid::D;
    static constexpr int F = Grid::F;
    static constexpr int NC = Grid::NC;
    static_assert(Cfg::Levels == 1 && !Cfg::hashed[0] && D >= 2, "one dense level of two or more dimensions");
    static constexpr int R = Cfg::resolution[0];                       // nodes per coordinate
    static constexpr int REST = static_cast<int>(detail::upow(static_cast<unsigned>(R), D - 2));   // nodes of the coordinates from 2 on
    static constexpr int OWNERS = (R + CPS - 1) / CPS;                 // per sorted coordinate
    static constexpr int COLUMN_FLOATS = REST * F;                     // all nodes that share their first two indices
    static constexpr int LOCAL_FLOATS = CPS * CPS * COLUMN_FLOATS;     // sums of one owner

    /** Where an owner keeps feature 0 of node (n0, n1, rest), rest = sum over d >= 2 of n_d R^(D-1-d). */
    __device__ __forceinline__ static int localElement(int n0, int n1, unsigned rest, int owner0, int owner1)
    {
        return (((n0 - owner0 * CPS) * CPS + (n1 - owner1 * CPS)) * REST + static_cast<int>(rest)) * F;
    }

    /** The element of the gradient table that local sum `local` of an owner stands for; valid: the node exists. */
    __device__ __forceinline__ static unsigned globalElement(int local, int owner0, int owner1, bool& valid)
    {
        const int column = local / COLUMN_FLOATS, within = local % COLUMN_FLOATS;
        const int n0 = owner0 * CPS + column / CPS, n1 = owner1 * CPS + column % CPS;
        valid = n0 < R && n1 < R;
        return static_cast<unsigned>(Cfg::memoryOffset[0])
            + (static_cast<unsigned>(n0) * static_cast<unsigned>(R) + static_cast<unsigned>(n1)) * static_cast<unsigned>(COLUMN_FLOATS)
            + static_cast<unsigned>(within);
    }

    /** Entries of the table around one slab: the nodes (a * CPS .. (a + 1) * CPS) in both sorted coordinates, all others. */
    static constexpr int REGION_NODES = CPS + 1;
    static constexpr int REGION_ENTRIES = REGION_NODES * REGION_NODES * REST;
    static constexpr int REGION_BYTES = REGION_ENTRIES * F * static_cast<int>(sizeof(typename Cfg::table_t));
    static constexpr int LDS_BYTES = ((LOCAL_FLOATS * 8 > REGION_BYTES ? LOCAL_FLOATS * 8 : REGION_BYTES) + 15) / 16 * 16;

    /** Place of node (n0, n1, rest) in the staged region of slab (a0, a1), in entries; valid: the node lies inside it. */
    __device__ __forceinline__ static int regionEntry(int n0, int n1, unsigned rest, int a0, int a1, bool& valid)
    {
        const int l0 = n0 - a0 * CPS, l1 = n1 - a1 * CPS;
        valid = l0 >= 0 && l0 < REGION_NODES && l1 >= 0 && l1 < REGION_NODES;
        return (l0 * REGION_NODES + l1) * REST + static_cast<int>(rest);
    }

    /** The position of the point of a row of the inputs in the unit box, as every kernel of the grid computes it. */
    __device__ __forceinline__ static void loadPosition(const float* __restrict__ row, int stride, const param_t& params,
                                                        bool rowsOfFloat4, float (&pos)[D])
    {
#pragma clang fp contract(off)
        float in[D];
        if (D == 4 && rowsOfFloat4) {
            const float4 v = *reinterpret_cast<const float4*>(row + Cfg::Start);
            in[0] = v.x, in[1 % D] = v.y, in[2 % D] = v.z, in[3 % D] = v.w;
        } else {
#pragma unroll
            for (int d = 0; d < D; ++d)
                in[d] = row[static_cast<long long>(d + Cfg::Start) * stride];
        }
#pragma unroll
        for (int d = 0; d < D; ++d) pos[d] = (in[d] - params.boundingBoxMin[d]) * params.boundingBoxInvSize[d];
    }

    /** Node indices of corner c (bit d: upper in dimension d) in the two sorted coordinates, and the rest of its index. */
    __device__ __forceinline__ static void cornerNode(const typename Grid::LevelSetup& s, int c, int& n0, int& n1, unsigned& rest)
    {
        constexpr unsigned M0 = detail::upow(static_cast<unsigned>(R), D - 1), M1 = detail::upow(static_cast<unsigned>(R), D - 2);
        n0 = static_cast<int>(((c & 1) ? s.termH[0] : s.termL[0]) / M0);
        n1 = static_cast<int>(((c & 2) ? s.termH[1] : s.termL[1]) / M1);
        rest = 0u;
#pragma unroll
        for (int d = 2; d < D; ++d) rest += ((c >> d) & 1) ? s.termH[d] : s.termL[d];
    }

    /** The node indices alone of the corners with bits 0 and 1 of c. */
    __device__ __forceinline__ static void sortedNode(const typename Grid::LevelSetup& s, int c, int& n0, int& n1)
    {
        n0 = static_cast<int>(((c & 1) ? s.termH[0] : s.termL[0]) / stride(0));
        n1 = static_cast<int>(((c & 2) ? s.termH[1] : s.termL[1]) / stride(1));
    }
    /** Entries between neighbours along a coordinate. */
    __device__ __host__ static constexpr unsigned stride(int d) { return detail::upow(static_cast<unsigned>(R), D - 1 - d); }
    static_assert(R >= 2 || D == 2, "two nodes along the other coordinates");
    /** Entries from the node that is the lower one along all other coordinates to that of bits `others` (bit d - 2: upper along d). */
    __device__ __host__ static constexpr int upperNodes(int others)
    {
        unsigned n = 0;
        for (int d = 2; d < D; ++d) n += ((others >> (d - 2)) & 1) ? stride(d) : 0u;
        return static_cast<int>(n);
    }

    /** The cell of the point in the two sorted coordinates, as the grid computes it. */
    __device__ __forceinline__ static void cell(const typename Grid::LevelSetup& s, int& c0, int& c1)
    {
        constexpr unsigned M0 = detail::upow(static_cast<unsigned>(R), D - 1), M1 = detail::upow(static_cast<unsigned>(R), D - 2);
        c0 = static_cast<int>(s.termL[0] / M0);
        c1 = static_cast<int>(s.termL[1] / M1);
    }

    __device__ __forceinline__ static bool insideBox(const typename Grid::LevelSetup& s)
    {
        bool inside = true;
#pragma unroll
        for (int d = 0; d < D; ++d) inside = inside && s.f[d] >= 0.f && s.f[d] <= 1.f;
        return inside;
    }

    /** The adjoints of a point, two halves to a word. */
    static constexpr int ADJOINT_WORDS = (F + 1) / 2;
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

    /** Whether none of the halves is NaN or infinite. */
    template <int N>
    __device__ __forceinline__ static bool finiteHalves(const unsigned (&words)[N])
    {
        u16x2 largest = {0, 0};
#pragma unroll
        for (int i = 0; i < N; ++i) largest = __builtin_elementwise_max(largest, __builtin_bit_cast(u16x2, words[i] & 0x7fff7fffu));
        return largest[0] < 0x7c00u && largest[1] < 0x7c00u;
    }

    __device__ __forceinline__ static float adjointAt(const unsigned (&words)[ADJOINT_WORDS], int i)
    {
        return static_cast<float>(__builtin_bit_cast(f16, static_cast<unsigned short>(words[i / 2] >> (16 * (i % 2)))));
    }

    /** The feature that a lane takes in a step. */
    __device__ __forceinline__ static int rotatedFeature(int step, int lane)
    {
        return (F & (F - 1)) == 0 ? ((step + lane) & (F - 1)) : ((step + lane % F) % F);
    }
    /** The adjoints in the order of rotatedFeature(): a power of two of them is moved by 4, 2 and 1 places, two in a word at a time. */
    __device__ __forceinline__ static void rotate(const unsigned (&words)[ADJOINT_WORDS], int lane, float (&rotated)[F])
    {
        if constexpr ((F & (F - 1)) == 0 && F > 1) {
            unsigned w[ADJOINT_WORDS];
#pragma unroll
            for (int i = 0; i < ADJOINT_WORDS; ++i) w[i] = words[i];
#pragma unroll
            for (int places = F / 2; places > 0; places /= 2) {
                unsigned moved[ADJOINT_WORDS];
                const unsigned move = (lane & places) ? ~0u : 0u;   // (as bits: selections become a search for an index)
#pragma unroll
                for (int i = 0; i < ADJOINT_WORDS; ++i) {
                    if (places >= 2) moved[i] = (w[(i + places / 2) % ADJOINT_WORDS] & move) | (w[i] & ~move);
                    else moved[i] = __builtin_amdgcn_alignbit(w[(i + 1) % ADJOINT_WORDS], w[i], (lane & 1) * 16);
                }
#pragma unroll
                for (int i = 0; i < ADJOINT_WORDS; ++i) w[i] = moved[i];
            }
#pragma unroll
            for (int i = 0; i < F; ++i) rotated[i] = adjointAt(w, i);
        } else {
#pragma unroll
            for (int step = 0; step < F; ++step) {
                const int i = rotatedFeature(step, lane);
                float a = adjointAt(words, 0);
#pragma unroll
                for (int k = 1; k < F; ++k) a = i == k ? adjointAt(words, k) : a;
                rotated[step] = a;
            }
        }
    }

    template <int N> struct Constant { static constexpr int value = N; };

    /**
     * The largest magnitude (bits without the sign) among the adjoints of points [begin, end) that are finite; first: the first
     * of their channels in tile 0. The adjoints of 64 points are F * 128 bytes side by side: a lane takes 8 points of a channel.
     */
    template <int ROW_CHANNELS, int BLOCK>
    __device__ __forceinline__ static unsigned largestAdjoint(const f16* __restrict__ first, int begin, int end, int lane)
    {
        typedef unsigned u32x4 __attribute__((ext_vector_type(4), aligned(4)));
        constexpr int CHUNKS = F * (TILE_POINTS / 8);   // of a tile
        u16x2 largest = {0, 0};
        if (begin >= end) return 0u;
        const int firstTile = begin / TILE_POINTS;
        const int chunks = ((end - 1) / TILE_POINTS - firstTile + 1) * CHUNKS;
        // GUARDED: without what lies behind the last chunk for a whole wavefront
        auto scan = [&](int i0, auto ahead, auto guarded) {
            constexpr int AHEAD = decltype(ahead)::value;
            constexpr bool GUARDED = decltype(guarded)::value != 0;
            const int wave0 = __builtin_amdgcn_readfirstlane(i0);
            u32x4 v[AHEAD];
#pragma unroll
            for (int k = 0; k < AHEAD; ++k) {
                if (GUARDED && wave0 + k * BLOCK >= chunks) continue;
                const int i = min(i0 + k * BLOCK, chunks - 1);   // (the last one again)
                v[k] = *reinterpret_cast<const u32x4*>(first + static_cast<long long>(firstTile + i / CHUNKS) * (ROW_CHANNELS * TILE_POINTS)
                                                       + i % CHUNKS * 8);
            }
#pragma unroll
            for (int k = 0; k < AHEAD; ++k) {
                if (GUARDED && wave0 + k * BLOCK >= chunks) continue;
                const int i = min(i0 + k * BLOCK, chunks - 1);
                const int p = (firstTile + i / CHUNKS) * TILE_POINTS + i % (TILE_POINTS / 8) * 8;
                unsigned words[4] = {v[k][0], v[k][1], v[k][2], v[k][3]};
                if (p < begin || p + 8 > end || !finiteHalves(words)) {
                    // others' points, and adjoints that are not finite (their points take the atomics), don't count
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        if (p + j < begin || p + j >= end || ((words[j / 2] >> (16 * (j % 2))) & 0x7c00u) == 0x7c00u)
                            words[j / 2] &= j % 2 ? 0xffffu : 0xffff0000u;
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) largest = __builtin_elementwise_max(largest, __builtin_bit_cast(u16x2, words[j] & 0x7fff7fffu));
            }
        };
        // So many loads of a lane at a time while a run has more than half of them for it (2^21 points of 8 features in 31 x 31 slabs: ten on
        // average; fewer features have fewer, and need the registers for more wavefronts), then up to half, and none for wavefronts that the
        // run does not reach: the workgroups of 2^20 points in 32 x 32 slabs have one or two (128^3 nodes x 2: the kernel 34 us, 58 with
        // ten whatever the run).
        constexpr int MANY = F >= 8 ? 10 : 4;
        int from = 0;
#pragma unroll 1
        for (; chunks - from > MANY / 2 * BLOCK; from += MANY * BLOCK) scan(from + lane, Constant<MANY>{}, Constant<0>{});
        if (from < chunks) scan(from + lane, Constant<MANY / 2>{}, Constant<1>{});
        return max(static_cast<unsigned>(largest[0]), static_cast<unsigned>(largest[1]));
    }

    /** The runs of the sorted batch that owner (o0, o1) visits: run r covers the slabs (a0, o1 - 1 | o1), a0 = o0 - 1 + r. */
    struct Runs
    {
        int begin[2], middle[2], end[2];   // points [begin, middle) lie in slab (a0, o1 - 1), [middle, end) in (a0, o1)
        __device__ __forceinline__ int points() const { return (end[0] - begin[0]) + (end[1] - begin[1]); }
    };
    __device__ __forceinline__ static Runs runsOf(int owner0, int owner1, const int* __restrict__ starts, int slabs0, int slabs1)
    {
        Runs runs;
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int a0 = owner0 - 1 + r;
            runs.begin[r] = runs.middle[r] = runs.end[r] = 0;
            if (a0 < 0 || a0 >= slabs0) continue;
            const int lo = owner1 - 1, hi = owner1;   // slabs of the second coordinate
            const int first = a0 * slabs1 + max(lo, 0), last = a0 * slabs1 + min(hi, slabs1 - 1);
            if (first > last) continue;
            runs.begin[r] = starts[first];
            runs.end[r] = starts[last + 1];
            // the boundary between slab lo and slab hi (all points belong to one of them if the other does not exist)
            runs.middle[r] = lo < 0 ? runs.begin[r] : hi > slabs1 - 1 ? runs.end[r] : starts[a0 * slabs1 + hi];
        }
        return runs;
    }
};

/**
 * totals: points per slab (slabs0 * slabs1 <= 1024 values, as PointOrderScan leaves them). Writes starts
 * (slabs + 1 values), the work items and their number. One workgroup of 1024 threads, as long as its chain of steps: 5.3 us, 7 with items
 * counted by an atomic in LDS, a lane at a time, and sums over the lanes by way of LDS.
 */
template <typename Cfg, int CPS>
__global__ void __launch_bounds__(1024) GridGradientColumnsPlan(
    int numel, const int* __restrict__ totals, int slabs0, int slabs1, int* __restrict__ starts,
    GridGradientColumnItem* __restrict__ items, int* __restrict__ itemCount, int maxItems)
{
    typedef GridGradientColumns<Cfg, CPS> Impl;
    __shared__ int sScan[GRID_GRADIENT_COLUMNS_MAX_SLABS + 1];
    __shared__ int sWave[16];
    const int tid = threadIdx.x;
    const int slabs = slabs0 * slabs1;
    const int lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    // the values of the lanes in front of this one, and those of all lanes
    auto scan = [&](int value, int& all) {
        const int inclusive = waveInclusiveScan(value);
        __syncthreads();   // (sWave of the scan before)
        if (lane == 63) sWave[wave] = inclusive;
        __syncthreads();
        const int sums = waveInclusiveScan(lane < 16 ? sWave[lane] : 0);
        all = __builtin_amdgcn_readlane(sums, 15);
        return (wave > 0 ? __builtin_amdgcn_readlane(sums, wave - 1) : 0) + inclusive - value;
    };
    int points;
    sScan[tid] = scan(tid < slabs ? totals[tid] : 0, points);
    if (tid == 1023) sScan[1024] = points;
    __syncthreads();
    if (tid < slabs) starts[tid] = sScan[tid];
    if (tid == 0) starts[slabs] = numel;
    // work items, in the order of the owners
    int itemsBefore = 0;
    for (int first = 0; first < Impl::OWNERS * Impl::OWNERS; first += 1024) {
        const int o = first + tid, o0 = o / Impl::OWNERS, o1 = o % Impl::OWNERS;
        // (the starts are read from LDS: the global copy is not visible to the whole workgroup yet; the totals
        // beyond the last slab are zero, so sScan[slabs] is the number of all points)
        const int visited = o < Impl::OWNERS * Impl::OWNERS ? Impl::runsOf(o0, o1, sScan, slabs0, slabs1).points() : 0;
        const int parts = (visited + GRID_GRADIENT_COLUMNS_PART_POINTS - 1) / GRID_GRADIENT_COLUMNS_PART_POINTS;
        int all;
        const int at = itemsBefore + scan(parts, all);
        for (int part = 0; part < parts; ++part)
            if (at + part < maxItems) items[at + part] = GridGradientColumnItem{o0, o1, part, parts};
        itemsBefore += all;
    }
    if (tid == 0) *itemCount = min(itemsBefore, maxItems);
}

/**
 * \tparam CPS cells per slab and sorted coordinate
 * \tparam ROW_CHANNELS, CHANNEL_OFFSET the tile layout of the adjoint of the encoded rows, as for the records kernel
 * \tparam INPUT_GRADIENTS 0: none; 1: from a gather of all corners; 2: from the position derivatives of the forward pass
 * inputs: the rows of the batch in sorted order; starts, items, itemCount: as GridGradientColumnsPlan wrote them.
 * Launched with as many workgroups as there can be work items; those beyond itemCount leave at once.
 * Dynamic LDS: GridGradientColumns::LDS_BYTES (the sums of an owner, then the entries of the table around its slab).
 */
template <typename Cfg, int CPS, int ROW_CHANNELS, int CHANNEL_OFFSET, int INPUT_GRADIENTS, int BLOCK>
__global__ void __launch_bounds__(BLOCK)
    // two workgroups per compute unit where the features of all corners take at most half of the 128 registers that this leaves
    __attribute__((amdgpu_waves_per_eu(EncodingHashGrid<Cfg>::NC * Cfg::Features * sizeof(typename Cfg::table_t) <= 256 ? 4 : 1)))
GridGradientColumnsKernel(
    int numel, const Tensor2Read<float> inputs, const half* __restrict__ adjEncodedH,
    const HashGridParams<typename Cfg::table_t, Cfg::Dim> params, const int* __restrict__ starts, int slabs0, int slabs1,
    const GridGradientColumnItem* __restrict__ items, const int* __restrict__ itemCount, Tensor2RW<float> adjInputs,
    const void* __restrict__ derivativesV)
{
    typedef GridGradientColumns<Cfg, CPS> Impl;
    typedef EncodingHashGrid<Cfg> Grid;
    typedef GridGradientRecords<Cfg, ROW_CHANNELS, CHANNEL_OFFSET, 8192, 256> Records;   // its gathers for the input gradients
    typedef GridGradientSlices<Cfg, 8192, false> Fixed;                                         // its fixed-point arithmetic
    constexpr int D = Cfg::Dim, F = Cfg::Features, NC = Grid::NC;
    extern __shared__ __align__(16) unsigned char sMemory[];
    long long* sSums = reinterpret_cast<long long*>(sMemory);
    __shared__ int sMaxBits;
    if (static_cast<int>(blockIdx.x) >= *itemCount) return;
    const GridGradientColumnItem item = items[blockIdx.x];
    const int tid = threadIdx.x;
    const f16* __restrict__ adjEncoded = reinterpret_cast<const f16*>(adjEncodedH);
    const typename Impl::Runs runs = Impl::runsOf(item.owner0, item.owner1, starts, slabs0, slabs1);

    // this part's share of both runs
    int begin[2], end[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const long long length = runs.end[r] - runs.begin[r];
        begin[r] = runs.begin[r] + static_cast<int>(length * item.part / item.parts);
        end[r] = runs.begin[r] + static_cast<int>(length * (item.part + 1) / item.parts);
        // (slab starts are sums of counts of this batch: never outside of it)
        begin[r] = max(0, min(begin[r], numel));
        end[r] = max(begin[r], min(end[r], numel));
    }

    // rows of four floats that lie side by side: one load
    const bool rowsOfFloat4 = D == 4 && Cfg::Start % 4 == 0 && inputs.strides_[1] == 1 && inputs.strides_[0] % 4 == 0
        && reinterpret_cast<unsigned long long>(inputs.data_) % 16 == 0;

    for (int i = tid; i < Impl::LOCAL_FLOATS; i += BLOCK) sSums[i] = 0;
    if (tid == 0) sMaxBits = 0;
    __syncthreads();

    // the largest adjoint among the points of this work item: the scale of the fixed-point sums
    {
        unsigned maxBits = 0u;
#pragma unroll 1
        for (int r = 0; r < 2; ++r)
            maxBits = max(maxBits, Impl::template largestAdjoint<ROW_CHANNELS, BLOCK>(adjEncoded + CHANNEL_OFFSET * TILE_POINTS, begin[r], end[r], tid));
        if (maxBits != 0u) atomicMax(&sMaxBits, static_cast<int>(maxBits));
    }
    __syncthreads();
    const unsigned maxBits = static_cast<unsigned>(sMaxBits);
    const int maxExponent = static_cast<int>(maxBits >> 10) - 14;   // |adjoint| < 2^maxExponent
    const long long terms = static_cast<long long>(NC) * max(1, (end[0] - begin[0]) + (end[1] - begin[1]));
    const int termsLog2 = 64 - __builtin_clzll(static_cast<unsigned long long>(terms));
    // A term is weight x adjoint in units of 2^-scaleExponent, formed in double precision and rounded there; the sum of all
    // terms that can meet in one element stays below 2^62.
    const int scaleExponent = min(Fixed::FIXED_BITS, 62 - termsLog2) - maxExponent;
    const double scale = ldexp(1.0, scaleExponent);
    float* __restrict__ gradients = params.parametersBackward;

#pragma unroll 1
    for (int r = 0; r < 2; ++r) {
        const int a0 = item.owner0 - 1 + r;
        // (the position and the adjoints of a lane's next point are loaded before it works on this one: with four
        // wavefronts per SIMD nothing else hides the latency of the loads)
        float nextPos[D];
        unsigned nextAdj[Impl::ADJOINT_WORDS];
        static_assert(BLOCK % TILE_POINTS == 0, "a lane's points lie at the same place of their tiles");
        const float* nextRow = inputs.data_ + static_cast<long long>(begin[r] + tid) * inputs.strides_[0];
        const f16* nextAdjRow = adjEncoded + static_cast<long long>((begin[r] + tid) / TILE_POINTS) * (ROW_CHANNELS * TILE_POINTS)
            + CHANNEL_OFFSET * TILE_POINTS + (begin[r] + tid) % TILE_POINTS;
        auto loadPoint = [&]() {
            Impl::loadPosition(nextRow, inputs.strides_[1], params, rowsOfFloat4, nextPos);
#pragma unroll
            for (int i = 0; i < Impl::ADJOINT_WORDS; ++i) {
                f16x2 two = {nextAdjRow[2 * i * TILE_POINTS], f16(0)};
                if (2 * i + 1 < F) two[1] = nextAdjRow[(2 * i + 1) * TILE_POINTS];
                nextAdj[i] = __builtin_bit_cast(unsigned, two);
            }
            nextRow += static_cast<long long>(BLOCK) * inputs.strides_[0];
            nextAdjRow += BLOCK * ROW_CHANNELS;
        };
        if (begin[r] + tid < end[r]) loadPoint();
#pragma unroll 1
        for (int p = begin[r] + tid; p < end[r]; p += BLOCK) {
            const int a1 = p < runs.middle[r] ? item.owner1 - 1 : item.owner1;
            const bool home = a0 == item.owner0 && a1 == item.owner1;
            float pos[D];
            unsigned adjWords[Impl::ADJOINT_WORDS];
#pragma unroll
            for (int d = 0; d < D; ++d) pos[d] = nextPos[d];
#pragma unroll
            for (int i = 0; i < Impl::ADJOINT_WORDS; ++i) adjWords[i] = nextAdj[i];
            if (p + BLOCK < end[r]) loadPoint();
            const typename Grid::LevelSetup s = Grid::setupLevel(0, pos);
            int c0, c1;
            Impl::cell(s, c0, c1);
            // Points that do not fit the scheme -- the same verdict in every workgroup that visits the point: outside
            // the box, in a cell of another slab than the sort's, or with an adjoint that is not finite (NaN and
            // infinity have no fixed-point form and reach the gradients through the atomics of the point's home).
            const bool regular = Impl::finiteHalves(adjWords) && Impl::insideBox(s) && c0 / CPS == a0 && c1 / CPS == a1;
            if (!regular && !home) continue;
            if (regular) {
                if (maxBits != 0u) {
                    // neighbouring lanes take the features in rotated order (an entry starts at a multiple of
                    // 8 F bytes: lanes that all add the same feature would meet on a few LDS banks)
                    float rotatedAdj[F];
                    Impl::rotate(adjWords, tid, rotatedAdj);
                    double rotated[F];
#pragma unroll
                    for (int i = 0; i < F; ++i) rotated[i] = static_cast<double>(rotatedAdj[i]);
                    // The corners of the pairs of sorted coordinates that are this owner's. Along the other
                    // coordinates the upper one is the next node: on the upper border (both are the last node) the
                    // pair is taken as the two last, with all of the weight on the upper.
                    typename Grid::LevelSetup t = s;
                    unsigned rest = 0u;
#pragma unroll
                    for (int d = 2; d < D; ++d) {
                        const bool last = s.termL[d] == s.termH[d];
                        t.f[d] = last ? 1.f : s.f[d];
                        rest += last ? s.termL[d] - Impl::stride(d) : s.termL[d];
                    }
#pragma unroll
                    for (int sorted = 0; sorted < 4; ++sorted) {
                        int n0, n1;
                        Impl::sortedNode(s, sorted, n0, n1);
                        if (n0 / CPS != item.owner0 || n1 / CPS != item.owner1) continue;
                        long long* sums = sSums + Impl::localElement(n0, n1, rest, item.owner0, item.owner1);
#pragma unroll
                        for (int others = 0; others < NC / 4; ++others) {
                            const double w = static_cast<double>(Grid::cornerWeight(t, sorted | (others << 2))) * scale;
#pragma unroll
                            for (int step = 0; step < F; ++step)
                                Fixed::ldsAddFixed(sums + Impl::rotatedFeature(step, tid) + Impl::upperNodes(others) * F, Fixed::toFixed(rotated[step], w));
                        }
                    }
                }
            } else {
                // home of a point that does not fit the scheme: all of its corners, with atomics
#pragma unroll 1
                for (int c = 0; c < NC; ++c) {
                    const float w = Grid::cornerWeight(s, c);
                    const unsigned element = Grid::cornerOffset(0, s, c);
#pragma unroll 1
                    for (int i = 0; i < F; ++i) {
                        const unsigned word = adjWords[i / 2] >> (16 * (i % 2));
                        unsafeAtomicAdd(gradients + element + i, w * static_cast<float>(__builtin_bit_cast(f16, static_cast<unsigned short>(word))));
                    }
                }
            }
        }
    }
    __syncthreads();

    // The sums of this owner, added with atomics (16 neighbouring floats per request): other workgroups may be adding
    // the corners of points that do not fit the scheme to the same elements at this moment, and the parts of a
    // split owner hold sums for the same elements.
    if (maxBits != 0u) {
        for (int i = tid; i < Impl::LOCAL_FLOATS; i += BLOCK) {
            const long long fixed = sSums[i];
            if (fixed == 0) continue;
            bool valid;
            const unsigned element = Impl::globalElement(i, item.owner0, item.owner1, valid);
            if (!valid) continue;
            const float v = static_cast<float>(ldexp(static_cast<double>(fixed), -scaleExponent));
            unsafeAtomicAdd(gradients + element, v);
        }
    }

    if constexpr (INPUT_GRADIENTS != 0) {
        // The grid's share of the gradient with respect to the input, for the points whose slab has the indices of
        // this owner (every point has one such home: a plain read-modify-write of its row). From the position
        // derivatives of the forward pass where it kept them; else from the entries of all corners, as the records
        // kernel gathers them -- but out of the LDS, which the sums have left: the entries around one slab are as
        // many bytes as an owner's sums (half tables) and are copied in with coalesced loads once, instead of
        // 2^D gathers of one entry per point (dense 4-D grid with 8 features, 2^21 points: 96 -> 32 us).
        const int a0 = item.owner0, a1 = item.owner1;
        if (a0 >= slabs0 || a1 >= slabs1) return;   // an owner of border nodes only: no slab of its own
        const int homeBegin = max(begin[1], min(runs.middle[1], end[1])), homeEnd = end[1];
        if (homeBegin >= homeEnd) return;           // (the same for the whole workgroup)
        typedef typename Cfg::table_t table_t;
        table_t* sRegion = reinterpret_cast<table_t*>(sMemory);
        if constexpr (INPUT_GRADIENTS == 1) {
            __syncthreads();   // the sums have been read
            // 16 bytes per load: the entries of one (n0, n1) are REST * F values side by side in the table and in the region
            constexpr int COLUMN_VALUES = Impl::REST * F;
            constexpr int WIDEST = 16 / static_cast<int>(sizeof(table_t));
            constexpr int PER_LOAD = COLUMN_VALUES % WIDEST == 0 ? WIDEST : COLUMN_VALUES % (WIDEST / 2) == 0 ? WIDEST / 2
                : COLUMN_VALUES % (WIDEST / 4) == 0 ? WIDEST / 4 : 1;
            typedef table_t load_t __attribute__((ext_vector_type(PER_LOAD)));
            for (int i = tid; i < Impl::REGION_NODES * Impl::REGION_NODES * (COLUMN_VALUES / PER_LOAD); i += BLOCK) {
                const int column = i / (COLUMN_VALUES / PER_LOAD), within = i % (COLUMN_VALUES / PER_LOAD);
                const int n0 = a0 * CPS + column / Impl::REGION_NODES, n1 = a1 * CPS + column % Impl::REGION_NODES;
                if (n0 < Impl::R && n1 < Impl::R) {
                    const table_t* src = params.parametersForward + Cfg::memoryOffset[0]
                        + (static_cast<long long>(n0) * Impl::R + n1) * COLUMN_VALUES + within * PER_LOAD;
                    *reinterpret_cast<load_t*>(sRegion + column * COLUMN_VALUES + within * PER_LOAD) = *reinterpret_cast<const load_t*>(src);
                }
            }
            __syncthreads();
        }
        const bool gradientRowsOfFloat4 = D == 4 && Cfg::Start % 4 == 0 && adjInputs.strides_[1] == 1 && adjInputs.strides_[0] % 4 == 0
            && reinterpret_cast<unsigned long long>(adjInputs.data_) % 16 == 0;
        auto gradientOf = [&](int q, int d) {
            return adjInputs.data_ + static_cast<long long>(q) * adjInputs.strides_[0] + static_cast<long long>(d + Cfg::Start) * adjInputs.strides_[1];
        };
        // (what a point needs is loaded before the lane works on the point in front of it)
        float nextPos[D], nextGradient[D], nextAdj[F];
        auto loadPoint = [&](int q) {
            Impl::loadPosition(inputs.data_ + static_cast<long long>(q) * inputs.strides_[0], inputs.strides_[1], params, rowsOfFloat4, nextPos);
            if (D == 4 && gradientRowsOfFloat4) {
                const float4 v = *reinterpret_cast<const float4*>(gradientOf(q, 0));
                nextGradient[0] = v.x, nextGradient[1 % D] = v.y, nextGradient[2 % D] = v.z, nextGradient[3 % D] = v.w;
            } else {
#pragma unroll
                for (int d = 0; d < D; ++d) nextGradient[d] = *gradientOf(q, d);
            }
            if constexpr (INPUT_GRADIENTS == 1) {
#pragma unroll
                for (int i = 0; i < F; ++i) nextAdj[i] = static_cast<float>(typename Records::Adjoints{adjEncodedH}(q, CHANNEL_OFFSET + i));
            }
        };
        if (homeBegin + tid < homeEnd) loadPoint(homeBegin + tid);
#pragma unroll 1
        for (int p = homeBegin + tid; p < homeEnd; p += BLOCK) {
            float pos[D], gradient[D], adj[F];
#pragma unroll
            for (int d = 0; d < D; ++d) pos[d] = nextPos[d], gradient[d] = nextGradient[d];
#pragma unroll
            for (int i = 0; i < F; ++i) adj[i] = INPUT_GRADIENTS == 1 ? nextAdj[i] : 0.f;
            if (p + BLOCK < homeEnd) loadPoint(p + BLOCK);
            float adjPos[D];
#pragma unroll
            for (int d = 0; d < D; ++d) adjPos[d] = 0.f;
            if constexpr (INPUT_GRADIENTS == 2) {
                Records::template positionGradientFromDerivatives<0>(
                    p, static_cast<const typename Records::DerivativeChunk*>(derivativesV), typename Records::Adjoints{adjEncodedH}, adjPos);
            } else {
                const typename Grid::LevelSetup s = Grid::setupLevel(0, pos);
                detail::HeldFeatures<F, table_t> held[NC];
                // (a point in a cell of another slab than the sort's -- within rounding of a slab boundary, on the upper
                // border -- may have corners outside the region: it gathers from the table)
                bool staged = true;
                int entry[NC];
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    int n0, n1;
                    unsigned rest;
                    Impl::cornerNode(s, c, n0, n1, rest);
                    bool valid;
                    entry[c] = Impl::regionEntry(n0, n1, rest, a0, a1, valid);
                    staged = staged && valid;
                }
                if (staged) {
#pragma unroll
                    for (int c = 0; c < NC; ++c) held[c].load(sRegion + entry[c] * F);
                } else {
                    Records::template loadHeld<0>(s, params, held);
                }
                Records::template positionGradient<0>(s, held, adj, adjPos);
            }
#pragma unroll
            for (int d = 0; d < D; ++d) gradient[d] += adjPos[d] * params.boundingBoxInvSize[d];
            if (D == 4 && gradientRowsOfFloat4) {
                *reinterpret_cast<float4*>(gradientOf(p, 0)) = make_float4(gradient[0], gradient[1 % D], gradient[2 % D], gradient[3 % D]);
            } else {
#pragma unroll
                for (int d = 0; d < D; ++d) *gradientOf(p, d) = gradient[d];
            }
        }
    }
}

/**
 * Test aid: for every point (one per lane) and corner, the element of the gradient table that the sum stands for
 * to which GridGradientColumnsKernel adds the corner -- through the place in the LDS of the owner of the corner's
 * node and back, as the kernel goes -- and its weight. Slots: corner (bit d: upper in dimension d).
 */
template <typename Cfg, int CPS>
__global__ void __launch_bounds__(256) GridGradientColumnsTraceKernel(
    long long numel, const Tensor2Read<float> inputs, unsigned* __restrict__ indices, float* __restrict__ weights,
    const HashGridParams<typename Cfg::table_t, Cfg::Dim> params)
{
    typedef GridGradientColumns<Cfg, CPS> Impl;
    typedef EncodingHashGrid<Cfg> Grid;
    constexpr int D = Cfg::Dim, NC = Grid::NC;
    for (long long index = blockIdx.x * static_cast<long long>(blockDim.x) + threadIdx.x; index < numel;
         index += static_cast<long long>(blockDim.x) * gridDim.x)
    {
        float pos[D];
        {
#pragma clang fp contract(off)
#pragma unroll
            for (int d = 0; d < D; ++d)
                pos[d] = (inputs.data_[index * inputs.strides_[0] + static_cast<long long>(d + Cfg::Start) * inputs.strides_[1]]
                          - params.boundingBoxMin[d]) * params.boundingBoxInvSize[d];
        }
        const typename Grid::LevelSetup s = Grid::setupLevel(0, pos);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            int n0, n1;
            unsigned rest;
            Impl::cornerNode(s, c, n0, n1, rest);
            const int o0 = n0 / CPS, o1 = n1 / CPS;
            bool valid;
            const unsigned element = Impl::globalElement(Impl::localElement(n0, n1, rest, o0, o1), o0, o1, valid);
            indices[index * NC + c] = valid ? element : 0xffffffffu;
            weights[index * NC + c] = Grid::cornerWeight(s, c);
        }
    }
}

QUICKMLP_KERNEL_NAMESPACE_END
