// Parameter gradients of a grid encoding without a global atomic per contribution: the
// contributions are first written as records, sorted by slice of the gradient table, and a
// workgroup per slice then sums its records in LDS and writes the slice once.
//
// Float atomics on device memory complete at about 21e9 requests per second on the whole
// device wherever the data lives (16e9 measured for atomics of 4 neighbouring floats, also where all
// of a level are issued by one die), and a hashed level offers nothing to combine (a batch of
// random points touches every entry about once). So the scatter of the fused backward kernel
// (EncodingHashGrid::scatterTile, 4.5 requests per point and level) bounds a train step. Here
// the backward kernel only stores the adjoint of the encoded rows. Then
//   GridGradientRecordsKernel  takes a region of consecutive points, one per lane, level by level: for every
//       pair of corners that are neighbours in memory it forms a record (the offsets of the two
//       entries within their slice, their weights, the adjoint of the level's features), sorts the
//       records of the region by the slice of the gradient table they belong to (a slice is a
//       run of 8192 or 16 384 floats, whose 64-bit sums take 64 or 128 KiB of LDS) in LDS, and copies them
//       out as they are: the records of a region and level lie without gaps at a place that is known beforehand,
//       and a row of `places` says where those of each slice begin. (Buckets per slice, in which every workgroup reserved room
//       with an atomic per slice and level: 25 us of atomics, and a batch of unevenly spread points found them full. 16
//       levels, 2^18 points with input gradients from derivatives: 124 -> 82 us, 80 with two barriers per level instead of three.) The levels of a region are shared out over several
//       workgroups. The grid's share of the gradient with respect to the input
//       (what EncodingHashGrid::adjoint computes, operation by operation) comes from the
//       entries of all corners, two that lie side by side with one load, or, where the forward
//       pass kept the derivatives of the features with respect to the position (PositionDerivativeLayout,
//       INPUT_GRADIENTS == 2), as adjoint x derivative from one or two coalesced loads per level; who computes it: see
//       GridGradientRecords::inputGradientsInline. Bound by the memory that
//       the records are written to: 268 MB of them for 2^18 points, with what it reads 400 MB at 5 TB/s, what a copy reaches;
//   GridGradientSlicesKernel   runs one workgroup per work item (level, slice, part of the
//       regions): it streams through its records, a segment in every region, and adds weight * adjoint to the slice in LDS,
//       then writes the slice, or adds it to the gradient tensor (with atomics only for a coarse level, whose
//       few slices receive all records of the level and are shared out over several work items, and for the first entry
//       of a slice, to which the slice in front adds as well). Bound by the memory that the records come from and by its additions in
//       turn: 2^18 points 76 us (52 of them for the records alone, at 5 TB/s, 9 for the stores of 50 MB); one level of 64^3 nodes x 4
//       floats, 2^20 points 33 us on half of the compute units, 25 without the additions. Tensors that hold nothing yet are written:
//       50 MB that nobody zeroes first nor reads again;
//   GridGradientExceptionsKernel   adds, with atomics, what has no record: the points outside of the box and, in hashed levels, upper
//       entries in another slice than the one behind the lower one's.
// The sums in LDS are 64-bit fixed point, added with integer atomics: ds_add_f32 completes one
// lane every three cycles on this hardware (0.32 lanes per clock and CU measured, whatever the
// addresses), ds_add_u64 3.5 lanes per clock. The scale is a power of two chosen per launch from the
// largest adjoint of the batch (which the records kernel finds on its way) and the number of
// records, such that no sum can overflow: at least 35 bits remain below the largest possible
// contribution at 2^24 records, and the sums do not depend on the order of the additions. Batches whose
// adjoints are not finite take the float additions, so that NaN and infinity reach the gradients. Weights
// are at most one for points inside the box; the pairs of points outside of it (extrapolated with weights
// beyond one, or NaN for a NaN coordinate) are exceptions.
// The adjoint pass of a standalone encoding gives its adjoints in floats. Its records hold floats (GridGradientLayout),
// the scale of a sum goes by the records of its work item, and a value that would still lose bits in it (floats span
// more than 64 bits) goes to the gradient tensor with an atomic: 3 of 10^5 in a batch of normally distributed adjoints
// (16 levels of 2^19 entries of 2 floats, 2^17 points: 458 us with atomics, 44 + 45 us; 2^14 points 60 -> 46 us).
// Two forms that were measured and dropped: a workgroup per slice that tests every point of
// the batch against its slice and recomputes the hits (the work of a hit falls to one lane of
// 64, 890 us for 2^18 points and 16 levels), and the same with the hits queued in LDS first (the
// queued hits gather their point's coordinates and adjoints at random: bound by line requests).
//
// Replaces, for batches that are large enough, the atomicAdd of
// src_cpp/include/qmlp/kernels/encoding_hashgrid.cuh:117-166,345-369 of the reference.

#include <qmlp/kernels/common.h>
#include <qmlp/kernels/encoding_hashgrid.h>
#include <qmlp/kernels/grid_gradient_items.h>

QUICKMLP_KERNEL_NAMESPACE_BEGIN

/** One work item of GridGradientSlicesKernel: the `floats` elements of the gradient table from
 *  element `first` on (slice `slice` of level `level`), part `part` of `parts` of its regions. */
struct GridGradientSlice
{
    int level;
    unsigned first;
    int floats;
    int slice;
    int part;
    int parts;       // > 1: other work items hold sums for the same slice, all add it with atomics
    int place;       // of the slice in a row of GridGradientWorkspace::places
    int slices;      // of the level
};

/**
 * The temporary memory of these kernels. A region is what one workgroup of the records kernel files of POINTS
 * consecutive points: per level POINTS * PAIRS records, sorted by slice and without gaps.
 */
struct GridGradientWorkspace
{
    unsigned* records;            // (levels, regions, recordsPerRegion)
    // (regions, PLACES): per level where the records of each slice begin, how many records there are, how many exceptions
    unsigned short* places;
    unsigned short* exceptions;   // (levels, regions, recordsPerRegion): pairs that are left to GridGradientExceptionsKernel
    unsigned* largest;            // per workgroup the largest magnitude among its adjoints (bits without the sign)
    int regions;
    int recordsPerRegion;
    int largestCount;
    int reserved;
};

/**
 * Where the records kernel finds the adjoints of the encoded rows. The fused backward kernels leave them as halves, tile
 * by tile of 64 points with the ROW_CHANNELS values of a row 64 apart; the adjoint pass of a standalone encoding is
 * given rows of floats with strides (ROW_CHANNELS == 0), and its records then hold floats.
 */
template <int ROW_CHANNELS>
struct GridGradientAdjoints
{
    const half* __restrict__ data;   //(tiles, ROW_CHANNELS, 64)
    __device__ __forceinline__ f16 operator()(int p, int channel) const
    {
        return reinterpret_cast<const f16*>(data)[static_cast<long long>(p / TILE_POINTS) * (ROW_CHANNELS * TILE_POINTS)
                                                  + channel * TILE_POINTS + p % TILE_POINTS];
    }
};
template <>
struct GridGradientAdjoints<0>
{
    Tensor2Read<float> rows;         //(points, channels)
    __device__ __forceinline__ float operator()(int p, int channel) const
    {
        return rows.data_[static_cast<long long>(p) * rows.strides_[0] + static_cast<long long>(channel) * rows.strides_[1]];
    }
};

/** \tparam FLOATS the adjoints are floats, else halves */
template <typename Cfg, int SLICE_FLOATS, bool FLOATS = false>
struct GridGradientLayout
{
    typedef EncodingHashGrid<Cfg> Grid;
    static constexpr int D = Grid::D;
    static constexpr int F = Grid::F;
    static constexpr int L = Grid::L;
    static constexpr int PAIRS = Grid::NC / 2 > 0 ? Grid::NC / 2 : 1;
    /** A record in 32-bit words: the offsets of the lower and of the upper entry within the slice (16 bits
     *  each), their two weights, F halves of adjoint; one word of padding where that makes it a multiple of
     *  16 bytes (records of 16 or 32 bytes move as whole vector loads and stores). With adjoints that are floats:
     *  the offsets, the share of the upper entry, F products of adjoint and weight of the pair, so that the
     *  records of 2 features take 16 bytes as well. */
    static constexpr int ADJOINT_WORDS = FLOATS ? F : (F + 1) / 2;
    static constexpr int FIRST_ADJOINT = FLOATS ? 2 : 3;
    static constexpr int RECORD_WORDS_USED = FIRST_ADJOINT + ADJOINT_WORDS;
    static constexpr int RECORD_WORDS = RECORD_WORDS_USED % 4 == 3 ? RECORD_WORDS_USED + 1 : RECORD_WORDS_USED;
    static_assert(SLICE_FLOATS <= 65536, "offsets within a slice are stored in 16 bits");

    /** Value i among the adjoint words. */
    __device__ __forceinline__ static float adjoint(const unsigned* words, int i)
    {
        if constexpr (FLOATS) return __builtin_bit_cast(float, words[i]);
        else return static_cast<float>(__builtin_bit_cast(f16, static_cast<unsigned short>(words[i / 2] >> (16 * (i % 2)))));
    }
    /** What a record adds to its lower and to its upper entry, as a multiple of its adjoint values. */
    __device__ __forceinline__ static void weights(const unsigned* record, float& wL, float& wH)
    {
        if constexpr (FLOATS) {
            wH = __builtin_bit_cast(float, record[1]);
            wL = 1.f - wH;
        } else {
            wL = __builtin_bit_cast(float, record[1]);
            wH = __builtin_bit_cast(float, record[2]);
        }
    }

    /** Records start at multiples of their size from a 16-byte aligned base (LDS or global memory): 16, 8 or 4 bytes at a time. */
    template <typename Pointer>
    __device__ __forceinline__ static void loadRecord(Pointer src, unsigned (&r)[RECORD_WORDS])
    {
        if constexpr (RECORD_WORDS % 4 == 0) {
#pragma unroll
            for (int v = 0; v < RECORD_WORDS / 4; ++v) {
                const uint4 q = reinterpret_cast<const uint4*>(src)[v];
                r[4 * v] = q.x, r[4 * v + 1] = q.y, r[4 * v + 2] = q.z, r[4 * v + 3] = q.w;
            }
        } else if constexpr (RECORD_WORDS % 2 == 0) {
#pragma unroll
            for (int v = 0; v < RECORD_WORDS / 2; ++v) {
                const uint2 q = reinterpret_cast<const uint2*>(src)[v];
                r[2 * v] = q.x, r[2 * v + 1] = q.y;
            }
        } else {
#pragma unroll
            for (int v = 0; v < RECORD_WORDS; ++v) r[v] = src[v];
        }
    }
    __device__ __forceinline__ static void storeRecord(unsigned* dst, const unsigned (&r)[RECORD_WORDS])
    {
        if constexpr (RECORD_WORDS % 4 == 0) {
#pragma unroll
            for (int v = 0; v < RECORD_WORDS / 4; ++v)
                reinterpret_cast<uint4*>(dst)[v] = make_uint4(r[4 * v], r[4 * v + 1], r[4 * v + 2], r[4 * v + 3]);
        } else if constexpr (RECORD_WORDS % 2 == 0) {
#pragma unroll
            for (int v = 0; v < RECORD_WORDS / 2; ++v) reinterpret_cast<uint2*>(dst)[v] = make_uint2(r[2 * v], r[2 * v + 1]);
        } else {
#pragma unroll
            for (int v = 0; v < RECORD_WORDS; ++v) dst[v] = r[v];
        }
    }

    __device__ __host__ static constexpr int levelFloats(int l)
    {
        return (l + 1 < L ? Cfg::memoryOffset[l + 1] : Cfg::ParameterCount) - Cfg::memoryOffset[l];
    }
    __device__ __host__ static constexpr int numSlices(int l) { return (levelFloats(l) + SLICE_FLOATS - 1) / SLICE_FLOATS; }
    /** Index of the first word of level l in a row of GridGradientWorkspace::places, and the words of a row. */
    __device__ __host__ static constexpr int firstPlace(int l)
    {
        int n = 0;
        for (int k = 0; k < l; ++k) n += numSlices(k) + 2;
        return n;
    }
    static constexpr int PLACES = firstPlace(L);

    /** Levels with few slices are summed by several work items each. */
    __device__ __host__ static constexpr int parts(int l) { return gridGradientParts(numSlices(l)); }
};

template <typename Cfg, int ROW_CHANNELS, int CHANNEL_OFFSET, int SLICE_FLOATS, int POINTS>
struct GridGradientRecords
{
    static constexpr bool FLOATS = ROW_CHANNELS == 0;
    typedef GridGradientLayout<Cfg, SLICE_FLOATS, FLOATS> Layout;
    typedef GridGradientAdjoints<ROW_CHANNELS> Adjoints;
    typedef EncodingHashGrid<Cfg> Grid;
    typedef typename Grid::param_t param_t;
    static constexpr int AW = Layout::ADJOINT_WORDS;
    static constexpr int D = Grid::D;
    static constexpr int F = Grid::F;
    static constexpr int PAIRS = Layout::PAIRS;
    static constexpr int RW = Layout::RECORD_WORDS;
    static constexpr int MAX_SLICES = 512;
    typedef PositionDerivativeLayout<Cfg> DerivativeLayout;
    typedef typename DerivativeLayout::chunk_t DerivativeChunk;

    /** The two table entries of pair c of a point (bit b of c: upper corner in the b-th dimension
     *  other than the pair's own) and the weight of the pair without its own dimension. */
    template <int LEVEL>
    __device__ __forceinline__ static void pairEntries(const typename Grid::LevelSetup& s, int c, unsigned& idxL,
                                                       unsigned& idxH, float& w)
    {
        constexpr bool hashed = Cfg::hashed[LEVEL];
        constexpr int PD = hashed ? 0 : D - 1;   // the dimension whose two corners are neighbours in memory
        unsigned rest = 0u;
        w = 1.f;
        int bit = 0;
#pragma unroll
        for (int d = D - 1; d >= 0; --d) {
            if (d == PD) continue;
            const bool hi = (c >> bit) & 1;
            ++bit;
            const unsigned t = hi ? s.termH[d] : s.termL[d];
            rest = hashed ? (rest ^ t) : (rest + t);
            w = w * (hi ? s.f[d] : (1.f - s.f[d]));
        }
        if (hashed) {
            idxL = (rest ^ s.termL[PD]) % Cfg::hashGridSize[LEVEL];
            idxH = (rest ^ s.termH[PD]) % Cfg::hashGridSize[LEVEL];
        } else {
            idxL = rest + s.termL[PD];
            idxH = rest + s.termH[PD];
        }
    }

    /** Two entries fit one load of 16 bytes: the entries of a pair that lie side by side in the table (all pairs of a
     *  dense level away from its border; in a hashed level those whose lower corner has an even first coordinate)
     *  come with one request instead of two. */
    static constexpr bool PAIR_LOADS = 2 * F * static_cast<int>(sizeof(typename Cfg::table_t)) <= 16;

    /** The corner (bit d: upper in dimension d) of pair c's lower or upper entry. */
    template <int LEVEL>
    __device__ __forceinline__ static constexpr int cornerOfPair(int c, bool upper)
    {
        constexpr int PD = Cfg::hashed[LEVEL] ? 0 : D - 1;
        int corner = upper ? (1 << PD) : 0, bit = 0;
        for (int d = D - 1; d >= 0; --d) {
            if (d == PD) continue;
            corner |= ((c >> bit) & 1) << d;
            ++bit;
        }
        return corner;
    }

    /** The F values from position 'first' on of a wider vector that one load brought in. */
    template <typename Wide>
    __device__ __forceinline__ static void takeHeld(detail::HeldFeatures<F, typename Cfg::table_t>& h, const Wide& w, int first)
    {
        constexpr int V = detail::HeldFeatures<F, typename Cfg::table_t>::V;
#pragma unroll
        for (int i = 0; i < F / V; ++i)
#pragma unroll
            for (int j = 0; j < V; ++j) h.part[i][j] = w[first + i * V + j];
    }

    template <int LEVEL>
    __device__ __forceinline__ static void loadHeld(const typename Grid::LevelSetup& s, const param_t& params,
                                                    detail::HeldFeatures<F, typename Cfg::table_t> (&held)[Grid::NC])
    {
        if constexpr (PAIR_LOADS) {
            loadHeldPairs<LEVEL>(s, params, held);
        } else {
#pragma unroll
            for (int c = 0; c < Grid::NC; ++c) held[c].load(params.parametersForward + Grid::cornerOffset(LEVEL, s, c));
        }
    }

    template <int LEVEL>
    __device__ __forceinline__ static void loadHeldPairs(const typename Grid::LevelSetup& s, const param_t& params,
                                                         detail::HeldFeatures<F, typename Cfg::table_t> (&held)[Grid::NC])
    {
        const typename Cfg::table_t* __restrict__ table = params.parametersForward + Cfg::memoryOffset[LEVEL];
#pragma unroll
        for (int c = 0; c < PAIRS; ++c) {
            unsigned idxL, idxH;
            float w;
            pairEntries<LEVEL>(s, c, idxL, idxH, w);
            loadHeldPair<LEVEL>(c, idxL, idxH, table, held);
        }
    }

    template <int LEVEL>
    __device__ __forceinline__ static void loadHeldPair(int c, unsigned idxL, unsigned idxH, const typename Cfg::table_t* __restrict__ table,
                                                              detail::HeldFeatures<F, typename Cfg::table_t> (&held)[Grid::NC])
    {
        typedef typename Cfg::table_t table_t;
        constexpr int ENTRY_BYTES = F * static_cast<int>(sizeof(table_t));
        // entries lie at multiples of their size: aligned to the largest power of two that divides it
        constexpr int ALIGN = (ENTRY_BYTES & -ENTRY_BYTES) >= 8 ? 8 : (ENTRY_BYTES & -ENTRY_BYTES);
        typedef table_t pair_t __attribute__((ext_vector_type(2 * F), aligned(ALIGN)));
        const int lower = cornerOfPair<LEVEL>(c, false), upper = cornerOfPair<LEVEL>(c, true);   // constants once the loop over c is unrolled
        if (idxH == idxL + 1u) {
            const pair_t both = *reinterpret_cast<const pair_t*>(table + idxL * F);
            takeHeld(held[lower], both, 0);
            takeHeld(held[upper], both, F);
        } else {
            held[lower].load(table + idxL * F);
            held[upper].load(table + idxH * F);
        }
    }

    /**
     * The record of pair c of a point in one level: the offsets of its two entries within the slice of the lower
     * one, their weights and the adjoint words. Returns the slice within the level that files it.
     * \param otherSlice called with (element of feature 0 in the table, weight, adjWords) for an upper entry that
     *    lies in another slice and not right behind this one (in a hashed level of more cells along a coordinate than a
     *    slice has entries): the record then keeps the lower entry only
     */
    template <int LEVEL, typename OtherSlice>
    __device__ __forceinline__ static int buildRecord(const typename Grid::LevelSetup& s, int c,
                                                      const unsigned (&adjWords)[AW], unsigned (&rec)[RW],
                                                      const OtherSlice& otherSlice)
    {
        constexpr int PD = Cfg::hashed[LEVEL] ? 0 : D - 1;
        constexpr unsigned base = static_cast<unsigned>(Cfg::memoryOffset[LEVEL]);
        unsigned idxL, idxH;
        float w;
        pairEntries<LEVEL>(s, c, idxL, idxH, w);
        const int bucket = static_cast<int>(idxL * F / SLICE_FLOATS);   // the slice of the lower entry files the record
        const unsigned sliceStart = static_cast<unsigned>(bucket) * SLICE_FLOATS;
        const unsigned eL = idxL * F - sliceStart;
        unsigned eH = idxH * F - sliceStart;                     // wraps if the upper entry lies below the slice
        float wH = w * s.f[PD];
        const float wL = w * (1.f - s.f[PD]);
        if (eH >= static_cast<unsigned>(SLICE_FLOATS + F)) {
            otherSlice(base + idxH * F, wH, adjWords);
            eH = eL;
            wH = 0.f;
        }
        rec[0] = eL | (eH << 16);
        if constexpr (FLOATS) {
            // (without an upper entry the lower one takes all of it: its own weight then goes into the products)
            const bool lowerOnly = eH == eL && wH == 0.f;
            rec[1] = lowerOnly ? 0u : __builtin_bit_cast(unsigned, s.f[PD]);
#pragma unroll
            for (int i = 0; i < F; ++i)
                rec[2 + i] = __builtin_bit_cast(unsigned, (lowerOnly ? wL : w) * Layout::adjoint(adjWords, i));
        } else {
            rec[1] = __builtin_bit_cast(unsigned, wL);
            rec[2] = __builtin_bit_cast(unsigned, wH);
#pragma unroll
            for (int i = 0; i < AW; ++i) rec[3 + i] = adjWords[i];
        }
#pragma unroll
        for (int v = Layout::RECORD_WORDS_USED; v < RW; ++v) rec[v] = 0u;
        return bucket;
    }

    /** Feature i of a level among the channels of the encoded rows. */
    template <int LEVEL>
    __device__ __forceinline__ static constexpr int channel(int i) { return CHANNEL_OFFSET + (Cfg::Concat ? LEVEL * F : 0) + i; }

    /** What an entry of GridGradientWorkspace::exceptions says: the lane and the pair, and whether the lower entry is in its record. */
    static constexpr unsigned EXCEPTION_PAIR_SHIFT = 10, EXCEPTION_UPPER_ONLY = 1u << 13;
    static_assert(POINTS <= 1024 && PAIRS <= 8, "an exception takes 16 bits");

    /** Registers worth holding across the sort of a level's records: 64 bytes of table entries per lane. */
    static constexpr bool DEFER_ENTRIES = Grid::NC * F * static_cast<int>(sizeof(typename Cfg::table_t)) <= 64;

    /** Most slices of a level of the grid. */
    __device__ __host__ static constexpr int mostSlices()
    {
        int most = 1;
        for (int l = 0; l < Cfg::Levels; ++l) most = Layout::numSlices(l) > most ? Layout::numSlices(l) : most;
        return most;
    }

    /**
     * Files the records of the workgroup's points in one level. sCount: zeros on entry and on return, MAX_SLICES + 1 words, as many in
     * sOther: every level counts in the one that the level in front of it did not use, which is zeroed meanwhile.
     * \tparam INPUT_GRADIENTS the level's share of the gradient with respect to the position is added to adjPos
     */
    template <int LEVEL, int INPUT_GRADIENTS>
    __device__ __forceinline__ static void runLevel(int p, int numel, int region, const float (&position)[D], const Adjoints& adjEncoded,
                                                    const GridGradientWorkspace& ws, unsigned* sStage, int*& sCount, int*& sOther, int* sStart,
                                                    unsigned& maxAdjBits, const param_t& params, const DerivativeChunk* __restrict__ derivatives,
                                                    float (&adjPos)[D])
    {
        constexpr int NS = Layout::numSlices(LEVEL);
        static_assert(NS <= MAX_SLICES, "the records of a slice are counted in LDS");
        int tid = threadIdx.x;
        const long long regionStart = (static_cast<long long>(LEVEL) * ws.regions + region) * (POINTS * PAIRS);
        // (nothing of a level is worked out, and held in registers, before the one in front of it has ended)
        float pos[D];
#pragma unroll
        for (int d = 0; d < D; ++d) {
            pos[d] = position[d];
            asm volatile("" : "+v"(pos[d]));
        }
        asm volatile("" : "+v"(p), "+v"(tid));
        const bool valid = p < numel;

        // my records of this level, in registers, and their places among the workgroup's records of the same slice
        unsigned rec[PAIRS][RW];
        int bucket[PAIRS], rank[PAIRS];
        const typename Grid::LevelSetup s = Grid::setupLevel(LEVEL, pos);
        bool filed = valid;
        detail::HeldFeatures<F, typename Cfg::table_t> held[Grid::NC];
        (void)held;
        if (valid) {
            if constexpr (INPUT_GRADIENTS == 1 && !DEFER_ENTRIES) {
                // the entries of all corners, for this grid's share of dL/dinput (a dense 4-D grid with 8 features
                // holds 64 registers: used at once)
                loadHeld<LEVEL>(s, params, held);
                positionGradient<LEVEL>(p, s, held, adjEncoded, adjPos);
            }
            unsigned adjWords[AW];
#pragma unroll
            for (int i = 0; i < AW; ++i) adjWords[i] = 0u;
#pragma unroll
            for (int i = 0; i < F; ++i) {
                // largest magnitude seen (as bits without the sign: ordered like the values, NaN above infinity)
                if constexpr (FLOATS) {
                    adjWords[i] = __builtin_bit_cast(unsigned, adjEncoded(p, channel<LEVEL>(i)));
                    maxAdjBits = max(maxAdjBits, adjWords[i] & 0x7fffffffu);
                } else {
                    const unsigned bits = __builtin_bit_cast(unsigned short, adjEncoded(p, channel<LEVEL>(i)));
                    adjWords[i / 2] |= bits << (16 * (i % 2));
                    maxAdjBits = max(maxAdjBits, bits & 0x7fffu);
                }
            }
            // The sums of the slice kernel are fixed point with a scale that counts on weights of at most one, which
            // holds while every fractional position lies in [0, 1]: for every point inside the box. A point outside of
            // it is extrapolated (the fractional position is not clamped) with weights that grow with its distance, a
            // NaN coordinate gives NaN weights: the pairs of such a point are exceptions and have no records (in a level of one
            // slice, where every lane has fixed places, records of zeros).
            bool inside = true;
#pragma unroll
            for (int d = 0; d < D; ++d) inside = inside && s.f[d] >= 0.f && s.f[d] <= 1.f;
            auto except = [&](int c, unsigned which) {
                const int at = atomicAdd(sCount + NS, 1);
                ws.exceptions[regionStart + at] = static_cast<unsigned short>(static_cast<unsigned>(tid) | (static_cast<unsigned>(c) << EXCEPTION_PAIR_SHIFT) | which);
            };
#pragma unroll
            for (int c = 0; c < PAIRS; ++c) {
                bool otherSlice = false;
                bucket[c] = buildRecord<LEVEL>(s, c, adjWords, rec[c], [&](unsigned, float, const unsigned (&)[AW]) { otherSlice = true; });
                // (a level of one slice needs no sorting: every lane has fixed places)
                rank[c] = NS == 1 ? tid * PAIRS + c : inside ? atomicAdd(sCount + bucket[c], 1) : 0;
                if (otherSlice && inside) except(c, EXCEPTION_UPPER_ONLY);
            }
            filed = NS == 1 || inside;
            if (!inside) {
#pragma unroll
                for (int c = 0; c < PAIRS; ++c) {
                    except(c, 0u);
#pragma unroll
                    for (int v = 1; v < (FLOATS ? 2 + F : 3); ++v) rec[c][v] = 0u;
                }
            }
        }
        if (NS == 1 && tid == 0) sCount[0] = min(POINTS, numel - (p - tid)) * PAIRS;
        ldsBarrier();   // also: the staging area of the previous level has been copied out

        // Where the records of each slice begin: every wavefront adds the counts up for itself (all of them write the same values), which
        // takes less than a barrier behind one of them that does it for all (16 levels, 2^18 / 2^17 floats / 2^15 points: 83 -> 80.5,
        // 44.3 -> 42.5, 13.3 -> 12.8 us).
        {
            unsigned short* places = ws.places + static_cast<long long>(region) * Layout::PLACES + Layout::firstPlace(LEVEL);
            const int waveLane = tid % 64;
            int running = 0;
#pragma unroll
            for (int b0 = 0; b0 < NS; b0 += 64) {
                const int b = b0 + waveLane;
                const int n = b < NS ? sCount[b] : 0;
                const int inclusive = waveInclusiveScan(n);
                if (b < NS) {
                    sStart[b] = running + inclusive - n;
                    if (tid < 64) places[b] = static_cast<unsigned short>(running + inclusive - n);
                }
                running += __builtin_amdgcn_readlane(inclusive, 63);
            }
            if (waveLane == 0) sStart[NS] = running;
            if (tid == 0) {
                places[NS] = static_cast<unsigned short>(running);
                places[NS + 1] = static_cast<unsigned short>(sCount[NS]);
            }
            waveLdsSync();
        }

        if constexpr (INPUT_GRADIENTS == 1 && DEFER_ENTRIES) {
            // The entries of all corners where they take few registers: loaded here and used at the end of the level, so
            // that the two steps in between hide their latency (the barriers order LDS only).
            if (valid) loadHeld<LEVEL>(s, params, held);
        }
        for (int b = tid; b <= mostSlices(); b += POINTS) sOther[b] = 0;
        if (filed) {
#pragma unroll
            for (int c = 0; c < PAIRS; ++c) Layout::storeRecord(sStage + (sStart[bucket[c]] + rank[c]) * RW, rec[c]);
        }
        const int total = sStart[NS];
        ldsBarrier();
        int* const counted = sCount;
        sCount = sOther;
        sOther = counted;

        // sorted by slice: the region as a whole
        unsigned* __restrict__ records = ws.records + regionStart * RW;
        for (int j = tid; j < total; j += POINTS) {
            unsigned r[RW];
            Layout::loadRecord(sStage + j * RW, r);
            Layout::storeRecord(records + j * RW, r);
        }

        if constexpr (INPUT_GRADIENTS == 1 && DEFER_ENTRIES) {
            if (valid) positionGradient<LEVEL>(p, s, held, adjEncoded, adjPos);
        }
        if constexpr (INPUT_GRADIENTS == 2) {
            if (valid) positionGradientFromDerivatives<LEVEL>(p, derivatives, adjEncoded, adjPos);
        }
    }

    /**
     * This level's share of the gradient with respect to the position from the derivatives of the level's features
     * that the forward pass stored (PositionDerivativeLayout): sum_i adjoint_i * d feature_i / d p_d, read with one
     * or a few coalesced loads instead of a gather of all corners of the cell.
     */
    template <int LEVEL>
    __device__ __forceinline__ static void positionGradientFromDerivatives(int p, const DerivativeChunk* __restrict__ derivatives,
                                                                           const Adjoints& adjEncoded, float (&adjPos)[D])
    {
        float values[DerivativeLayout::VALUES];
        DerivativeLayout::load(derivatives + DerivativeLayout::chunkIndex(p / TILE_POINTS, 0, 0, p % TILE_POINTS), LEVEL, values);
        float lvl[D];
#pragma unroll
        for (int d = 0; d < D; ++d) lvl[d] = 0.f;
#pragma unroll
        for (int i = 0; i < F; ++i) {
            const float adj = static_cast<float>(adjEncoded(p, channel<LEVEL>(i)));
#pragma unroll
            for (int d = 0; d < D; ++d) lvl[d] += adj * values[i * D + d];
        }
        const float scale = Cfg::ResolutionFactor ? static_cast<float>(Cfg::resolution[LEVEL] - 1) : 1.f;
#pragma unroll
        for (int d = 0; d < D; ++d) adjPos[d] += scale * lvl[d];
    }

    /**
     * This level's share of the gradient with respect to the position, operation by operation as
     * EncodingHashGrid::adjoint computes it (same corner order, same products), so both give the same bits.
     */
    template <int LEVEL>
    __device__ __forceinline__ static void positionGradient(int p, const typename Grid::LevelSetup& s,
                                                            const detail::HeldFeatures<F, typename Cfg::table_t> (&held)[Grid::NC],
                                                            const Adjoints& adjEncoded, float (&adjPos)[D])
    {
        float adjFeat[F];
#pragma unroll
        for (int i = 0; i < F; ++i) adjFeat[i] = static_cast<float>(adjEncoded(p, channel<LEVEL>(i)));
        positionGradient<LEVEL>(s, held, adjFeat, adjPos);
    }

    /** The same from the adjoint of the level's features as floats. */
    template <int LEVEL>
    __device__ __forceinline__ static void positionGradient(const typename Grid::LevelSetup& s,
                                                            const detail::HeldFeatures<F, typename Cfg::table_t> (&held)[Grid::NC],
                                                            const float (&adjFeat)[F], float (&adjPos)[D])
    {
        float lvl[D];
#pragma unroll
        for (int d = 0; d < D; ++d) lvl[d] = 0.f;
#pragma unroll
        for (int c = 0; c < Grid::NC; ++c) {
            float v[F];
            held[c].toFloat(v);
            float dot = 0.f;
#pragma unroll
            for (int i = 0; i < F; ++i) dot += adjFeat[i] * v[i];
#pragma unroll
            for (int d = 0; d < D; ++d) {
                float prod = 1.f;
#pragma unroll
                for (int e = D - 1; e >= 0; --e)
                    if (e != d) prod *= ((c >> e) & 1) ? s.f[e] : (1.f - s.f[e]);
                lvl[d] += (((c >> d) & 1) ? prod : -prod) * dot;
            }
        }
        const float scale = Cfg::ResolutionFactor ? static_cast<float>(Cfg::resolution[LEVEL] - 1) : 1.f;
#pragma unroll
        for (int d = 0; d < D; ++d) adjPos[d] += scale * lvl[d];
    }

    /**
     * The input gradients that a workgroup computes beside the records that it files (INPUT_GRADIENTS, or 0: left to another
     * workgroup). The entries of all corners level by level with the records: the wavefronts of the chip then pass through the tables
     * together, the sort of a level hides the loads, and regions are as small as it takes to fill the chip (adjoint pass of 16 levels of
     * floats, 2^15 / 2^16 / 2^17 / 2^18 points 89 / 117 / 171 / 313 us; with a workgroup more per region for all of them 177 / 198 / 255 / 475).
     * One level is left to workgroups of their own (32^4 nodes x 8, 2^18 / 2^19 points 143 / 247 us, within the records kernel 158 / 285), as
     * are stored derivatives, which are read at the rate of the memory, unless the records take the registers of a second workgroup anyway (64^3 nodes x 4 halves, 2^20 points 152 us
     * inline and 164 apart; 512^3 cells hashed to 2 halves 139 and 129).
     */
    template <int INPUT_GRADIENTS>
    __device__ __host__ static constexpr int inputGradientsInline()
    {
        return INPUT_GRADIENTS == 1 ? (Cfg::Levels > 1 ? 1 : 0) : INPUT_GRADIENTS == 2 ? (Cfg::Levels == 1 && PAIRS * RW > 16 ? 2 : 0) : 0;
    }

    /** Two workgroups of 1024 lanes per compute unit where the records of a lane leave room for it in 64 registers. */
    template <int INPUT_GRADIENTS>
    __device__ __host__ static constexpr int wavesPerSimd()
    {
        return PAIRS * RW <= 16 && INPUT_GRADIENTS != 1 && inputGradientsInline<INPUT_GRADIENTS>() == 0 ? 8 : POINTS >= 1024 ? 4 : 1;
    }

    /** The levels from LEVEL to END - 1. */
    template <int LEVEL, int END, int INPUT_GRADIENTS, typename... Args>
    __device__ __forceinline__ static void runLevels(Args&&... args)
    {
        if constexpr (LEVEL < END) {
            runLevel<LEVEL, INPUT_GRADIENTS>(args...);
            runLevels<LEVEL + 1, END, INPUT_GRADIENTS>(args...);
        }
    }

    /** The levels of one of GROUPS groups. */
    template <int G, int GROUPS, int INPUT_GRADIENTS, typename... Args>
    __device__ __forceinline__ static void runGroup(int group, Args&&... args)
    {
        if constexpr (G + 1 < GROUPS) {
            if (group == G) runLevels<Cfg::Levels * G / GROUPS, Cfg::Levels * (G + 1) / GROUPS, INPUT_GRADIENTS>(args...);
            else runGroup<G + 1, GROUPS, INPUT_GRADIENTS>(group, args...);
        } else {
            runLevels<Cfg::Levels * G / GROUPS, Cfg::Levels, INPUT_GRADIENTS>(args...);
        }
    }

    /** The gradient of a point with respect to its position from stored derivatives. */
    template <int LEVEL>
    __device__ __forceinline__ static void positionGradientsFromDerivatives(int p, const Adjoints& adjEncoded,
                                                                            const DerivativeChunk* __restrict__ derivatives, float (&adjPos)[D])
    {
        if constexpr (LEVEL < Cfg::Levels) {
            if (LEVEL % 4 == 0) {   // (those of four levels in registers at a time)
                asm volatile("" : "+v"(p));
#pragma unroll
                for (int d = 0; d < D; ++d) asm volatile("" : "+v"(adjPos[d]));
            }
            positionGradientFromDerivatives<LEVEL>(p, derivatives, adjEncoded, adjPos);
            positionGradientsFromDerivatives<LEVEL + 1>(p, adjEncoded, derivatives, adjPos);
        }
    }

    /** The gradient of a point with respect to its position from the entries of all corners of a grid of one level. */
    __device__ __forceinline__ static void positionGradientOfOneLevel(int p, const Tensor2Read<float>& inputs, const Adjoints& adjEncoded,
                                                                      const param_t& params, float (&adjPos)[D])
    {
        float pos[D];
        loadPosition(inputs, p, params, pos);
        const typename Grid::LevelSetup s = Grid::setupLevel(0, pos);
        detail::HeldFeatures<F, typename Cfg::table_t> held[Grid::NC];
        loadHeld<0>(s, params, held);
        positionGradient<0>(p, s, held, adjEncoded, adjPos);
    }

    /** Adds adjPos to the gradient with respect to the input of point p, or writes it. */
    __device__ __forceinline__ static void storeInputGradient(const Tensor2RW<float>& adjInputs, int p, const param_t& params, int overwrite,
                                                              const float (&adjPos)[D])
    {
        // every point belongs to one lane of one workgroup: a plain read-modify-write
#pragma unroll
        for (int d = 0; d < D; ++d) {
            float* adj = adjInputs.data_ + (static_cast<long long>(p) * adjInputs.strides_[0]
                                            + static_cast<long long>(d + Cfg::Start) * adjInputs.strides_[1]);
            const float before = overwrite ? 0.f : *adj;
            *adj = before + adjPos[d] * params.boundingBoxInvSize[d];
        }
    }

    __device__ __forceinline__ static void loadPosition(const Tensor2Read<float>& inputs, int p, const param_t& params, float (&pos)[D])
    {
#pragma clang fp contract(off)
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const float in = inputs.data_[static_cast<long long>(p) * inputs.strides_[0] + static_cast<long long>(d + Cfg::Start) * inputs.strides_[1]];
            pos[d] = (in - params.boundingBoxMin[d]) * params.boundingBoxInvSize[d];
        }
    }

    /** Zeroes the elements of the gradient tensor that the slice kernel adds to with atomics; index: of the thread. */
    template <int LEVEL>
    __device__ __forceinline__ static void zeroShared(int index, int threads, float* __restrict__ gradients)
    {
        if constexpr (LEVEL < Cfg::Levels) {
            constexpr int SLICES = Layout::numSlices(LEVEL);
            constexpr bool WHOLE = Layout::parts(LEVEL) > 1;
            constexpr int COUNT = WHOLE ? Layout::levelFloats(LEVEL) : (SLICES - 1) * F;   // (the first entry of every slice but the first)
            float* __restrict__ level = gradients + Cfg::memoryOffset[LEVEL];
            for (int i = index; i < COUNT; i += threads) level[WHOLE ? i : (i / F + 1) * SLICE_FLOATS + i % F] = 0.f;
            zeroShared<LEVEL + 1>(index, threads, gradients);
        }
    }

    /** Adds one entry of GridGradientWorkspace::exceptions to the gradient tensor. */
    template <int LEVEL>
    __device__ __forceinline__ static void addException(unsigned exception, int firstPoint, const Tensor2Read<float>& inputs,
                                                        const Adjoints& adjEncoded, const param_t& params)
    {
        constexpr int PD = Cfg::hashed[LEVEL] ? 0 : D - 1;
        const int p = firstPoint + static_cast<int>(exception & ((1u << EXCEPTION_PAIR_SHIFT) - 1u));
        const int c = static_cast<int>(exception >> EXCEPTION_PAIR_SHIFT) & 7;
        float pos[D];
        loadPosition(inputs, p, params, pos);
        const typename Grid::LevelSetup s = Grid::setupLevel(LEVEL, pos);
        unsigned idxL, idxH;
        float w;
        pairEntries<LEVEL>(s, c, idxL, idxH, w);
        const float wL = w * (1.f - s.f[PD]), wH = w * s.f[PD];
        float* __restrict__ grad = params.parametersBackward + Cfg::memoryOffset[LEVEL];
#pragma unroll 1
        for (int i = 0; i < F; ++i) {
            const float adj = static_cast<float>(adjEncoded(p, channel<LEVEL>(i)));
            if (!(exception & EXCEPTION_UPPER_ONLY)) unsafeAtomicAdd(grad + idxL * F + i, wL * adj);
            unsafeAtomicAdd(grad + idxH * F + i, wH * adj);
        }
    }
};

/**
 * \tparam GROUPS the levels are shared out over so many workgroups
 * \tparam INPUT_GRADIENTS 0: none; 1: from the entries of all corners (of several levels with GROUPS == 1 only); 2: from stored
 * derivatives; by another workgroup per region, or by those that file the records (GridGradientRecords::inputGradientsInline)
 * \tparam POINTS points (= lanes) of a workgroup; its records of one level are staged in LDS
 * \tparam ROW_CHANNELS, CHANNEL_OFFSET where the adjoints of this grid lie, see GridGradientAdjoints
 * Launched with a multiple of the workgroups of a region; without those of input gradients they are workspace.largestCount.
 */
template <typename Cfg, int ROW_CHANNELS, int CHANNEL_OFFSET, int SLICE_FLOATS, int POINTS, int INPUT_GRADIENTS, int GROUPS>
__global__ void __launch_bounds__(POINTS) __attribute__((amdgpu_waves_per_eu(GridGradientRecords<Cfg, ROW_CHANNELS, CHANNEL_OFFSET, SLICE_FLOATS, POINTS>::template wavesPerSimd<INPUT_GRADIENTS>())))
GridGradientRecordsKernel(
    int numel,
    const Tensor2Read<float> inputs,          //shape (numel, Cin)
    const GridGradientAdjoints<ROW_CHANNELS> adjEncoded,
    const HashGridParams<typename Cfg::table_t, Cfg::Dim> params,
    const GridGradientWorkspace workspace,
    int overwrite,                            //the gradient tensor holds nothing yet
    Tensor2RW<float> adjInputs,               //INPUT_GRADIENTS: shape (numel, Cin), this grid's share of dL/dinput is added
    int overwriteInput,                       //... or written
    const void* __restrict__ derivativesV)    //INPUT_GRADIENTS == 2: the position derivatives of this grid that the forward pass stored
{
    typedef GridGradientRecords<Cfg, ROW_CHANNELS, CHANNEL_OFFSET, SLICE_FLOATS, POINTS> Impl;
    constexpr int D = Cfg::Dim;
    constexpr int INLINE = Impl::template inputGradientsInline<INPUT_GRADIENTS>();
    constexpr int WORKGROUPS = GROUPS + (INPUT_GRADIENTS != INLINE ? 1 : 0);   // of a region
    extern __shared__ __align__(16) unsigned char sMemory[];
    unsigned* sStage = reinterpret_cast<unsigned*>(sMemory);              // POINTS * PAIRS records
    int* sCount = reinterpret_cast<int*>(sStage + POINTS * Impl::PAIRS * Impl::RW);
    int* sOther = sCount + Impl::MAX_SLICES + 1;
    int* sStart = sOther + Impl::MAX_SLICES + 1;
    // (by few workgroups: the others only pass by)
    constexpr int ZEROING = 64;
    if (overwrite && blockIdx.x < ZEROING)
        Impl::template zeroShared<0>(blockIdx.x * POINTS + threadIdx.x, min(ZEROING, static_cast<int>(gridDim.x)) * POINTS, params.parametersBackward);
    // Adjoints in rows: a row holds all levels, so that the groups follow one another and every die finds the rows of its
    // regions in its L2 again (16 levels, 2^17 points: 44 us, 62 with the groups of a region side by side), which takes as many
    // workgroups to a group as is a multiple of the dies (2^17 + 64 points, adjoint pass: 90 us, 115 with 129 workgroups). Adjoints of
    // tiles: nothing is shared, and the slice kernel reads what lies in memory region by region faster (2^18 points: 82 and
    // 84 us, 90 and 95 with the groups one behind the other).
    const int step = gridDim.x / WORKGROUPS;
    const int group = Impl::FLOATS ? blockIdx.x / step : blockIdx.x % WORKGROUPS, first = Impl::FLOATS ? blockIdx.x % step : blockIdx.x / WORKGROUPS;
    const auto* derivatives = static_cast<const typename Impl::DerivativeChunk*>(derivativesV);
    if constexpr (INPUT_GRADIENTS != INLINE) {
        if (group == GROUPS) {
            for (int p = first * POINTS + threadIdx.x; p < numel; p += step * POINTS) {
                float adjPos[D];
#pragma unroll
                for (int d = 0; d < D; ++d) adjPos[d] = 0.f;
                if constexpr (INPUT_GRADIENTS == 2) Impl::template positionGradientsFromDerivatives<0>(p, adjEncoded, derivatives, adjPos);
                else Impl::positionGradientOfOneLevel(p, inputs, adjEncoded, params, adjPos);
                Impl::storeInputGradient(adjInputs, p, params, overwriteInput, adjPos);
            }
            return;
        }
    }
    unsigned maxAdjBits = 0u;
    for (int b = threadIdx.x; b <= Impl::MAX_SLICES; b += POINTS) sCount[b] = sOther[b] = 0;
    ldsBarrier();
    for (int region = first; region < workspace.regions; region += step) {
        const int p = region * POINTS + threadIdx.x;
        float pos[D], adjPos[D];
#pragma unroll
        for (int d = 0; d < D; ++d) pos[d] = adjPos[d] = 0.f;
        if (p < numel) Impl::loadPosition(inputs, p, params, pos);
        Impl::template runGroup<0, GROUPS, INLINE>(group, p, numel, region, pos, adjEncoded, workspace, sStage, sCount, sOther, sStart,
                                                   maxAdjBits, params, derivatives, adjPos);
        if constexpr (INLINE != 0) {
            if (p < numel) Impl::storeInputGradient(adjInputs, p, params, overwriteInput, adjPos);
        }
    }
    // the largest adjoint of the workgroup
    if (maxAdjBits != 0u) atomicMax(sCount, static_cast<int>(maxAdjBits));
    __syncthreads();
    if (threadIdx.x == 0) workspace.largest[first * GROUPS + group] = static_cast<unsigned>(sCount[0]);
}

template <typename Cfg, int ROW_CHANNELS, int CHANNEL_OFFSET, int SLICE_FLOATS>
struct GridGradientExceptions
{
    typedef GridGradientRecords<Cfg, ROW_CHANNELS, CHANNEL_OFFSET, SLICE_FLOATS, 1024> Records;
    typedef typename Records::Layout Layout;

    /** Where a row of GridGradientWorkspace::places says how many exceptions a level has. */
    __device__ __forceinline__ static int placeOfCount(int level)
    {
        int place = 0;
#pragma unroll
        for (int l = 0; l < Cfg::Levels; ++l)
            if (level == l) place = Layout::firstPlace(l) + Layout::numSlices(l) + 1;
        return place;
    }

    /** Adds an exception of a level. */
    template <int LEVEL>
    __device__ __forceinline__ static void add(int level, unsigned exception, int firstPoint, const Tensor2Read<float>& inputs,
                                               const typename Records::Adjoints& adjEncoded, const typename Records::param_t& params)
    {
        if constexpr (LEVEL < Cfg::Levels) {
            if (level == LEVEL) Records::template addException<LEVEL>(exception, firstPoint, inputs, adjEncoded, params);
            else add<LEVEL + 1>(level, exception, firstPoint, inputs, adjEncoded, params);
        }
    }
};

/**
 * What the records leave out, added to the gradient tensor with atomics behind the slice kernel: the points outside of the box,
 * and in hashed levels of more cells along a coordinate than a slice has entries upper entries far away. Most batches have
 * none: every lane looks up the number of exceptions of one list (a region and a level), and a launch that finds none takes 4 us. Lists
 * are shared out in parts of one exception per lane, neighbouring parts over neighbouring workgroups, as points outside of the box
 * often lie next to each other in a batch. Bound by the atomics. (A wavefront per region, which walked through its lists alone: 16
 * levels, 2^17 points, the first 64th of them outside 1332 us for the adjoint pass, the first quarter 1427; shared out 168 and 479, and without points outside 95.)
 */
template <typename Cfg, int ROW_CHANNELS, int CHANNEL_OFFSET, int SLICE_FLOATS>
__global__ void __launch_bounds__(GRID_GRADIENT_EXCEPTIONS_BLOCK) GridGradientExceptionsKernel(
    const Tensor2Read<float> inputs, const GridGradientAdjoints<ROW_CHANNELS> adjEncoded,
    const HashGridParams<typename Cfg::table_t, Cfg::Dim> params, const GridGradientWorkspace workspace)
{
    typedef GridGradientExceptions<Cfg, ROW_CHANNELS, CHANNEL_OFFSET, SLICE_FLOATS> Impl;
    constexpr int BLOCK = GRID_GRADIENT_EXCEPTIONS_BLOCK;
    __shared__ int sCount[BLOCK];
    __shared__ unsigned long long sFound[BLOCK / 64];
    const int tid = threadIdx.x;
    const unsigned parts = (workspace.recordsPerRegion + BLOCK - 1) / BLOCK;   // of a list
    const unsigned items = static_cast<unsigned>(workspace.regions) * Cfg::Levels * parts;
    for (unsigned i0 = 0; blockIdx.x + i0 * gridDim.x < items; i0 += BLOCK) {
        // the parts of this workgroup: blockIdx.x + (i0 + lane) * gridDim.x
        const unsigned item = blockIdx.x + (i0 + tid) * gridDim.x;
        int count = 0;
        if (item < items) {
            const unsigned list = item / parts, part = item - list * parts, region = list / Cfg::Levels;
            count = workspace.places[static_cast<long long>(region) * Impl::Layout::PLACES + Impl::placeOfCount(static_cast<int>(list - region * Cfg::Levels))];
            count -= static_cast<int>(part * BLOCK);
        }
        const unsigned long long found = __ballot(count > 0);
        if (tid % 64 == 0) sFound[tid / 64] = found;
        sCount[tid] = count;
        __syncthreads();
        for (int w = 0; w < BLOCK / 64; ++w) {
            unsigned long long left = sFound[w];
            while (left != 0) {
                const int from = w * 64 + __builtin_ctzll(left);
                left &= left - 1;
                if (tid >= sCount[from]) continue;
                const unsigned which = blockIdx.x + (i0 + from) * gridDim.x;
                const unsigned list = which / parts, part = which - list * parts, region = list / Cfg::Levels;
                const int level = static_cast<int>(list - region * Cfg::Levels);
                const unsigned short* exceptions = workspace.exceptions
                    + (static_cast<long long>(level) * workspace.regions + region) * workspace.recordsPerRegion + part * BLOCK;
                Impl::template add<0>(level, exceptions[tid], static_cast<int>(region) * (workspace.recordsPerRegion / Impl::Records::PAIRS), inputs,
                                      adjEncoded, params);
            }
        }
        __syncthreads();   // sFound and sCount have been read
    }
}

template <typename Cfg, int SLICE_FLOATS, int LEVEL>
struct GridGradientTraceLevels
{
    template <typename Words>
    __device__ __forceinline__ static void run(const float (&pos)[Cfg::Dim], const Words& adjWords, unsigned* idx, float* w)
    {
        if constexpr (LEVEL < Cfg::Levels) {
            typedef GridGradientRecords<Cfg, 16, 0, SLICE_FLOATS, 256> Impl;
            typedef EncodingHashGrid<Cfg> Grid;
            constexpr int NC = Grid::NC;
            const typename Grid::LevelSetup s = Grid::setupLevel(LEVEL, pos);
#pragma unroll
            for (int c = 0; c < Impl::PAIRS; ++c) {
                unsigned rec[Impl::RW];
                unsigned otherElement = 0u;
                float otherWeight = 0.f;
                bool other = false;
                const int bucket = Impl::template buildRecord<LEVEL>(s, c, adjWords, rec,
                    [&](unsigned element, float weight, const Words&) { other = true; otherElement = element; otherWeight = weight; });
                // (the pairs of a point outside the box are added by GridGradientExceptionsKernel, entry by entry as decoded here)
                const unsigned sliceStart = static_cast<unsigned>(Cfg::memoryOffset[LEVEL]) + static_cast<unsigned>(bucket) * SLICE_FLOATS;
                idx[LEVEL * NC + 2 * c] = sliceStart + (rec[0] & 0xffffu);
                w[LEVEL * NC + 2 * c] = __builtin_bit_cast(float, rec[1]);
                if (NC > 1) {
                    idx[LEVEL * NC + 2 * c + 1] = other ? otherElement : sliceStart + (rec[0] >> 16);
                    w[LEVEL * NC + 2 * c + 1] = other ? otherWeight : __builtin_bit_cast(float, rec[2]);
                }
            }
            GridGradientTraceLevels<Cfg, SLICE_FLOATS, LEVEL + 1>::run(pos, adjWords, idx, w);
        }
    }
};

/**
 * Test aid: for every point (one per lane) and level, the table elements and weights that the records of
 * GridGradientRecords::buildRecord stand for, decoded as the slice kernel decodes them (its slice +
 * 16-bit offset), and the entries that are exceptions because they lie in another slice.
 * Slots as in CornerTrace: level * 2^Dim + 2 * pair (+ 1 for the upper entry).
 */
template <typename Cfg, int SLICE_FLOATS>
__global__ void __launch_bounds__(256) GridGradientTraceKernel(
    long long numel, const Tensor2Read<float> inputs, unsigned* __restrict__ indices, float* __restrict__ weights,
    const HashGridParams<typename Cfg::table_t, Cfg::Dim> params)
{
    typedef GridGradientRecords<Cfg, 16, 0, SLICE_FLOATS, 256> Impl;
    typedef EncodingHashGrid<Cfg> Grid;
    constexpr int D = Cfg::Dim, F = Cfg::Features, NC = Grid::NC;
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
        unsigned* idx = indices + index * (Cfg::Levels * NC);
        float* w = weights + index * (Cfg::Levels * NC);
        unsigned adjWords[(F + 1) / 2];
#pragma unroll
        for (int i = 0; i < (F + 1) / 2; ++i) adjWords[i] = 0x3c003c00u;   // 1.0 | 1.0
        GridGradientTraceLevels<Cfg, SLICE_FLOATS, 0>::run(pos, adjWords, idx, w);
    }
}

template <typename Cfg, int SLICE_FLOATS, bool FLOATS>
struct GridGradientSlices
{
    typedef GridGradientLayout<Cfg, SLICE_FLOATS, FLOATS> Layout;
    typedef EncodingHashGrid<Cfg> Grid;
    static constexpr int F = Grid::F;
    static constexpr int RW = Layout::RECORD_WORDS;
    static constexpr int BLOCK = 1024;

    /**
     * v * 2^scaleExponent as a 64-bit integer (scale: that power of two; |v * scale| < 2^51), rounded to nearest: the
     * sum with 1.5 * 2^52 has the integer in the low bits of its mantissa. Three instructions, two of them in double
     * precision; split into two words in single precision it takes nine.
     */
    static constexpr int FIXED_BITS = 51;
    __device__ __forceinline__ static long long toFixed(double v, double scale)
    {
        const double shifted = __builtin_fma(v, scale, 6755399441055744.0);
        return __builtin_bit_cast(long long, shifted) - 0x4338000000000000ll;
    }

    __device__ __forceinline__ static void ldsAddFixed(long long* p, long long v)
    {
        typedef __attribute__((address_space(3))) unsigned long long lds_u64;
        __hip_atomic_fetch_add((lds_u64*)p, static_cast<unsigned long long>(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }

    /** Two workgroups per compute unit where the LDS has room for two. */
    static constexpr int WAVES_PER_SIMD = SLICE_FLOATS <= 8192 && RW <= 4 ? 8 : 4;

    /** Sums of a slice and of the entry behind it. */
    static constexpr int SUMS = SLICE_FLOATS + F;
    /** What the workgroup keeps in LDS beside the sums. */
    static constexpr int SEGMENTS = BLOCK;      // regions that are looked up together
    static constexpr int WAVES = BLOCK / 64;
    static constexpr int SMALL = FLOATS ? 256 : 0;
    static constexpr int MOST_TERMS_WITH_LIST = 3 << 16;   // of a work item; of normally distributed adjoints about a hundred are on the list then
    struct Shared
    {
        unsigned segments[SEGMENTS];            // where the records of the slice begin and end in each region (16 bits each), or parts of them
        unsigned short regions[SEGMENTS];       // of these parts, counted from the first region that is looked up
        int place[SEGMENTS];                    // among all parts, of the first one of each region
        unsigned largest[WAVES];
        int records[WAVES];
        int longest[WAVES];
        int smallCount;
        float smallValues[SMALL + 1];
        unsigned short smallElements[SMALL + 1];
    };

    /** Where the records of the slice begin and end in a region. */
    __device__ __forceinline__ static unsigned segmentOf(const GridGradientWorkspace& ws, const GridGradientSlice& item, int region)
    {
        const unsigned short* place = ws.places + static_cast<long long>(region) * Layout::PLACES + item.place;
        return place[0] | (static_cast<unsigned>(place[1]) << 16);
    }

    /** Sum over the lanes in front of this one, of a workgroup; total: over all. All of them call this. */
    __device__ __forceinline__ static int scan(int tid, int n, int (&waves)[WAVES], int& total)
    {
        int inclusive = n;
#pragma unroll
        for (int d = 1; d < 64; d *= 2) {
            const int other = __shfl_up(inclusive, d, 64);
            if (tid % 64 >= d) inclusive += other;
        }
        __syncthreads();
        if (tid % 64 == 63) waves[tid / 64] = inclusive;
        __syncthreads();
        const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
        int before = 0;
        total = 0;
#pragma unroll 1
        for (int w = 0; w < WAVES; ++w) {
            const int of = __builtin_amdgcn_readfirstlane(waves[w]);
            if (w < wave) before += of;
            total += of;
        }
        return before + inclusive - n;
    }

    /** Groups of so many lanes (the logarithm) take the records of a segment: half of what it holds where points are spread evenly, 8 to all. */
    __device__ __forceinline__ static int groupLog2(const GridGradientWorkspace& ws, const GridGradientSlice& item)
    {
        int log2 = 3;
        while (log2 < 10 && (4 << log2) * item.slices <= ws.recordsPerRegion) ++log2;
        return log2;
    }
    static constexpr int STEPS = 3;   // records per lane of a part of a segment
    static constexpr unsigned LONG_SEGMENTS = 1u << 31;   // beside a magnitude: some segment holds more than twice what a part does

    /** Whether the longest segment holds more than twice a group's share of all records of a work item. */
    __device__ __forceinline__ static bool isUneven(const GridGradientWorkspace& ws, const GridGradientSlice& item, int begin, int end, Shared& shared)
    {
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));   // (nothing of this is worked out, and held in registers, for batches that do not need it)
        int records = 0, longest = 0;
        for (int r = begin + tid; r < end; r += BLOCK) {
            const unsigned s = segmentOf(ws, item, r);
            const int size = static_cast<int>(s >> 16) - static_cast<int>(s & 0xffffu);
            records += size;
            longest = max(longest, size);
        }
        int all;
        (void)scan(tid, records, shared.records, all);
#pragma unroll
        for (int d = 32; d > 0; d /= 2) longest = max(longest, __shfl_xor(longest, d, 64));
        if (tid % 64 == 0) shared.longest[tid / 64] = longest;
        __syncthreads();
#pragma unroll 1
        for (int w = 0; w < WAVES; ++w) longest = max(longest, shared.longest[w]);
        return static_cast<long long>(__builtin_amdgcn_readfirstlane(longest)) * (BLOCK >> groupLog2(ws, item)) > 2ll * all;
    }

    /**
     * Calls add(record) for the records of a work item. The records of a slice lie in segments, one per region, of
     * recordsPerRegion / (slices of the level) records where the points are spread evenly. A group of lanes takes segments as one stream of
     * records: a lane that is through with one goes on in the group's next, so that every load and every addition is that of whole
     * wavefronts, and the loads of the next records are under way while these are added. (A segment at a time, three records per lane,
     * left a third of the additions to lanes without a record, and nothing was under way meanwhile: four levels of halves, 2^20
     * points 307 us for the adjoint pass, now 266; a dense 4-D grid of 8 features, four records to a segment, 2^19 points 207 and 177; 16
     * levels, 2^18 points 197 and 187.) Where neighbours in the batch are neighbours in space as well (samples along rays, a
     * batch in some order) a few segments may hold most records, and the groups that took them would work on alone (`uneven`): segments
     * are then cut into parts of STEPS records per lane first. (Left to one group: one level of 64^3 nodes x 4 floats, adjoint pass of
     * 2^17 samples along rays 98 us; cut 34, points at random 29.)
     * shared.segments holds the first SEGMENTS regions.
     * \tparam RARE passes that few batches need, as little code as possible: cut into parts in any case
     */
    template <bool RARE, typename Add>
    __device__ __forceinline__ static void forEachRecord(const GridGradientWorkspace& ws, const GridGradientSlice& item, int begin, int end,
                                                         bool uneven, Shared& shared, const Add& add)
    {
        const int log2 = groupLog2(ws, item);
        if (!RARE && !uneven) {
            for (int r0 = begin; r0 < end; r0 += SEGMENTS) {
                const int count = min(SEGMENTS, end - r0);
                if (r0 != begin) {
                    __syncthreads();   // the segments in front of these have been read
                    if (static_cast<int>(threadIdx.x) < count) shared.segments[threadIdx.x] = segmentOf(ws, item, r0 + threadIdx.x);
                    __syncthreads();
                }
                forEachPart<false, false>(threadIdx.x, ws, item, r0, count, log2, shared, add);
            }
            return;
        }
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));   // (nothing of this is worked out, and held in registers, for batches that do not need it)
        const int most = STEPS << log2;
        for (int r0 = begin; r0 < end; r0 += SEGMENTS) {
            const int count = min(SEGMENTS, end - r0);
            int all;
            {
                const unsigned segment = tid < count ? segmentOf(ws, item, r0 + tid) : 0u;
                const int size = static_cast<int>(segment >> 16) - static_cast<int>(segment & 0xffffu);
                shared.place[tid] = scan(tid, (size + most - 1) / most, shared.records, all);
            }
            for (int q0 = 0; q0 < all; q0 += SEGMENTS) {
                if (q0 > 0) __syncthreads();   // those in front of these have been read
                const unsigned segment = tid < count ? segmentOf(ws, item, r0 + tid) : 0u;
                const int place = shared.place[tid] - q0;
                int at = max(place, 0);
                for (int j = static_cast<int>(segment & 0xffffu) + (at - place) * most, to = static_cast<int>(segment >> 16); j < to && at < SEGMENTS; j += most, ++at) {
                    shared.segments[at] = static_cast<unsigned>(j) | (static_cast<unsigned>(min(j + most, to)) << 16);
                    shared.regions[at] = static_cast<unsigned short>(tid);
                }
                __syncthreads();
                forEachPart<true, RARE>(tid, ws, item, r0, min(SEGMENTS, all - q0), log2, shared, add);
            }
        }
    }

    /** ... for so many segments of the regions from r0 on, or parts of them. */
    template <bool PARTS, bool RARE, typename Add>
    __device__ __forceinline__ static void forEachPart(int tid, const GridGradientWorkspace& ws, const GridGradientSlice& item, int r0, int count, int log2,
                                                       const Shared& shared, const Add& add)
    {
        // (records of a lane under way while as many are added: of wide ones fewer keep the memory busy; dense 4-D grid of 8 features, 40 B,
        // 2^20 points 349 us for the adjoint pass with one, 368 with two; 4 levels of 16 B, 2^20 points 275 and 266)
        constexpr int LOADS = RARE || RW > 4 ? 1 : 2;
        const int groups = BLOCK >> log2, lanes = 1 << log2;
        const unsigned* first = ws.records + (static_cast<long long>(item.level) * ws.regions + r0) * ws.recordsPerRegion * RW;
        // this lane is at record `at` of part s, which begins at word `base` (a thousand regions take less than 2^27) and has `size`
        int s = tid >> log2, at = tid & (lanes - 1), size = 0;
        unsigned base = 0u;
        auto look = [&] {
            const unsigned places = shared.segments[s], region = PARTS ? shared.regions[s] : static_cast<unsigned>(s);
            size = static_cast<int>(places >> 16) - static_cast<int>(places & 0xffffu);
            base = (region * static_cast<unsigned>(ws.recordsPerRegion) + (places & 0xffffu)) * RW;
        };
        // (loads without a branch around them: only then those of the next records can be in flight while these are added)
        auto load = [&](unsigned (&rec)[LOADS][RW]) {
            int loaded = 0;
#pragma unroll
            for (int u = 0; u < LOADS; ++u) {
                while (at >= size && s < count) {
                    at -= size;
                    s += groups;
                    if (s < count) look();
                }
                Layout::loadRecord(first + (s < count ? base + static_cast<unsigned>(at * RW) : 0u), rec[u]);
                at += lanes;
                loaded += s < count ? 1 : 0;
            }
            return loaded;
        };
        auto addAll = [&](const unsigned (&rec)[LOADS][RW], int loaded) {
#pragma unroll
            for (int u = 0; u < LOADS; ++u)
                if (u < loaded) add(rec[u]);
        };
        if (s < count) look();
        if constexpr (RARE || PARTS) {
            for (;;) {
                unsigned rec[LOADS][RW];
                const int loaded = load(rec);
                if (loaded == 0) return;
                addAll(rec, loaded);
            }
        }
        unsigned these[LOADS][RW], next[LOADS][RW];
        int loaded = load(these);
        while (loaded > 0) {
            const int more = load(next);
            addAll(these, loaded);
            if (more == 0) break;
            loaded = load(these);
            addAll(next, more);
        }
    }

    /** Calls term(element, value) for the terms of a record. */
    template <typename Term>
    __device__ __forceinline__ static void forEachTerm(const unsigned (&rec)[RW], const Term& term)
    {
        const int tid = threadIdx.x;
        const unsigned eL = rec[0] & 0xffffu, eH = rec[0] >> 16;   // both inside this slice
        float wL, wH;
        Layout::weights(rec, wL, wH);
#pragma unroll
        for (int step = 0; step < F; ++step) {
            // Neighbouring lanes take the features in rotated order: an entry starts at a multiple of
            // 8 * F bytes, so lanes that all add feature `step` meet on a few LDS banks (measured on a
            // dense grid with 8 features: conflicts 90 % of the LDS cycles of this kernel).
            const int i = (F & (F - 1)) == 0 ? ((step + tid) & (F - 1)) : ((step + tid % F) % F);
            unsigned word = rec[Layout::FIRST_ADJOINT];
            const int at = FLOATS ? i : i >> 1;
#pragma unroll
            for (int w = 1; w < Layout::ADJOINT_WORDS; ++w) word = at == w ? rec[Layout::FIRST_ADJOINT + w] : word;
            const float adj = FLOATS ? __builtin_bit_cast(float, word)
                : static_cast<float>(__builtin_bit_cast(f16, static_cast<unsigned short>(word >> (16 * (i & 1)))));
            term(eL + i, wL * adj);
            term(eH + i, wH * adj);
        }
    }

    /** \param overwrite the elements of the slice are written, whatever is there; those that others add to as well are zero */
    __device__ __forceinline__ static void run(int numel, const GridGradientWorkspace& ws, float* __restrict__ gradients,
                                               const GridGradientSlice item, int overwrite, long long* sSlice, Shared& shared)
    {
        const int tid = threadIdx.x;
        const int begin = static_cast<int>(static_cast<long long>(ws.regions) * item.part / item.parts);
        const int end = static_cast<int>(static_cast<long long>(ws.regions) * (item.part + 1) / item.parts);
        // everything that has to be looked up first, in flight while the sums are zeroed
        const unsigned segment = tid < min(SEGMENTS, end - begin) ? segmentOf(ws, item, begin + tid) : 0u;
        unsigned largest = 0u;
        for (int i = tid; i < ws.largestCount; i += BLOCK) largest = max(largest, ws.largest[i]);
        const int sums = item.floats < SLICE_FLOATS ? item.floats : SUMS;
        for (int i = tid; i < sums; i += BLOCK) sSlice[i] = 0;
        int records = static_cast<int>(segment >> 16) - static_cast<int>(segment & 0xffffu);
        const int most = 2 * STEPS << groupLog2(ws, item);   // twice a part of a segment
        bool some = records > most;
        for (int r = begin + SEGMENTS + tid; r < end; r += BLOCK) {
            const unsigned s = segmentOf(ws, item, r);
            const int size = static_cast<int>(s >> 16) - static_cast<int>(s & 0xffffu);
            records += size;
            some = some || size > most;
        }
        const bool any = __ballot(some) != 0;
#pragma unroll
        for (int d = 32; d > 0; d /= 2) {
            largest = max(largest, static_cast<unsigned>(__shfl_xor(static_cast<int>(largest), d, 64)));
            if constexpr (FLOATS) records += __shfl_xor(records, d, 64);
        }
        shared.segments[tid] = segment;
        if (tid % 64 == 0) {
            shared.largest[tid / 64] = largest | (any ? LONG_SEGMENTS : 0u);
            if constexpr (FLOATS) shared.records[tid / 64] = records;
        }
        if (tid == 0) shared.smallCount = 0;
        __syncthreads();
        unsigned maxBits = 0u, flags = 0u;
        int allRecords = 0;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            maxBits = max(maxBits, shared.largest[w] & ~LONG_SEGMENTS);
            flags |= shared.largest[w];
            if constexpr (FLOATS) allRecords += shared.records[w];
        }
        const bool uneven = (__builtin_amdgcn_readfirstlane(flags) & LONG_SEGMENTS) != 0 && isUneven(ws, item, begin, end, shared);
        const bool finite = maxBits < (FLOATS ? 0x7f800000u : 0x7c00u);
        // |adjoint| < 2^maxExponent: 2^(biased exponent - 14) of halves, 2^(biased exponent - 126) of floats, subnormals included
        const int maxExponent = FLOATS ? static_cast<int>(maxBits >> 23) - 126 : static_cast<int>(maxBits >> 10) - 14;
        // Terms of at most the largest adjoint (weights <= 1) that one sum may take. Halves: those of the whole batch, so that
        // a slice gives the same bits however its records are split. Floats need the bits below more: the records of this
        // work item (the two weights of a record make at most one).
        const unsigned long long terms = FLOATS ? static_cast<unsigned long long>(allRecords) + 1ull
                                                : static_cast<unsigned long long>(2 * Layout::PAIRS) * static_cast<unsigned long long>(numel);
        const int termsLog2 = 64 - __builtin_clzll(terms);
        const int scaleExponent = min(61 - termsLog2, FIXED_BITS) - maxExponent;
        const double scale = ldexp(1.0, scaleExponent), unit = ldexp(1.0, -scaleExponent);
        float* sFloat = reinterpret_cast<float*>(sSlice);
        // Floats span more than the 64 bits of a sum: a value of which the sum would lose bits is added to the gradient tensor. Of few
        // records behind the sums, from a list (or if that is full by another pass over the records); many records have more
        // of these than a list holds, as each halves the unit of the sums: they are added right away, to what is there or to zeros.
        // (One level of 64^3 nodes x 4, 2^20 points: a second pass for lists that were full made 64 us of 33.)
        const float smallest = ldexpf(1.f, 23 - scaleExponent);
        (void)smallest;
        float* __restrict__ grad = gradients + item.first;
        const int firstOwn = item.parts > 1 ? sums : item.slice > 0 ? F : 0;   // (see below)
        const bool direct = FLOATS && static_cast<long long>(__builtin_amdgcn_readfirstlane(allRecords)) * (2 * F) > MOST_TERMS_WITH_LIST;
        if (direct) {
            if (overwrite)
                for (int i = firstOwn + tid; i < min(sums, SLICE_FLOATS); i += BLOCK) grad[i] = 0.f;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wavefront's stores have been carried out
            __syncthreads();
        }
        if (maxBits == 0u) {
            // all adjoints are zero: nothing to add
        } else if (finite) {
            forEachRecord<false>(ws, item, begin, end, uneven, shared, [&](const unsigned (&rec)[RW]) {
                forEachTerm(rec, [&](unsigned element, float v) {
                    if constexpr (FLOATS) {
                        if (fabsf(v) < smallest) {
                            if (v != 0.f && direct) {
                                unsafeAtomicAdd(grad + element, v);
                            } else if (v != 0.f) {
                                const int at = atomicAdd(&shared.smallCount, 1);
                                if (at < SMALL) {
                                    shared.smallValues[at] = v;
                                    shared.smallElements[at] = static_cast<unsigned short>(element);
                                }
                            }
                            return;
                        }
                    }
                    ldsAddFixed(sSlice + element, toFixed(v, scale));
                });
            });
        } else {
            forEachRecord<true>(ws, item, begin, end, uneven, shared, [&](const unsigned (&rec)[RW]) {
                forEachTerm(rec, [&](unsigned element, float v) { Grid::ldsAdd(sFloat + element, v); });
            });
        }
        if (direct) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wavefront's atomics have been carried out
        __syncthreads();
        // Added to the gradient tensor: with atomics (16 neighbouring floats per request) where other work
        // items hold sums for the same slice (parts > 1), and for the first entry of a slice and the one behind it, to
        // which two slices add; else this workgroup is the only writer of its slice in this launch.
        auto sumOf = [&](int i) { return finite ? static_cast<float>(static_cast<double>(sSlice[i]) * unit) : sFloat[i]; };
        if (direct) {
#pragma unroll 1
            for (int i = tid; i < sums; i += BLOCK) {
                const float v = sumOf(i);
                if (v == 0.f) continue;
                if (i < firstOwn || i >= SLICE_FLOATS) unsafeAtomicAdd(grad + i, v);
                // (read behind this workgroup's own atomics: they have ended, but the L1 does not know of them)
                else grad[i] = __hip_atomic_load(grad + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + v;
            }
            return;
        }
        for (int i = tid; i < sums; i += BLOCK) {
            const float v = sumOf(i);
            if (i < firstOwn || i >= SLICE_FLOATS) {
                if (v != 0.f) unsafeAtomicAdd(grad + i, v);
            } else if (overwrite) {
                grad[i] = v;
            } else if (v != 0.f) {
                grad[i] += v;
            }
        }
        if constexpr (FLOATS) {
            const int small = shared.smallCount;
            if (small == 0) return;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wavefront's stores have been carried out
            __syncthreads();
            if (small <= SMALL) {
                if (tid < small) unsafeAtomicAdd(grad + shared.smallElements[tid], shared.smallValues[tid]);
            } else {
                // (the segments of the first regions, where others have taken their place)
                shared.segments[tid] = tid < min(SEGMENTS, end - begin) ? segmentOf(ws, item, begin + tid) : 0u;
                __syncthreads();
                forEachRecord<true>(ws, item, begin, end, uneven, shared, [&](const unsigned (&rec)[RW]) {
                    forEachTerm(rec, [&](unsigned element, float v) {
                        if (fabsf(v) < smallest && v != 0.f) unsafeAtomicAdd(grad + element, v);
                    });
                });
            }
        }
    }
};

/** One workgroup of 1024 lanes per work item; `items` is indexed by the workgroup; (SLICE_FLOATS + Features) * 8 bytes of dynamic LDS. */
template <typename Cfg, int SLICE_FLOATS, bool FLOATS>
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(GridGradientSlices<Cfg, SLICE_FLOATS, FLOATS>::WAVES_PER_SIMD)))
GridGradientSlicesKernel(
    int numel, const GridGradientWorkspace workspace, float* __restrict__ gradients, const GridGradientSlice* __restrict__ items, int overwrite)
{
    typedef GridGradientSlices<Cfg, SLICE_FLOATS, FLOATS> Impl;
    extern __shared__ __align__(16) unsigned char sMemory[];
    __shared__ typename Impl::Shared shared;
    Impl::run(numel, workspace, gradients, items[blockIdx.x], overwrite, reinterpret_cast<long long*>(sMemory), shared);
}

QUICKMLP_KERNEL_NAMESPACE_END
