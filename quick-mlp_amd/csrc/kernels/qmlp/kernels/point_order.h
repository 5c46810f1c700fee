// Orders the points of a batch by the slab of a grid they fall into, so that the
// wavefronts that run side by side gather from the same few megabytes of the table and
// find them in L1 / L2, and the lanes of one gather instruction fall onto fewer cache lines. A counting sort over at most 1024 slabs in three launches, without
// atomics on device memory (a first version reserved the ranges with one returning atomic per
// slab and workgroup: 256 workgroups on the same 64 cache lines took 120 us):
//   PointOrderCount   one histogram per workgroup (summed in LDS) over its chunk of the batch,
//   PointOrderScan    per slab, the running sum over the workgroups (in place) and the total,
//   PointOrderScatter scans the totals into slab offsets, sorts its chunk in LDS and writes
//                     it to slab offset + running sum + rank in the chunk: a copy of the
//                     input rows in sorted order and, per sorted position, the index of the
//                     point in the caller's batch (and, for training passes, per point its sorted position).
// The order of the points of one chunk inside a slab depends on the timing of the wavefronts;
// the fused kernel evaluates every point on its own, so its results do not.
// No counterpart in the reference, which evaluates the points in the order given.

#include <qmlp/kernels/common.h>
#include <qmlp/kernels/point_order_key.h>

QUICKMLP_KERNEL_NAMESPACE_BEGIN

constexpr int POINT_ORDER_MAX_SLABS = 1024;
constexpr int POINT_ORDER_BLOCK = 1024;
constexpr int POINT_ORDER_POINTS_PER_THREAD = 4;    // a workgroup's chunk: 4096 points (offsets in it take 12 bits)
constexpr int POINT_ORDER_SCAN_SLABS = 16;          // slabs per workgroup of PointOrderScan

/**
 * The chunk of this workgroup. Workgroups go to the 8 dies in turn; a die takes consecutive chunks, whose points of a slab lie side by
 * side in the sorted batch: what is read or written of a line by several of them meets in its L2.
 */
__device__ __forceinline__ unsigned pointOrderChunk()
{
    constexpr unsigned dies = DIES;
    const unsigned die = blockIdx.x % dies;
    return die * (gridDim.x / dies) + min(die, gridDim.x % dies) + blockIdx.x / dies;
}

/** Slab of one coordinate value, clamped to the box (the comparisons are false for NaN, which then lands in slab 0). */
__device__ __forceinline__ int pointOrderSlab1(float value, float lo, float scale, int slabs)
{
    const float p = (value - lo) * scale;
    return p > 0.f ? static_cast<int>(fminf(p, static_cast<float>(slabs - 1))) : 0;
}

/** Slab of a point: up to three grid coordinates, clamped to the box. channel(c): the value of input channel c. */
template <typename Channel>
__device__ __forceinline__ int pointOrderSlabOf(const Channel& channel, const PointOrderKey& key)
{
    int s = pointOrderSlab1(channel(key.channel0), key.min0, key.scale0, key.slabs0);
    if (key.slabs1 > 1) {
        const int s1 = pointOrderSlab1(channel(key.channel1), key.min1, key.scale1, key.slabs1);
        if (key.slabs2 > 1) {
            const int s2 = pointOrderSlab1(channel(key.channel2), key.min2, key.scale2, key.slabs2);
            if (key.interleave12) {
                // bit b of s1 to position 2b + 1, of s2 to 2b (at most 5 bits each)
                int z = 0;
#pragma unroll
                for (int b = 0; b < 5; ++b) z |= ((s1 >> b) & 1) << (2 * b + 1) | ((s2 >> b) & 1) << (2 * b);
                s = s * (key.slabs1 * key.slabs2) + z;
            } else {
                s = (s * key.slabs1 + s1) * key.slabs2 + s2;
            }
        } else {
            s = s * key.slabs1 + s1;
        }
    }
    return s;
}

/** Slab of the point in row `index` of the inputs. */
__device__ __forceinline__ int pointOrderSlab(const Tensor2Read<float>& inputs, long long index, const PointOrderKey& key)
{
    const float* row = inputs.data_ + index * inputs.strides_[0];
    const long long channelStride = inputs.strides_[1];
    return pointOrderSlabOf([&](int c) { return row[static_cast<long long>(c) * channelStride]; }, key);
}

/** histogram: (workgroups, POINT_ORDER_MAX_SLABS), every entry is written. */
__global__ void __launch_bounds__(POINT_ORDER_BLOCK) PointOrderCount(
    int numel, const Tensor2Read<float> inputs, const PointOrderKey key, int* __restrict__ histogram)
{
    __shared__ int sCount[POINT_ORDER_MAX_SLABS];
    sCount[threadIdx.x] = 0;
    __syncthreads();
    const long long chunk = static_cast<long long>(blockIdx.x) * (POINT_ORDER_BLOCK * POINT_ORDER_POINTS_PER_THREAD);
#pragma unroll
    for (int k = 0; k < POINT_ORDER_POINTS_PER_THREAD; ++k) {
        const long long index = chunk + k * POINT_ORDER_BLOCK + threadIdx.x;
        if (index < numel) atomicAdd(&sCount[pointOrderSlab(inputs, index, key)], 1);
    }
    __syncthreads();
    histogram[blockIdx.x * POINT_ORDER_MAX_SLABS + threadIdx.x] = sCount[threadIdx.x];
}

/**
 * histogram[w][slab] becomes the number of points of the slab in the chunks before w,
 * totals[slab] their number in all chunks. A workgroup takes POINT_ORDER_SCAN_SLABS slabs; 64 groups of
 * its threads take a 64th of the chunks each: sum, exchange through LDS (a wavefront adds up a slab's), running sum; a thread's first chunks
 * stay in its registers in between. All loads of a batch are asked for without a branch for the lane, behind which each would be
 * waited for (512 chunks 6.7 -> 5.2 us, 147 chunks 4.9 -> 3.2). (64 workgroups: with 16 workgroups of 64 slabs the pass took 8 us for 256
 * chunks and 13 us for 512.)
 */
__global__ void __launch_bounds__(POINT_ORDER_BLOCK) PointOrderScan(int chunks, int* __restrict__ histogram, int* __restrict__ totals)
{
    constexpr int GROUPS = POINT_ORDER_BLOCK / POINT_ORDER_SCAN_SLABS;
    constexpr int BATCH = 8;   // loads in flight
    static_assert(GROUPS == WAVE_SIZE && POINT_ORDER_BLOCK / WAVE_SIZE == POINT_ORDER_SCAN_SLABS, "a wavefront per slab, a lane per group");
    __shared__ int sPartial[POINT_ORDER_SCAN_SLABS][GROUPS + 1];
    const int local = threadIdx.x % POINT_ORDER_SCAN_SLABS, group = threadIdx.x / POINT_ORDER_SCAN_SLABS;
    int* const counts = histogram + blockIdx.x * POINT_ORDER_SCAN_SLABS + local;
    const int perGroup = (chunks + GROUPS - 1) / GROUPS;
    const int begin = min(group * perGroup, chunks), end = min(begin + perGroup, chunks);
    int v[BATCH], sum = 0;
    auto load = [&](int w0) {
#pragma unroll
        for (int j = 0; j < BATCH; ++j) v[j] = counts[min(w0 + j, chunks - 1) * POINT_ORDER_MAX_SLABS];
#pragma unroll
        for (int j = 0; j < BATCH; ++j) v[j] = w0 + j < end ? v[j] : 0;
    };
    for (int w0 = begin + BATCH; w0 < end; w0 += BATCH) {
        load(w0);
#pragma unroll
        for (int j = 0; j < BATCH; ++j) sum += v[j];
    }
    load(begin);   // (last: they are still held below)
#pragma unroll
    for (int j = 0; j < BATCH; ++j) sum += v[j];
    sPartial[local][group] = sum;
    __syncthreads();
    {
        const int slab = threadIdx.x / WAVE_SIZE, lane = threadIdx.x % WAVE_SIZE;
        const int own = sPartial[slab][lane], inclusive = waveInclusiveScan(own);
        sPartial[slab][lane] = inclusive - own;
        if (lane == WAVE_SIZE - 1) totals[blockIdx.x * POINT_ORDER_SCAN_SLABS + slab] = inclusive;
    }
    __syncthreads();
    int running = sPartial[local][group];
    for (int w0 = begin; w0 < end; w0 += BATCH) {
        if (w0 > begin) load(w0);
#pragma unroll
        for (int j = 0; j < BATCH; ++j) {
            if (w0 + j < end) counts[(w0 + j) * POINT_ORDER_MAX_SLABS] = running;
            running += v[j];
        }
    }
}

/** Exclusive scan over the POINT_ORDER_MAX_SLABS values held one per thread of the workgroup. */
__device__ __forceinline__ int pointOrderBlockScan(int value, int* sWaveSum)
{
    constexpr int WAVES = POINT_ORDER_MAX_SLABS / WAVE_SIZE;
    static_assert(WAVES <= WAVE_SIZE, "a lane per wavefront");
    const int lane = threadIdx.x % WAVE_SIZE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
    const int inclusive = waveInclusiveScan(value);
    __syncthreads();   // sWaveSum may still be read from a previous scan
    if (lane == WAVE_SIZE - 1) sWaveSum[wave] = inclusive;
    __syncthreads();
    const int sums = waveInclusiveScan(lane < WAVES ? sWaveSum[lane] : 0);
    return (wave > 0 ? __builtin_amdgcn_readlane(sums, wave - 1) : 0) + inclusive - value;
}

/** The channels of N input rows, all of them asked for before the first is waited for; one load of 8, 12 or 16 bytes where the layout allows it
 *  (vectorChannels > 0: rows of that many channels with unit stride between them, aligned to the vector). index(k): the row, one that is there. */
template <int MAX_CHANNELS, int N, typename Index>
__device__ __forceinline__ void pointOrderLoadRows(const Tensor2Read<float>& inputs, const Index& index, int vectorChannels, float (&rows)[N][MAX_CHANNELS])
{
    typedef float f32x2a __attribute__((ext_vector_type(2)));
    typedef float f32x3a __attribute__((ext_vector_type(3), aligned(4)));
    typedef float f32x4a __attribute__((ext_vector_type(4)));
    const float* src[N];
#pragma unroll
    for (int k = 0; k < N; ++k) src[k] = inputs.data_ + index(k) * inputs.strides_[0];
    // (the branches fill vectors: stores to the array in each of them become one store to an address that depends on the
    // branch, and the array moves to scratch memory)
    f32x4a first[N] = {};
    if (MAX_CHANNELS >= 4 && vectorChannels == 4) {
#pragma unroll
        for (int k = 0; k < N; ++k) first[k] = *reinterpret_cast<const f32x4a*>(src[k]);
    } else if (MAX_CHANNELS >= 3 && vectorChannels == 3) {
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const f32x3a v = *reinterpret_cast<const f32x3a*>(src[k]);
            first[k] = f32x4a{v[0], v[1], v[2], 0.f};
        }
    } else if (MAX_CHANNELS >= 2 && vectorChannels == 2) {
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const f32x2a v = *reinterpret_cast<const f32x2a*>(src[k]);
            first[k] = f32x4a{v[0], v[1], 0.f, 0.f};
        }
    } else {
#pragma unroll
        for (int c = 0; c < 4 && c < MAX_CHANNELS; ++c)
            if (c < inputs.sizes_[1]) {
#pragma unroll
                for (int k = 0; k < N; ++k) first[k][c] = src[k][static_cast<long long>(c) * inputs.strides_[1]];
            }
    }
#pragma unroll
    for (int k = 0; k < N; ++k)
#pragma unroll
        for (int c = 0; c < 4 && c < MAX_CHANNELS; ++c) rows[k][c] = first[k][c];
#pragma unroll
    for (int c = 4; c < MAX_CHANNELS; ++c)
#pragma unroll
        for (int k = 0; k < N; ++k) rows[k][c] = c < inputs.sizes_[1] ? src[k][static_cast<long long>(c) * inputs.strides_[1]] : 0.f;
}

/** How the rows of inputs can be loaded as one vector each (pointOrderLoadRows), 0 if they cannot. */
__device__ __forceinline__ int pointOrderVectorChannels(const Tensor2Read<float>& inputs)
{
    const int channels = inputs.sizes_[1];
    if (inputs.strides_[1] != 1) return 0;
    const unsigned long long base = reinterpret_cast<unsigned long long>(inputs.data_);
    if (channels == 4 && inputs.strides_[0] % 4 == 0 && base % 16 == 0) return 4;
    if (channels == 3) return 3;   // three words from an address that is a multiple of four
    if (channels == 2 && inputs.strides_[0] % 2 == 0 && base % 8 == 0) return 2;
    return 0;
}

/** Writes the channels of one row of the sorted copy; one store of 8, 12 or 16 bytes where the rows came as vectors. */
template <int MAX_CHANNELS>
__device__ __forceinline__ void pointOrderStoreRow(float* __restrict__ sortedInputs, long long position, int channels, int vectorChannels,
                                                   const float (&row)[MAX_CHANNELS])
{
    typedef float f32x3a __attribute__((ext_vector_type(3), aligned(4)));
    if (MAX_CHANNELS >= 4 && vectorChannels == 4) {
        *reinterpret_cast<float4*>(sortedInputs + position * 4) = make_float4(row[0], row[1], row[2 % MAX_CHANNELS], row[3 % MAX_CHANNELS]);
    } else if (MAX_CHANNELS >= 3 && vectorChannels == 3) {
        const f32x3a v = {row[0], row[1], row[2 % MAX_CHANNELS]};
        *reinterpret_cast<f32x3a*>(sortedInputs + position * 3) = v;
    } else if (MAX_CHANNELS >= 2 && vectorChannels == 2) {
        *reinterpret_cast<float2*>(sortedInputs + position * 2) = make_float2(row[0], row[1]);
    } else {
#pragma unroll
        for (int c = 0; c < MAX_CHANNELS; ++c)
            if (c < channels) sortedInputs[position * channels + c] = row[c];
    }
}

/** An entry of the sorted chunk in LDS. */
template <bool STAGED_ROWS> struct PointOrderEntry { typedef unsigned int type; };
template <> struct PointOrderEntry<true> { typedef unsigned short type; };

/**
 * The workgroup sorts its chunk by slab in LDS, then walks the sorted chunk with consecutive lanes on
 * consecutive positions, so that the stores of a wavefront fall into a few runs (a scatter straight from the
 * unsorted chunk sent every lane's stores to a line of their own and took 80 us for 2^21 points).
 * Rows of up to four channels are read once, in the order given (consecutive lanes, consecutive rows), and wait
 * in LDS at their sorted place. Reading them a second time in sorted order, as wider rows still are, asks for 64
 * lines per instruction, many of which the chunks of the other workgroups have meanwhile pushed out of the L2 (14 us for
 * 2^21 rows of 16 bytes). Two workgroups share a compute unit, so that one loads while the other stores. Bound by the lines that are written
 * in part: a chunk has four rows for a slab, and the chunk behind it the next four of the same line (pointOrderChunk: 2^21 rows of 16 bytes
 * 27 -> 21 us, 10^6 rows 15 -> 13, 700 000 rows 11; 75 MB at 3.5 TB/s). With the slab of each sorted point in LDS too, one workgroup had
 * 94 KiB, and its rows went through scratch memory, because the compiler turned choices among registers into
 * addresses: 40 and 17 us.
 * \tparam MAX_CHANNELS at least the number of input channels (4, 8, 16)
 */
template <int MAX_CHANNELS>
__global__ void __launch_bounds__(POINT_ORDER_BLOCK) PointOrderScatter(
    int numel, const Tensor2Read<float> inputs, const PointOrderKey key,
    const int* __restrict__ histogram,  // as PointOrderScan left it
    const int* __restrict__ totals,
    float* __restrict__ sortedInputs,   // (numel, inputs.sizes_[1]), dense, 16-byte aligned
    int* __restrict__ order,            // (numel): sorted position -> index in the batch
    int* __restrict__ placement)        // null, or (numel): index in the batch -> sorted position (consecutive lanes, consecutive words)
{
    constexpr int CHUNK = POINT_ORDER_BLOCK * POINT_ORDER_POINTS_PER_THREAD;
    constexpr bool STAGE_ROWS = MAX_CHANNELS <= 4;
    // 78 KiB with staged rows: two workgroups per compute unit
    __shared__ int sCount[POINT_ORDER_MAX_SLABS];        // points of the chunk per slab; then from a place in the sorted chunk to that in the batch
    __shared__ unsigned short sLocalStart[POINT_ORDER_MAX_SLABS];   // of a slab in the sorted chunk
    __shared__ int sWaveSum[POINT_ORDER_BLOCK / WAVE_SIZE];
    // sorted chunk: the offset of the point in the chunk (the slab then comes from the row again), or slab << 16 | offset
    typedef typename PointOrderEntry<STAGE_ROWS>::type entry_t;
    __shared__ entry_t sSorted[CHUNK];
    __shared__ __align__(16) float sRows[STAGE_ROWS ? CHUNK * MAX_CHANNELS : 4];   // the rows of the sorted chunk
    const int t = threadIdx.x;

    const int channels = inputs.sizes_[1];
    const int vectorChannels = pointOrderVectorChannels(inputs);
    const unsigned chunkIndex = pointOrderChunk();
    const long long chunk = static_cast<long long>(chunkIndex) * CHUNK;
    const int chunkPoints = static_cast<int>(min(static_cast<long long>(CHUNK), numel - chunk));
    auto slabOf = [&](const float (&row)[MAX_CHANNELS]) {
        static_assert(MAX_CHANNELS >= 4, "a row in a vector");
        // (single values that the compiler knows nothing about: a choice among those of an array it makes an index into scratch memory)
        float v0 = row[0], v1 = row[1], v2 = row[2], v3 = row[3];
        asm("" : "+v"(v0), "+v"(v1), "+v"(v2), "+v"(v3));
        return pointOrderSlabOf([&](int c) { return c == 0 ? v0 : c == 1 ? v1 : c == 2 ? v2 : v3; }, key);
    };
    constexpr int N = POINT_ORDER_POINTS_PER_THREAD;
    int slab[N], rank[N];
    float rows[STAGE_ROWS ? N : 1][MAX_CHANNELS] = {};
    (void)rows;
    const int before = histogram[chunkIndex * POINT_ORDER_MAX_SLABS + t], total = totals[t];
    // (lanes behind the last point: that one again)
    if constexpr (STAGE_ROWS)
        pointOrderLoadRows<MAX_CHANNELS>(inputs, [&](int k) { return chunk + min(k * POINT_ORDER_BLOCK + t, chunkPoints - 1); }, vectorChannels, rows);
    sCount[t] = 0;
    const int slabStart = pointOrderBlockScan(total, sWaveSum) + before;   // holds a barrier after sCount = 0
#pragma unroll
    for (int k = 0; k < N; ++k) {
        slab[k] = 0;
        rank[k] = 0;
        const int j = k * POINT_ORDER_BLOCK + t;
        if (j < chunkPoints) {
            if constexpr (STAGE_ROWS) slab[k] = slabOf(rows[k]);
            else slab[k] = pointOrderSlab(inputs, chunk + j, key);
            rank[k] = atomicAdd(&sCount[slab[k]], 1);
        }
    }
    __syncthreads();
    const int localStart = pointOrderBlockScan(sCount[t], sWaveSum);
    sLocalStart[t] = static_cast<unsigned short>(localStart);   // (4096 only behind the last point)
    sCount[t] = slabStart - localStart;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < POINT_ORDER_POINTS_PER_THREAD; ++k) {
        const int j = k * POINT_ORDER_BLOCK + t;
        if (j < chunkPoints) {
            const int at = sLocalStart[slab[k]] + rank[k];
            sSorted[at] = static_cast<entry_t>(STAGE_ROWS ? j : slab[k] << 16 | j);
            if (placement) placement[chunk + j] = sCount[slab[k]] + at;
            if constexpr (STAGE_ROWS) {
#pragma unroll
                for (int c = 0; c < MAX_CHANNELS; ++c) sRows[at * MAX_CHANNELS + c] = rows[k][c];
            }
        }
    }
    __syncthreads();

    if constexpr (STAGE_ROWS) {
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const int j = k * POINT_ORDER_BLOCK + t;
            if (j >= chunkPoints) continue;
            float row[MAX_CHANNELS];
#pragma unroll
            for (int c = 0; c < MAX_CHANNELS; ++c) row[c] = sRows[j * MAX_CHANNELS + c];
            const long long position = sCount[slabOf(row)] + j;
            order[position] = static_cast<int>(chunk + sSorted[j]);
            pointOrderStoreRow<MAX_CHANNELS>(sortedInputs, position, channels, vectorChannels, row);
        }
    } else {
        // (two rows of up to 16 channels in flight)
        constexpr int AHEAD = 2;
#pragma unroll 1
        for (int k0 = 0; k0 < N; k0 += AHEAD) {
            float row[AHEAD][MAX_CHANNELS];
            auto entryOf = [&](int k) -> unsigned { return sSorted[min((k0 + k) * POINT_ORDER_BLOCK + t, chunkPoints - 1)]; };
            pointOrderLoadRows<MAX_CHANNELS>(inputs, [&](int k) { return chunk + (entryOf(k) & 0xffffu); }, vectorChannels, row);
#pragma unroll
            for (int k = 0; k < AHEAD; ++k) {
                const int j = (k0 + k) * POINT_ORDER_BLOCK + t;
                if (j >= chunkPoints) continue;
                const unsigned entry = entryOf(k);
                const long long position = sCount[entry >> 16] + j;
                order[position] = static_cast<int>(chunk + (entry & 0xffffu));
                pointOrderStoreRow<MAX_CHANNELS>(sortedInputs, position, channels, vectorChannels, row[k]);
            }
        }
    }
}

/**
 * Rows that were computed in the sorted order, added to the caller's tensor: dst[j, c] += src[placement[j], c]
 * (src dense), or written to it. The rows of dst are walked in their own order, so the read-modify-write is coalesced
 * and only the reads of src are scattered (2^21 rows of 16 bytes: 76 us as a scatter through `order`, whose rows of 16
 * bytes each cost a line read and a line written). Rows of 16 bytes move as one load and one store, four rows of a lane
 * in flight (43 us with a lane per element, 27 us so, written and not added to). Bound by the lines of src: a chunk's rows of a slab are
 * half a line, and the rest of it belongs to the chunks beside it, which the same die therefore takes (22 us; 10^6 rows 13 -> 10).
 */
__global__ void __launch_bounds__(POINT_ORDER_BLOCK) PointOrderGatherAddRows(
    long long elements, int channels, const float* __restrict__ src, const int* __restrict__ placement, Tensor2RW<float> dst, int overwrite)
{
    if (channels == 4 && dst.strides_[1] == 1 && dst.strides_[0] % 4 == 0 && reinterpret_cast<unsigned long long>(dst.data_) % 16 == 0
        && reinterpret_cast<unsigned long long>(src) % 16 == 0) {
        constexpr int ROWS = 4;
        const long long rows = elements / 4;
        for (long long first = static_cast<long long>(pointOrderChunk()) * (ROWS * POINT_ORDER_BLOCK) + threadIdx.x; first < rows;
             first += static_cast<long long>(gridDim.x) * (ROWS * POINT_ORDER_BLOCK)) {
            // (lanes behind the last row: that one again)
            int from[ROWS];
            float4 v[ROWS], old[ROWS];
#pragma unroll
            for (int k = 0; k < ROWS; ++k) from[k] = placement[min(first + k * POINT_ORDER_BLOCK, rows - 1)];
#pragma unroll
            for (int k = 0; k < ROWS; ++k) {
                v[k] = reinterpret_cast<const float4*>(src)[from[k]];
                old[k] = make_float4(0.f, 0.f, 0.f, 0.f);
            }
            if (!overwrite) {
#pragma unroll
                for (int k = 0; k < ROWS; ++k)
                    old[k] = *reinterpret_cast<const float4*>(dst.data_ + min(first + k * POINT_ORDER_BLOCK, rows - 1) * dst.strides_[0]);
            }
#pragma unroll
            for (int k = 0; k < ROWS; ++k) {
                const long long row = first + k * POINT_ORDER_BLOCK;
                if (row < rows)
                    *reinterpret_cast<float4*>(dst.data_ + row * dst.strides_[0])
                        = make_float4(old[k].x + v[k].x, old[k].y + v[k].y, old[k].z + v[k].z, old[k].w + v[k].w);
            }
        }
        return;
    }
    for (long long e = static_cast<long long>(blockIdx.x) * POINT_ORDER_BLOCK + threadIdx.x; e < elements;
         e += static_cast<long long>(gridDim.x) * POINT_ORDER_BLOCK) {
        const long long row = e / channels;
        const int c = static_cast<int>(e - row * channels);
        float* target = dst.data_ + row * dst.strides_[0] + static_cast<long long>(c) * dst.strides_[1];
        const float v = src[static_cast<long long>(placement[row]) * channels + c];
        *target = overwrite ? v : *target + v;
    }
}

QUICKMLP_KERNEL_NAMESPACE_END
