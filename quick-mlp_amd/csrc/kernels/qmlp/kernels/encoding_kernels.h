// Template of the standalone encoding kernels (fp32 in, fp32 out). Everything in
// $$..$$ is replaced by the host before compilation.
// Replaces src_cpp/include/qmlp/kernels/encoding_kernels.cuh:26-62 of the reference.

#include <qmlp/kernels/common.h>
#include <qmlp/kernels/arrays.h>
#include <qmlp/kernels/encoding_level_shares.h>

$$INCLUDES$$

QUICKMLP_KERNEL_NAMESPACE_BEGIN

/**
 * One lane per point. The rows of a wavefront's 64 points are put together in LDS and written side by side (a lane that
 * writes its own row touches one line per value and point; 16 levels of 2 floats, 2^17 points 80 -> 70 us, where the
 * lines of the gathers bound it).
 * A grid whose levels stand next to each other in the output may be evaluated by GROUPS times as many workgroups, each
 * of them a few of the levels: a small batch leaves few wavefronts, each of which waits for one level's entries after the
 * other's (2^10 / 2^14 / 2^15 / 2^16 / 2^17 points 21 / 30 / 32 / 42 / 70 us, with 8 groups 6.5 / 13 / 23 / 48 / 91 us; the
 * same with half tables 17 / 30 / 30 / 35 / 49 and 6.4 / 10 / 17 / 33 / 62 us: the rows are then written in pieces).
 */
__global__ void __launch_bounds__(256) EncodingForwardKernel(
    long long numel,
    const Tensor2Read<float> inputs,  //shape (numel, Cin)
    Tensor2RW<float> outputs          //shape (numel, Cout), unit stride along the channels
    $$ENCODING_PARAMETERS$$)
{
    constexpr int GROUPS = $$LEVEL_GROUPS$$;
    constexpr int CHANNELS = $$GROUP_CHANNELS$$;   // of the widest group
    constexpr bool STAGED = CHANNELS > 1 && CHANNELS <= 62;
    constexpr int PITCH = CHANNELS | 1;
    __shared__ float sRows[256 / WAVE_SIZE][STAGED ? TILE_POINTS * PITCH : 1];
    const int lane = threadIdx.x % WAVE_SIZE;
    float* rows = sRows[threadIdx.x / WAVE_SIZE];
    const int group = blockIdx.x % GROUPS;
    const int firstChannel = $$FIRST_CHANNEL$$, channels = $$CHANNELS$$;   // of this group
    for (long long tileBase = (blockIdx.x / GROUPS * static_cast<long long>(blockDim.x / WAVE_SIZE) + threadIdx.x / WAVE_SIZE) * TILE_POINTS;
         tileBase < numel; tileBase += static_cast<long long>(blockDim.x) * (gridDim.x / GROUPS))
    {
        const long long index = tileBase + lane;
        if (index < numel) {
            const StridedArray<const float> encodingInput{inputs.data_ + index * inputs.strides_[0], inputs.strides_[1]};
            WrappedArray<float> encodingOutput{STAGED ? rows + lane * PITCH : outputs.data_ + index * outputs.strides_[0] + firstChannel};
            $$CALL_ENCODINGS_FORWARD$$
        }
        if constexpr (STAGED) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            const int points = static_cast<int>(min(numel - tileBase, static_cast<long long>(TILE_POINTS)));
            for (int i = lane; i < points * CHANNELS; i += WAVE_SIZE) {
                const int row = i / CHANNELS, channel = i % CHANNELS;
                if (channel < channels) outputs.data_[(tileBase + row) * outputs.strides_[0] + firstChannel + channel] = rows[row * PITCH + channel];
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
    }
}

#if $$BY_LEVELS$$
/**
 * Larger batches of grids of many levels, rows without gaps: the dies share out the levels (encoding_level_shares.h), so that a
 * level's table is brought into the L2 of one die, or two, instead of all eight. Workgroups go to the dies in turn. A wavefront takes one
 * level of 64 points; the values of a tile of 64 points lie level by level where its rows will be, for EncodingRowsKernel.
 * 16 levels of 2^19 entries of 2 floats, 2^16 / 2^17 / 2^18 / 2^20 points: 37 / 64 / 116 / 437 us with EncodingRowsKernel,
 * EncodingForwardKernel 42 / 70 / 182 / 771 (of 2 halves 29 / 49 / 95 / 364 and 35 / 49 / 132 / 568; which of them:
 * IEncoding::forwardByLevels). Bound by the lines of 128 bytes that the L1s get from the L2, 64 to 68 per point.
 */
__global__ void __launch_bounds__(256) EncodingLevelsKernel(
    long long numel,
    const Tensor2Read<float> inputs,  //shape (numel, Cin)
    float* __restrict__ outputs       //(numel, Cout) without gaps
    $$ENCODING_PARAMETERS$$)
{
    typedef $$ENCODING$$ Encoding;
    constexpr int L = Encoding::L, F = Encoding::F;
    static_assert(ENCODING_LEVEL_WAVES == 256 / WAVE_SIZE, "a workgroup");
    constexpr int TILES[L] = {$$LEVEL_TILES$$};   // of a wavefront
    const int lane = threadIdx.x % WAVE_SIZE;
    const int tiles = static_cast<int>((numel + TILE_POINTS - 1) / TILE_POINTS);
    int left = blockIdx.x % DIES * (gridDim.x / DIES) + blockIdx.x / DIES, level = -1, perWave = 1;
#pragma unroll
    for (int l = 0; l < L; ++l) {
        const int workgroups = (tiles + TILES[l] * ENCODING_LEVEL_WAVES - 1) / (TILES[l] * ENCODING_LEVEL_WAVES);
        if (level < 0) {
            if (left < workgroups) {
                level = l;
                perWave = TILES[l];
            } else {
                left -= workgroups;
            }
        }
    }
    if (level < 0) return;
    const int first = left * perWave * ENCODING_LEVEL_WAVES + threadIdx.x / WAVE_SIZE;
    for (int i = 0; i < perWave; ++i) {
        const int tile = first + i * ENCODING_LEVEL_WAVES;
        if (tile >= tiles) return;
        const long long begin = static_cast<long long>(tile) * TILE_POINTS;
        const int points = static_cast<int>(min(numel - begin, static_cast<long long>(TILE_POINTS)));
        if (lane >= points) return;   // (of the last tile)
        const StridedArray<const float> encodingInput{inputs.data_ + (begin + lane) * inputs.strides_[0], inputs.strides_[1]};
        float features[F];
        Encoding::featuresOfLevel(level, encodingInput, cEncoding, features);
        float* target = outputs + begin * (L * F) + (level * points + lane) * F;
#pragma unroll
        for (int c = 0; c < F; ++c) target[c] = features[c];
    }
}

/** The values of EncodingLevelsKernel, tile by tile, into rows in their place. A wavefront reads a tile before it writes it. */
__global__ void __launch_bounds__(TILE_POINTS) EncodingRowsKernel(long long numel, float* outputs)
{
    typedef $$ENCODING$$ Encoding;
    constexpr int L = Encoding::L, F = Encoding::F, CHANNELS = L * F, PITCH = CHANNELS | 1;
    static_assert(CHANNELS <= ENCODING_ROWS_MAX_CHANNELS, "LDS of a workgroup");
    __shared__ float rows[TILE_POINTS * PITCH];
    const int lane = threadIdx.x;
    const long long tileBase = blockIdx.x * static_cast<long long>(TILE_POINTS);
    const int points = static_cast<int>(min(numel - tileBase, static_cast<long long>(TILE_POINTS)));
    float* tile = outputs + tileBase * CHANNELS;
    if (lane < points) {
        float values[CHANNELS];
#pragma unroll
        for (int l = 0; l < L; ++l)
#pragma unroll
            for (int i = 0; i < F; ++i) values[l * F + i] = tile[(l * points + lane) * F + i];
#pragma unroll
        for (int c = 0; c < CHANNELS; ++c) rows[lane * PITCH + c] = values[c];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if constexpr (CHANNELS % 4 == 0) {
        typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
        for (int i = lane; i < points * (CHANNELS / 4); i += WAVE_SIZE) {
            const float* from = rows + i / (CHANNELS / 4) * PITCH + i % (CHANNELS / 4) * 4;
            *reinterpret_cast<f32x4u*>(tile + 4 * i) = f32x4u{from[0], from[1], from[2], from[3]};
        }
    } else {
        for (int i = lane; i < points * CHANNELS; i += WAVE_SIZE) tile[i] = rows[i / CHANNELS * PITCH + i % CHANNELS];
    }
}
#endif

#if $$SHARED_TILE$$
// Small batches of grids of many levels: the wavefronts of a workgroup share the levels of 64 points, which one wavefront
// would walk through one after the other (16 levels of 2 halves, 2^13 points, both gradients: 75 -> 41 us).
__global__ void __launch_bounds__(512) EncodingAdjointSharedKernel(
    long long numel,
    const Tensor2Read<float> inputs,      //shape (numel, Cin)
    const Tensor2Read<float> adjOutputs,  //shape (numel, Cout)
    Tensor2RW<float> adjInputs            //shape (numel, Cin), accumulated
    $$ENCODING_PARAMETERS$$)
{
    typedef $$ENCODING$$ Encoding;
    constexpr int WAVES = $$SHARED_WAVES$$;   // of the workgroup
    constexpr bool INPUT_GRADIENTS = $$INPUT_GRADIENTS$$;
    __shared__ float sLevels[INPUT_GRADIENTS ? Encoding::L * Encoding::D * TILE_POINTS : 1];
    const int lane = threadIdx.x % WAVE_SIZE;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
    for (long long tileBase = static_cast<long long>(blockIdx.x) * TILE_POINTS; tileBase < numel; tileBase += static_cast<long long>(gridDim.x) * TILE_POINTS) {
        const long long index = tileBase + lane, point = min(index, numel - 1);
        const StridedArray<const float> encodingInput{inputs.data_ + point * inputs.strides_[0], inputs.strides_[1]};
        const StridedArray<const float> encodingAdjOutput{adjOutputs.data_ + point * adjOutputs.strides_[0], adjOutputs.strides_[1]};
        Encoding::adjointShared<WAVES, INPUT_GRADIENTS, $$PARAMETER_GRADIENTS$$>(
            wave, lane, tileBase, numel, inputs, encodingInput, encodingAdjOutput,
            [&](int pt, int c) { return adjOutputs.data_[(tileBase + pt) * adjOutputs.strides_[0] + static_cast<long long>(c) * adjOutputs.strides_[1]]; },
            cEncoding, sLevels);
        if constexpr (INPUT_GRADIENTS) {
            __syncthreads();
            if (wave == 0 && index < numel) {
                StridedArray<float> encodingAdjInput{adjInputs.data_ + index * adjInputs.strides_[0], adjInputs.strides_[1]};
                Encoding::finishShared(encodingAdjInput, cEncoding, sLevels, lane);
            }
            __syncthreads();
        }
    }
}
#endif

// One wavefront takes 64 consecutive points at a time: one lane per point for the input
// gradients, then all lanes together for the parameter gradients of grid encodings (groups
// of lanes add neighbouring table entries in one atomic request).
__global__ void __launch_bounds__(256) EncodingAdjointKernel(
    long long numel,
    const Tensor2Read<float> inputs,      //shape (numel, Cin)
    const Tensor2Read<float> adjOutputs,  //shape (numel, Cout)
    Tensor2RW<float> adjInputs            //shape (numel, Cin), accumulated
    $$ENCODING_PARAMETERS$$)
{
    const int lane = threadIdx.x % WAVE_SIZE;
    const long long wavesPerBlock = blockDim.x / WAVE_SIZE;
    const long long stride = wavesPerBlock * gridDim.x * TILE_POINTS;
    for (long long tileBase = (blockIdx.x * wavesPerBlock + threadIdx.x / WAVE_SIZE) * TILE_POINTS; tileBase < numel;
         tileBase += stride)
    {
        const long long index = tileBase + lane;
        if (index < numel) {
            const StridedArray<const float> encodingInput{inputs.data_ + index * inputs.strides_[0], inputs.strides_[1]};
            const StridedArray<const float> encodingAdjOutput{adjOutputs.data_ + index * adjOutputs.strides_[0], adjOutputs.strides_[1]};
            StridedArray<float> encodingAdjInput{adjInputs.data_ + index * adjInputs.strides_[0], adjInputs.strides_[1]};
            $$CALL_ENCODINGS_ADJOINT$$
        }
        $$CALL_ENCODINGS_SCATTER$$
    }
}

// Test aid: table offsets and interpolation weights of every corner of every level.
__global__ void EncodingCornersKernel(
    long long numel,
    const Tensor2Read<float> inputs,  //shape (numel, Cin)
    unsigned* __restrict__ indices,   //shape (numel, perPoint)
    float* __restrict__ weights,      //shape (numel, perPoint)
    int perPoint
    $$ENCODING_PARAMETERS$$)
{
    for (long long index = blockIdx.x * static_cast<long long>(blockDim.x) + threadIdx.x; index < numel;
         index += static_cast<long long>(blockDim.x) * gridDim.x)
    {
        const StridedArray<const float> encodingInput{inputs.data_ + index * inputs.strides_[0], inputs.strides_[1]};
        unsigned* cornerIndices = indices + index * perPoint;
        float* cornerWeights = weights + index * perPoint;
        (void)encodingInput; (void)cornerIndices; (void)cornerWeights;
        $$CALL_ENCODINGS_CORNERS$$
    }
}

// Test aid: the same two arrays, written by the code the fused kernels run. MODE 1: the
// gathers of the forward pass (one lane per point); MODE 2: the gradient scatter of the
// backward pass (one wavefront per 64 points), which records where it would add.
template <int MODE>
__global__ void __launch_bounds__(256) EncodingTraceKernel(
    long long numel,
    const Tensor2Read<float> inputs,  //shape (numel, Cin)
    unsigned* __restrict__ indices,   //shape (numel, perPoint)
    float* __restrict__ weights,      //shape (numel, perPoint)
    int perPoint
    $$ENCODING_PARAMETERS$$)
{
    if constexpr (MODE == 1) {
        for (long long index = blockIdx.x * static_cast<long long>(blockDim.x) + threadIdx.x; index < numel;
             index += static_cast<long long>(blockDim.x) * gridDim.x)
        {
            const StridedArray<const float> encodingInput{inputs.data_ + index * inputs.strides_[0], inputs.strides_[1]};
            unsigned* cornerIndices = indices + index * perPoint;
            float* cornerWeights = weights + index * perPoint;
            (void)encodingInput; (void)cornerIndices; (void)cornerWeights;
            $$CALL_ENCODINGS_TRACE_GATHER$$
        }
    } else {
        const int lane = threadIdx.x % WAVE_SIZE;
        const long long wavesPerBlock = blockDim.x / WAVE_SIZE;
        const long long stride = wavesPerBlock * gridDim.x * TILE_POINTS;
        (void)lane;
        for (long long tileBase = (blockIdx.x * wavesPerBlock + threadIdx.x / WAVE_SIZE) * TILE_POINTS; tileBase < numel;
             tileBase += stride)
        {
            $$CALL_ENCODINGS_TRACE_SCATTER$$
        }
    }
}

QUICKMLP_KERNEL_NAMESPACE_END
