// Template of the standalone encoding kernels (fp32 in, fp32 out). Everything in
// $$..$$ is replaced by the host before compilation.
// Replaces src_cpp/include/qmlp/kernels/encoding_kernels.cuh:26-62 of the reference.

#include <qmlp/kernels/common.h>
#include <qmlp/kernels/arrays.h>

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
