// Template of the adjoint kernel that runs the layers again and sums all weight gradients, workgroup by workgroup.
// The host code generator replaces everything in $$..$$ before the source is handed to the compiler.
//
// A workgroup of 4 or 8 wavefronts takes tiles of 32 points per wavefront. From the encoded input (read from the
// forward memory, or, where the only encoding is an identity, straight from the input rows: the training pass then
// stores nothing at all) a wavefront runs the layers forward, keeps the pre-activations in registers, and goes back
// layer by layer; the weight gradients of a layer are formed by the workgroup from rows in LDS
// (layer_cooperative.h), two workgroup barriers per layer. For the adjoint of the encoded input: the input gradients
// of identity encodings are added here, those of grids are left to the kernels behind this one.
//
// 16 -> 64 x 4 -> 4, 10^6 points: 128 us under the profiler (154 with the adjoint of ReLU as comparisons, its output computed three times and the rows of a
// tile waited for one after the other). 683 vector instructions per 32 points, 172 of them matrix products: a SIMD issues the former for 27 % of the
// time and has its matrix cores busy for 27 %, which hardly overlap, the LDS is at work for half of it (conflicts 15 %), wavefronts wait
// for a third of theirs, and 173 MB of memory traffic make 1.4 TB/s. 4 -> 128 -> 64 -> 48 -> 4 with sines, 2^20 points: 231 us (302 while it spilled
// 232 bytes per lane), vector instructions 52 %, matrix cores 18 %, LDS 34 %. Slower or the same: one wavefront per SIMD with all gradient tiles
// and no barriers (+25 %), or with 64 points (+20 %); fewer vector instructions (outputs of the sines kept or the first layer's pre-activations
// formed again by matrix instructions, masks left out of full tiles: 0 to 2 %); other paddings of the rows; other orders between the barriers.
//
// Replaces, like network_backward.h, NetworkKernelBackward of the reference
// (src_cpp/include/qmlp/kernels/network_backward.cuh:33-114) and its weight update
// (network_weight_update_block.cuh:356-494).

#include <qmlp/kernels/common.h>
#include <qmlp/kernels/arrays.h>
#include <qmlp/kernels/layer_cooperative.h>

$$INCLUDES$$

QUICKMLP_KERNEL_NAMESPACE_BEGIN

namespace activations
{
$$DEFINE_ACTIVATIONS$$
    // stands for "no activation": the input of the first layer
    struct passthrough_
    {
        static __device__ __forceinline__ half forward(half x) { return x; }
        static __device__ __forceinline__ f16x4 forward4(f16x4 x) { return x; }
    };
}

__global__ void __launch_bounds__($$BLOCK_SIZE$$) $$KERNEL_ATTRIBUTES$$ NetworkKernelBackwardCooperative(
    int numel,
    const Tensor2Read<float> inputs,      //shape (numel, Cin)
    const Tensor2Read<float> adjOutputs,  //shape (numel, Cout)
    Tensor2RW<float> adjInputs,           //shape (numel, Cin), accumulated; unused without input gradients
    const half* __restrict__ networkParametersH,
    const half* __restrict__ forwardTmpMemoryH,  //the encoded input, 64-point tiles (unused with DIRECT_INPUT)
    half* __restrict__ adjointTmpMemoryH,        //receives the adjoint of the encoded input (STORE_ENCODED_ADJOINT)
    float* __restrict__ partialGradients,        //partialSlices x the layout of the parameters; workgroup b stores the sums of
    int partialSlices,                           //its tiles into slice b (and zeroes slices b + k * gridDim.x)
    const int* __restrict__ adjOutputOrder,      //nullptr, or (numel) the row of adjOutputs that belongs to point p
    int overwriteInputs                          //adjInputs holds nothing yet: written, not added to
    $$ENCODING_PARAMETERS$$)
{
    constexpr int NUM_INPUTS = $$NUM_INPUTS$$;
    constexpr int ENCODED_CHANNELS = $$ENCODED_CHANNELS$$;
    constexpr int CHANNELS_IN = $$CHANNELS_IN$$;
    constexpr int CHANNELS_OUT = $$CHANNELS_OUT$$;
    constexpr int KT0 = CHANNELS_IN / 16;
    constexpr int MTL = CHANNELS_OUT / 16;
    constexpr int WAVES = $$BLOCK_SIZE$$ / WAVE_SIZE;
    constexpr int NUM_PARAMETERS = $$NUM_PARAMETERS$$;
    constexpr int ROWS_PER_WAVE = $$ROWS_PER_WAVE$$;   // halves
    constexpr bool HAS_INPUT_GRADIENTS = $$HAS_INPUT_GRADIENTS$$;         // of encodings that are differentiated here
    constexpr bool NEEDS_ENCODING_ADJOINT = $$NEEDS_ENCODING_ADJOINT$$;   // here or in the kernels behind this one
    constexpr bool STORE_ENCODED_ADJOINT = $$STORE_ENCODED_ADJOINT$$;
    // >= 0: the only encoding is an identity encoding of the input channels from this one on
    constexpr int DIRECT_INPUT_START = $$DIRECT_INPUT_START$$;
    constexpr bool DIRECT_INPUT = DIRECT_INPUT_START >= 0;
    (void)ENCODED_CHANNELS; (void)NUM_INPUTS;

    const f16* __restrict__ networkParameters = reinterpret_cast<const f16*>(networkParametersH);
    const f16* __restrict__ forwardTmpMemory = reinterpret_cast<const f16*>(forwardTmpMemoryH);
    f16* __restrict__ adjointTmpMemory = reinterpret_cast<f16*>(adjointTmpMemoryH);
    (void)forwardTmpMemory; (void)adjointTmpMemory;

    extern __shared__ __align__(16) unsigned char sMemory[];
    f16* sParams = reinterpret_cast<f16*>(sMemory);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
    const int lane = threadIdx.x % WAVE_SIZE;
    const int g = lane >> 4, r = lane & 15;
    f16* sRowsAll = sParams + $$LDS_PARAM_HALVES$$;
    f16* sRows = sRowsAll + wave * ROWS_PER_WAVE;

$$STAGE_PARAMETERS$$
$$DECLARE_WEIGHT_GRADIENTS$$
    __syncthreads();

    const int numTiles = (numel + TILE_POINTS - 1) / TILE_POINTS;
    const int actualChannelsOut = adjOutputs.sizes_[1];
    const bool adjOutputRowsOfFloat4 = actualChannelsOut % 4 == 0 && adjOutputs.strides_[1] == 1 && adjOutputs.strides_[0] % 4 == 0
        && reinterpret_cast<unsigned long long>(adjOutputs.data_) % 16 == 0;
    const bool inputRowsOfFloat4 = DIRECT_INPUT && DIRECT_INPUT_START % 4 == 0 && ENCODED_CHANNELS % 4 == 0 && inputs.strides_[1] == 1
        && inputs.strides_[0] % 4 == 0 && reinterpret_cast<unsigned long long>(inputs.data_) % 16 == 0;
    (void)inputRowsOfFloat4;
    const int numGroups = (numel + WAVES * COOP_POINTS - 1) / (WAVES * COOP_POINTS);

    // What a wavefront reads of its 32 points: dL/dy and the input rows, or the encoded input as the forward kernel stored it
    // (channel-major tiles of 64 points, zero outside the batch). Asked for a group of tiles ahead, and without a branch
    // around any load but what is the same for the whole launch: behind branches for lanes every load was waited for
    // before the next was asked for, six times the latency of the memory per tile. Lanes without a point or
    // a channel read another one's, which takeChannels leaves out.
    f32x4 dyAhead[COOP_NT][MTL];
    f32x4 inputAhead[DIRECT_INPUT ? COOP_NT : 1][DIRECT_INPUT ? KT0 : 1];
    f16x2 encodedAhead[DIRECT_INPUT ? 1 : KT0][4];
    (void)inputAhead; (void)encodedAhead;
    auto loadRows = [&](int group) {
        const int ahead = (group < numGroups ? group : numGroups - 1) * WAVES + wave;
        int point[COOP_NT];
#pragma unroll
        for (int nt = 0; nt < COOP_NT; ++nt) point[nt] = min(ahead * COOP_POINTS + 2 * r + nt, numel - 1);
        auto loadAdjoints = [&](const int (&rows)[COOP_NT]) {
            if (adjOutputRowsOfFloat4) {
#pragma unroll
                for (int nt = 0; nt < COOP_NT; ++nt)
#pragma unroll
                    for (int m = 0; m < MTL; ++m)
                        dyAhead[nt][m] = *reinterpret_cast<const f32x4*>(adjOutputs.data_ + static_cast<long long>(rows[nt]) * adjOutputs.strides_[0]
                                                                         + min(16 * m + 4 * g, actualChannelsOut - 4));
            } else {
#pragma unroll
                for (int nt = 0; nt < COOP_NT; ++nt)
#pragma unroll
                    for (int m = 0; m < MTL; ++m)
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            dyAhead[nt][m][i] = adjOutputs.data_[static_cast<long long>(rows[nt]) * adjOutputs.strides_[0]
                                                                 + static_cast<long long>(min(16 * m + 4 * g + i, actualChannelsOut - 1)) * adjOutputs.strides_[1]];
            }
        };
        // (twice, and the order waited for at once: merged, the way without an order would wait wherever the other one might have to)
        if (adjOutputOrder) {
            int rows[COOP_NT];
#pragma unroll
            for (int nt = 0; nt < COOP_NT; ++nt) rows[nt] = adjOutputOrder[point[nt]];
#pragma unroll
            for (int nt = 0; nt < COOP_NT; ++nt) asm volatile("" : "+v"(rows[nt]));
            loadAdjoints(rows);
        } else {
            loadAdjoints(point);
        }
        if constexpr (DIRECT_INPUT) {
            if (inputRowsOfFloat4) {
#pragma unroll
                for (int nt = 0; nt < COOP_NT; ++nt)
#pragma unroll
                    for (int t = 0; t < KT0; ++t)
                        inputAhead[nt][t] = *reinterpret_cast<const f32x4*>(inputs.data_ + static_cast<long long>(point[nt]) * inputs.strides_[0] + DIRECT_INPUT_START
                                                                            + min(16 * t + 4 * g, ENCODED_CHANNELS - 4));
            } else {
#pragma unroll
                for (int nt = 0; nt < COOP_NT; ++nt)
#pragma unroll
                    for (int t = 0; t < KT0; ++t)
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            inputAhead[nt][t][i] = inputs.data_[static_cast<long long>(point[nt]) * inputs.strides_[0]
                                                                + static_cast<long long>(DIRECT_INPUT_START + min(16 * t + 4 * g + i, ENCODED_CHANNELS - 1)) * inputs.strides_[1]];
            }
        } else {
            const int tileAhead = ahead >> 1;
            const f16* encTile = forwardTmpMemory + static_cast<long long>(tileAhead < numTiles ? tileAhead : numTiles - 1) * (CHANNELS_IN * TILE_POINTS)
                + (ahead & 1) * COOP_POINTS + 2 * r;
#pragma unroll
            for (int t = 0; t < KT0; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) encodedAhead[t][i] = *reinterpret_cast<const f16x2*>(encTile + (16 * t + 4 * g + i) * TILE_POINTS);
        }
    };
    // (fp32 -> fp16, zero outside batch / real channels)
    auto takeChannels = [&](f32x4 v, bool pv, int c, int channels) {
        f16x4 out = toF16(v);
#pragma unroll
        for (int i = 0; i < 4; ++i) out[i] = pv && c + i < channels ? out[i] : static_cast<f16>(0);
        return out;
    };
    loadRows(blockIdx.x);
    for (int group = blockIdx.x; group < numGroups; group += gridDim.x)
    {
        const int half32 = group * WAVES + wave;               // this wavefront's 32 points
        const int point0 = half32 * COOP_POINTS + 2 * r;       // points 2r and 2r + 1 of them
        const int tile = half32 >> 1;
        unsigned valid[COOP_NT];
        f16x4 dyOut[COOP_NT][MTL];
        f16x4 x0[COOP_NT][KT0];
#pragma unroll
        for (int nt = 0; nt < COOP_NT; ++nt) {
            const bool pv = point0 + nt < numel;
            valid[nt] = pv ? ~0u : 0u;
#pragma unroll
            for (int m = 0; m < MTL; ++m) dyOut[nt][m] = takeChannels(dyAhead[nt][m], pv, 16 * m + 4 * g, actualChannelsOut);
            if constexpr (DIRECT_INPUT) {
#pragma unroll
                for (int t = 0; t < KT0; ++t) x0[nt][t] = takeChannels(inputAhead[nt][t], pv, 16 * t + 4 * g, ENCODED_CHANNELS);
            }
        }
        if constexpr (!DIRECT_INPUT) {
#pragma unroll
            for (int t = 0; t < KT0; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    x0[0][t][i] = encodedAhead[t][i][0];
                    x0[1][t][i] = encodedAhead[t][i][1];
                }
        }

        // the layers forward, pre-activations kept; then last to first
$$CALL_NETWORK_LAYERS$$

        if constexpr (STORE_ENCODED_ADJOINT) {
            if (tile < numTiles) {
                f16* adjTile = adjointTmpMemory + static_cast<long long>(tile) * (CHANNELS_IN * TILE_POINTS) + (half32 & 1) * COOP_POINTS + 2 * r;
#pragma unroll
                for (int t = 0; t < KT0; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const f16x2 v = {dxIn[0][t][i], dxIn[1][t][i]};
                        *reinterpret_cast<f16x2*>(adjTile + (16 * t + 4 * g + i) * TILE_POINTS) = v;
                    }
            }
        }
        if constexpr (HAS_INPUT_GRADIENTS && DIRECT_INPUT) {
            // a lane holds the gradients of 4 channels side by side
            const bool rowsOfFloat4 = DIRECT_INPUT_START % 4 == 0 && adjInputs.strides_[1] == 1 && adjInputs.strides_[0] % 4 == 0
                && reinterpret_cast<unsigned long long>(adjInputs.data_) % 16 == 0;
#pragma unroll
            for (int nt = 0; nt < COOP_NT; ++nt) {
                if (point0 + nt >= numel) continue;
                float* row = adjInputs.data_ + static_cast<long long>(point0 + nt) * adjInputs.strides_[0]
                    + static_cast<long long>(DIRECT_INPUT_START) * adjInputs.strides_[1];
#pragma unroll
                for (int t = 0; t < KT0; ++t) {
                    const int c = 16 * t + 4 * g;
                    if (16 * t + 15 < ENCODED_CHANNELS && rowsOfFloat4) {
                        f32x4* target = reinterpret_cast<f32x4*>(row + c);
                        f32x4 v = __builtin_convertvector(dxIn[nt][t], f32x4);
                        if (!overwriteInputs) v = *target + v;
                        *target = v;
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            if (c + i < ENCODED_CHANNELS) {
                                float* target = row + static_cast<long long>(c + i) * adjInputs.strides_[1];
                                const float v = static_cast<float>(dxIn[nt][t][i]);
                                *target = overwriteInputs ? v : *target + v;
                            }
                    }
                }
            }
        }
        if constexpr (HAS_INPUT_GRADIENTS && !DIRECT_INPUT) {
            // the adjoint of the encoded input: registers -> a row per point (the rows of this wavefront are free: the last
            // barrier of layer 0 is behind) -> one lane per point
            constexpr int STAGE_STRIDE = CHANNELS_IN + 8;
#pragma unroll
            for (int nt = 0; nt < COOP_NT; ++nt)
#pragma unroll
                for (int t = 0; t < KT0; ++t)
                    *reinterpret_cast<f16x4*>(sRows + (2 * r + nt) * STAGE_STRIDE + 16 * t + 4 * g) = dxIn[nt][t];
            waveLdsSync();
            const int index = half32 * COOP_POINTS + lane;
            if (lane < COOP_POINTS && index < numel) {
                StaticArray<float, NUM_INPUTS> encodingInput;
#pragma unroll
                for (int i = 0; i < NUM_INPUTS; ++i)
                    encodingInput[i] = inputs.data_[static_cast<long long>(index) * inputs.strides_[0]
                                                    + static_cast<long long>(i) * inputs.strides_[1]];
                StaticArray<float, NUM_INPUTS> adjEncodingInput;
#pragma unroll
                for (int i = 0; i < NUM_INPUTS; ++i) adjEncodingInput[i] = 0.f;
                WrappedArray<const f16> adjEncodingOutput{sRows + lane * STAGE_STRIDE};
$$CALL_ENCODINGS$$
                float* adjRow = adjInputs.data_ + static_cast<long long>(index) * adjInputs.strides_[0];
#pragma unroll
                for (int i = 0; i < NUM_INPUTS; ++i) {
                    float* target = adjRow + static_cast<long long>(i) * adjInputs.strides_[1];
                    *target = overwriteInputs ? adjEncodingInput[i] : *target + adjEncodingInput[i];
                }
            }
            waveLdsSync();
        }
    }
$$STORE_WEIGHT_GRADIENTS$$
}

QUICKMLP_KERNEL_NAMESPACE_END
