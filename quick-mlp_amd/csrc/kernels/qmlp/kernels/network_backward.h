// Template of the fused adjoint kernel. The host code generator replaces everything
// in $$..$$ before the source is handed to the runtime compiler.
//
// Per 64-point wavefront tile: dL/dy is loaded straight into the accumulator layout
// of the matrix cores, each layer (last to first) applies the activation adjoint on
// the stored pre-activations and contracts with the transposed weights
// (dX = W^T dpre, the same MFMA path as the forward pass with the weight tiles
// staged transposed). For the weight gradients dpre is either stored for the weight-update
// kernels or, where the gradient tiles of all layers fit into the registers of a wavefront,
// contracted with the layer input right here (Layer::weightGradient), the workgroup storing
// its partial sums after its last tile. Where all layers are summed here, the training pass may
// have kept the encoded input only: the kernel then runs the layers forward once more per tile
// (Layer::forwardKeep) instead of reading their pre-activations back. The adjoint of
// the encoded input finally goes through the LDS staging rows to one lane per point,
// which accumulates input gradients and scatter-adds grid gradients with hardware
// fp32 atomics.
//
// Replaces NetworkKernelBackward of the reference
// (src_cpp/include/qmlp/kernels/network_backward.cuh:33-114). Unlike the reference it
// never reads dL/dy beyond the real output channels: padded channels are zero.

#include <qmlp/kernels/common.h>
#include <qmlp/kernels/arrays.h>
#include <qmlp/kernels/layer.h>

$$INCLUDES$$

QUICKMLP_KERNEL_NAMESPACE_BEGIN

namespace activations
{
$$DEFINE_ACTIVATIONS$$
    // stands for "no activation": the stored input of the first layer is its input
    struct passthrough_
    {
        static __device__ __forceinline__ half forward(half x) { return x; }
    };
}

/**
 * dst (cin, cout) row-major = transpose of src (cout, cin) row-major. Run before the adjoint
 * kernel for layers whose weights are too large to stay in LDS: the adjoint kernel then reads
 * its matrix-core operands (rows of W^T) from global memory with two 8-byte loads per lane.
 */
__global__ void __launch_bounds__(256) TransposeWeightsKernel(const half* __restrict__ src, half* __restrict__ dst,
                                                              int cout, int cin)
{
    __shared__ half tile[16][17];
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const int tilesX = cin / 16;
    for (int t = blockIdx.x; t < tilesX * (cout / 16); t += gridDim.x) {
        const int o0 = (t / tilesX) * 16, k0 = (t % tilesX) * 16;
        tile[ty][tx] = src[(o0 + ty) * cin + k0 + tx];
        __syncthreads();
        dst[(k0 + ty) * cout + o0 + tx] = tile[tx][ty];
        __syncthreads();
    }
}

__global__ void __launch_bounds__($$BLOCK_SIZE$$) $$KERNEL_ATTRIBUTES$$ NetworkKernelBackward(
    int numel,
    const Tensor2Read<float> inputs,      //shape (numel, Cin)
    const Tensor2Read<float> adjOutputs,  //shape (numel, Cout)
    Tensor2RW<float> adjInputs,           //shape (numel, Cin), accumulated; unused without input gradients
    const half* __restrict__ networkParametersH,
    const half* __restrict__ forwardTmpMemoryH,  //written by the forward kernel
    half* __restrict__ adjointTmpMemoryH,        //receives dpre if weight gradients are requested
    const half* __restrict__ transposedWeightsH, //W^T of the layers whose weights do not stay in LDS, or nullptr
    float* __restrict__ partialGradients,        //FUSED_WEIGHT_UPDATE: partialSlices x the layout of the parameters; workgroup b
    int partialSlices                            //stores the sums of its tiles into slice b (and zeroes slices b + k * gridDim.x)
#if $$HAS_OUTPUT_ORDER$$
    // Networks whose batches may train in sorted order: nullptr, or (numel) the row of adjOutputs that belongs to
    // point p. The parameter and its code exist only in the kernels of such networks: with them the run-time compiler
    // scheduled the kernel of 64 -> 64 x 4 -> 4 (which never sorts) so that it took 689 instead of 372 us.
    , const int* __restrict__ adjOutputOrder
#endif
    $$ENCODING_PARAMETERS$$)
{
    constexpr int NUM_INPUTS = $$NUM_INPUTS$$;
    constexpr int ENCODED_CHANNELS = $$ENCODED_CHANNELS$$;
    constexpr int CHANNELS_IN = $$CHANNELS_IN$$;
    constexpr int CHANNELS_OUT = $$CHANNELS_OUT$$;
    constexpr int KT0 = CHANNELS_IN / 16;
    constexpr int MTL = CHANNELS_OUT / 16;
    constexpr int STAGE_STRIDE = CHANNELS_IN + 8;
    constexpr int LDS_PARAM_HALVES = $$LDS_PARAM_HALVES$$;
    constexpr int WAVES = $$BLOCK_SIZE$$ / WAVE_SIZE;
    constexpr bool HAS_INPUT_GRADIENTS = $$HAS_INPUT_GRADIENTS$$;
    constexpr bool HAS_NETWORK_GRADIENTS = $$HAS_NETWORK_GRADIENTS$$;
    constexpr bool HAS_ENCODING_GRADIENTS = $$HAS_ENCODING_GRADIENTS$$;
    // Some layers' weights are staged into a shared LDS buffer right before the layer runs:
    // the wavefronts of the workgroup then walk the tiles and layers in lockstep (workgroup
    // barriers inside the loop), wavefronts without a tile work on zeros.
    constexpr bool HAS_STREAMED_LAYERS = $$HAS_STREAMED_LAYERS$$;
    // the adjoint of the encoded input is only needed if something sits behind it
    constexpr bool NEEDS_ENCODING_ADJOINT = $$NEEDS_ENCODING_ADJOINT$$;
    // true: the adjoint of the encoded rows is stored (channel-major per tile, behind the adjoint
    // pre-activations) for the kernels that sum the parameter gradients of grids slice by slice
    constexpr bool STORE_ENCODED_ADJOINT = $$STORE_ENCODED_ADJOINT$$;
    constexpr int OFFSET_ENCODED_ADJOINT = $$OFFSET_ENCODED_ADJOINT$$;   // channels in front of that region
    // false: nothing in this kernel reads the adjoint of an encoded row point by point
    constexpr bool NEEDS_STAGED_ADJOINT = $$NEEDS_STAGED_ADJOINT$$;
    // true: the weight gradients are summed in this kernel and dpre is not stored
    constexpr bool FUSED_WEIGHT_UPDATE = $$FUSED_WEIGHT_UPDATE$$;
    // true, for small batches of networks with grids of many levels: the workgroup takes one tile, its first wavefront runs the
    // layers and all of them share the levels of the grids, which one wavefront would walk through one after the other (16
    // levels of 2 halves, 64 -> 64 -> 64 -> 1, 2000 points, with input gradients: 84 -> 33 us)
    constexpr bool SHARED_TILE = $$SHARED_TILE$$;
    constexpr int GROUP_TILES = SHARED_TILE ? 1 : WAVES;
    constexpr bool STORE_DPRE = HAS_NETWORK_GRADIENTS;   // of the layers that have a weight-update kernel
    (void)FUSED_WEIGHT_UPDATE;
    constexpr int NUM_PARAMETERS = $$NUM_PARAMETERS$$;
    (void)STORE_DPRE; (void)NUM_PARAMETERS;
    (void)ENCODED_CHANNELS; (void)NUM_INPUTS; (void)KT0; (void)STAGE_STRIDE;

    const f16* __restrict__ networkParameters = reinterpret_cast<const f16*>(networkParametersH);
    const f16* __restrict__ forwardTmpMemory = reinterpret_cast<const f16*>(forwardTmpMemoryH);
    f16* __restrict__ adjointTmpMemory = reinterpret_cast<f16*>(adjointTmpMemoryH);
    const f16* __restrict__ transposedWeights = reinterpret_cast<const f16*>(transposedWeightsH);
    (void)transposedWeights;

    extern __shared__ __align__(16) unsigned char sMemory[];
    f16* sParams = reinterpret_cast<f16*>(sMemory);
    const int wave = threadIdx.x / WAVE_SIZE;
    const int lane = threadIdx.x % WAVE_SIZE;
    const int g = lane >> 4, r = lane & 15;
    f16* sStage = sParams + LDS_PARAM_HALVES + (SHARED_TILE ? 0 : wave) * (TILE_POINTS * STAGE_STRIDE);
    (void)sStage;
    // FUSED_WEIGHT_UPDATE: this wavefront's tile of adjoint pre-activations, a row of 64 points per channel
    f16* sTranspose = reinterpret_cast<f16*>(sMemory + $$OFFSET_TRANSPOSE$$) + wave * $$TRANSPOSE_HALVES$$;
    (void)sTranspose;
    // RECOMPUTE: behind it, this wavefront's tile of the input of the layer whose weight gradients are being summed
    f16* sLayerInput = sTranspose + $$LAYER_INPUT_OFFSET$$;
    (void)sLayerInput;

    // stage the transposed weights in operand order
$$STAGE_PARAMETERS$$
    // FUSED_WEIGHT_UPDATE: the gradient tiles of this wavefront, summed over its tiles of the batch
$$DECLARE_WEIGHT_GRADIENTS$$
    // gradients of coarse grid levels are summed in LDS first (zeroed here, added to the
    // gradient tensor once per workgroup after the loop over the tiles)
$$ZERO_LDS_GRADIENTS$$
    __syncthreads();

    const int numTiles = (numel + TILE_POINTS - 1) / TILE_POINTS;
    const long long numel64 = static_cast<long long>(numTiles) * TILE_POINTS;
    const int actualChannelsOut = adjOutputs.sizes_[1];
    const bool adjOutputRowsOfFloat2 = actualChannelsOut == 2 && adjOutputs.strides_[1] == 1 && adjOutputs.strides_[0] % 2 == 0
        && reinterpret_cast<unsigned long long>(adjOutputs.data_) % 8 == 0;
    const bool adjOutputRowsOfFloat4 = actualChannelsOut % 4 == 0 && adjOutputs.strides_[1] == 1 && adjOutputs.strides_[0] % 4 == 0
        && reinterpret_cast<unsigned long long>(adjOutputs.data_) % 16 == 0;
    // Kernels that run the layers again read little per tile: dL/dy and the encoded input of this wavefront's next tile
    // are asked for one tile ahead, behind the order of a sorted batch (the row of dL/dy) that is asked for two ahead. A
    // wavefront's tiles follow each other with nothing else to hide the latency of three dependent loads (12 -> 16 -> 32 x 3
    // -> 2 with a grid, 2^21 points: 154 -> 92 us; 112 while the rows of a tile were waited for one after the other).
    constexpr bool LOADS_AHEAD = $$RECOMPUTES$$ && MTL == 1 && KT0 <= 2 && !HAS_STREAMED_LAYERS;
    const int firstTile = static_cast<int>(blockIdx.x) * WAVES + wave, tileStep = static_cast<int>(gridDim.x) * WAVES;
    (void)firstTile; (void)tileStep;
    // No branch around a load but what is the same for the whole launch: behind branches for lanes every load was waited for before the next
    // was asked for. Lanes without a point or a channel read another one's, which is left out below.
#if $$HAS_OUTPUT_ORDER$$
    // a batch that trains in sorted order: the rows of dL/dy of this wavefront's next tile, asked for one tile ahead
    int adjRowAhead[NT];
    auto loadRows = [&](int tile) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) adjRowAhead[nt] = min(tile * TILE_POINTS + 4 * r + nt, numel - 1);
        if (adjOutputOrder) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) adjRowAhead[nt] = adjOutputOrder[adjRowAhead[nt]];
        }
    };
    loadRows(firstTile < numTiles ? firstTile : numTiles - 1);
#endif
    f32x4 dyAhead[NT][MTL];
    auto loadAdjoints = [&](int tile) {
        const float* row[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
#if $$HAS_OUTPUT_ORDER$$
            const long long adjRow = adjRowAhead[nt];
#else
            const long long adjRow = min(tile * TILE_POINTS + 4 * r + nt, numel - 1);
#endif
            row[nt] = adjOutputs.data_ + adjRow * adjOutputs.strides_[0];
        }
        (void)tile;
        if (adjOutputRowsOfFloat4) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int m = 0; m < MTL; ++m) dyAhead[nt][m] = *reinterpret_cast<const f32x4*>(row[nt] + min(16 * m + 4 * g, actualChannelsOut - 4));
        } else if (MTL == 1 && adjOutputRowsOfFloat2) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const f32x2 two = *reinterpret_cast<const f32x2*>(row[nt]);
                dyAhead[nt][0] = __builtin_shufflevector(two, two, 0, 1, -1, -1);   // (nobody looks at the others)
            }
        } else {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int m = 0; m < MTL; ++m)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        dyAhead[nt][m][i] = row[nt][static_cast<long long>(min(16 * m + 4 * g + i, actualChannelsOut - 1)) * adjOutputs.strides_[1]];
        }
    };
    f16x4 encodedAhead[LOADS_AHEAD ? KT0 : 1][4];
    (void)encodedAhead;
    auto loadAhead = [&](int tile) {
        const int last = numTiles - 1;
        const int t0 = tile < last ? tile : last;   // (behind the last tile nobody looks at what is loaded)
        loadAdjoints(t0);
#if $$HAS_OUTPUT_ORDER$$
        loadRows(t0 + tileStep < last ? t0 + tileStep : last);
#endif
        const f16* encTile = forwardTmpMemory + static_cast<long long>(t0) * (CHANNELS_IN * TILE_POINTS);
#pragma unroll
        for (int t = 0; t < KT0; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                encodedAhead[LOADS_AHEAD ? t : 0][i] = *reinterpret_cast<const f16x4*>(encTile + (16 * t + 4 * g + i) * TILE_POINTS + 4 * r);
    };
    if constexpr (LOADS_AHEAD) loadAhead(firstTile);
    for (int tileBase = blockIdx.x * GROUP_TILES; tileBase < numTiles; tileBase += gridDim.x * GROUP_TILES)
    {
        const int tile = SHARED_TILE ? tileBase : tileBase + wave;
        if (!HAS_STREAMED_LAYERS && tile >= numTiles) continue;
        const bool tileValid = tile < numTiles;
        const int tileRead = tileValid ? tile : numTiles - 1;   // stored intermediates are read from a valid tile
        (void)tileRead;
        if (!SHARED_TILE || wave == 0) {
        // dL/dy -> accumulator layout (fp32 -> fp16), zero outside batch / real channels
        f16x4 dyOut[NT][MTL];
        int validMask = 0;
        if constexpr (LOADS_AHEAD) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const bool pv = tile * TILE_POINTS + 4 * r + nt < numel;
                validMask |= pv ? (1 << nt) : 0;
#pragma unroll
                for (int m = 0; m < MTL; ++m) {
                    dyOut[nt][m] = toF16(dyAhead[nt][m]);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (!pv || 16 * m + 4 * g + i >= actualChannelsOut) dyOut[nt][m][i] = static_cast<f16>(0);
                }
            }
        } else {
            // (a point after the other, behind its own branch: by way of the arrays of the loads ahead, which then lie in scratch memory, the kernel
            // of 30 000 points behind 32^4 nodes x 8 took 35 us, 30 so)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const int p = tile * TILE_POINTS + 4 * r + nt;
                const bool pv = p < numel;
                validMask |= pv ? (1 << nt) : 0;
#if $$HAS_OUTPUT_ORDER$$
                const long long adjRow = adjRowAhead[nt];
                {
                    const long long ahead = static_cast<long long>(p) + static_cast<long long>(tileStep) * TILE_POINTS;
                    adjRowAhead[nt] = (adjOutputOrder && ahead < numel) ? adjOutputOrder[ahead] : static_cast<int>(ahead < numel ? ahead : 0);
                }
#else
                const long long adjRow = p;
#endif
                const float* row = adjOutputs.data_ + adjRow * adjOutputs.strides_[0];
                if (adjOutputRowsOfFloat2 || adjOutputRowsOfFloat4) {
                    // channels side by side in memory: four per load (a lane holds channels
                    // 16m+4g .. +3 of its points), a row of two channels as one 8-byte load
#pragma unroll
                    for (int m = 0; m < MTL; ++m) {
                        dyOut[nt][m] = f16x4{0, 0, 0, 0};
                        const int c = 16 * m + 4 * g;
                        if (adjOutputRowsOfFloat4 && pv && c < actualChannelsOut) dyOut[nt][m] = toF16(*reinterpret_cast<const f32x4*>(row + c));
                    }
                    if (!adjOutputRowsOfFloat4 && pv && g == 0) {
                        const f32x2 two = *reinterpret_cast<const f32x2*>(row);
                        dyOut[nt][0][0] = static_cast<f16>(two[0]);
                        dyOut[nt][0][1] = static_cast<f16>(two[1]);
                    }
                } else {
#pragma unroll
                    for (int m = 0; m < MTL; ++m)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int c = 16 * m + 4 * g + i;
                            float v = 0.f;
                            if (pv && c < actualChannelsOut) v = row[static_cast<long long>(c) * adjOutputs.strides_[1]];
                            dyOut[nt][m][i] = static_cast<f16>(v);
                        }
                }
            }
        }

        // RECOMPUTE: the training pass kept the encoded input only; the layers run again, their pre-activations stay in registers
$$RECOMPUTE_FORWARD$$
        // layers, last to first
$$CALL_NETWORK_LAYERS$$

        if constexpr (STORE_ENCODED_ADJOINT) {
            if (tileValid) {
                f16* adjTile = adjointTmpMemory + (static_cast<long long>(OFFSET_ENCODED_ADJOINT) * numel64
                                                   + static_cast<long long>(tile) * (CHANNELS_IN * TILE_POINTS));
#pragma unroll
                for (int t = 0; t < KT0; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const f16x4 v = {dxIn[0][t][i], dxIn[1][t][i], dxIn[2][t][i], dxIn[3][t][i]};
                        *reinterpret_cast<f16x4*>(adjTile + (16 * t + 4 * g + i) * TILE_POINTS + 4 * r) = v;
                    }
            }
        }
        if constexpr (NEEDS_ENCODING_ADJOINT && NEEDS_STAGED_ADJOINT) {
            // adjoint of the encoded input: registers -> one staging row per point
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int t = 0; t < KT0; ++t)
                    *reinterpret_cast<f16x4*>(sStage + (16 * nt + r) * STAGE_STRIDE + 16 * t + 4 * g) = dxIn[nt][t];
        }
        }
        if constexpr (NEEDS_ENCODING_ADJOINT && NEEDS_STAGED_ADJOINT) {
            if constexpr (SHARED_TILE) {
                __syncthreads();
$$CALL_SHARED_ENCODINGS$$
                __syncthreads();   // (the next tile also waits: its rows are those of this one)
            } else {
                waveLdsSync();
            }

            const int index = tile * TILE_POINTS + lane;
            if (index < numel && (!SHARED_TILE || wave == 0)) {
                StaticArray<float, NUM_INPUTS> encodingInput;
#pragma unroll
                for (int i = 0; i < NUM_INPUTS; ++i)
                    encodingInput[i] = inputs.data_[static_cast<long long>(index) * inputs.strides_[0]
                                                    + static_cast<long long>(i) * inputs.strides_[1]];
                StaticArray<float, NUM_INPUTS> adjEncodingInput;
#pragma unroll
                for (int i = 0; i < NUM_INPUTS; ++i) adjEncodingInput[i] = 0.f;
                WrappedArray<const f16> adjEncodingOutput{sStage + stageRow(lane) * STAGE_STRIDE};

$$CALL_ENCODINGS$$

                if constexpr (HAS_INPUT_GRADIENTS) {
                    float* adjRow = adjInputs.data_ + static_cast<long long>(index) * adjInputs.strides_[0];
#if $$HAS_OUTPUT_ORDER$$
                    // (the rows of a sorted batch are the host's own, this kernel is the first to write them)
                    if (adjOutputOrder) {
                        if (NUM_INPUTS % 4 == 0 && adjInputs.strides_[1] == 1 && adjInputs.strides_[0] % 4 == 0
                            && reinterpret_cast<unsigned long long>(adjInputs.data_) % 16 == 0) {
#pragma unroll
                            for (int i = 0; i + 3 < NUM_INPUTS; i += 4)
                                *reinterpret_cast<float4*>(adjRow + i) = make_float4(adjEncodingInput[i], adjEncodingInput[i + 1],
                                                                                    adjEncodingInput[i + 2], adjEncodingInput[i + 3]);
                        } else {
#pragma unroll
                            for (int i = 0; i < NUM_INPUTS; ++i) adjRow[static_cast<long long>(i) * adjInputs.strides_[1]] = adjEncodingInput[i];
                        }
                    } else
#endif
                    if (!HAS_ENCODING_GRADIENTS && NUM_INPUTS % 4 == 0 && adjInputs.strides_[1] == 1 && adjInputs.strides_[0] % 4 == 0
                        && reinterpret_cast<unsigned long long>(adjInputs.data_) % 16 == 0) {
                        // the channels of a row side by side: four per load and store. Kept to
                        // kernels without a grid scatter: in front of the gradient atomics of a grid
                        // no gain was measurable.
                        // What a row holds is read before any of it is written, 16 channels at a time: all of a wide row took the registers of the
                        // layers (128 -> 64 -> 64 -> 64: 1320 bytes of scratch, forward and backward of 300 000 points 430 -> 500 us).
#pragma unroll
                        for (int first = 0; first < NUM_INPUTS; first += 16) {
                            float4 before[4];
#pragma unroll
                            for (int i = first; i < first + 16 && i + 3 < NUM_INPUTS; i += 4) before[(i - first) / 4] = *reinterpret_cast<const float4*>(adjRow + i);
#pragma unroll
                            for (int i = first; i < first + 16 && i + 3 < NUM_INPUTS; i += 4) {
                                const float4 v = before[(i - first) / 4];
                                *reinterpret_cast<float4*>(adjRow + i) = make_float4(v.x + adjEncodingInput[i], v.y + adjEncodingInput[i + 1],
                                                                                    v.z + adjEncodingInput[i + 2], v.w + adjEncodingInput[i + 3]);
                            }
                        }
                    } else {
#pragma unroll
                        for (int first = 0; first < NUM_INPUTS; first += 16) {
                            float before[16];
#pragma unroll
                            for (int i = first; i < first + 16 && i < NUM_INPUTS; ++i) before[i - first] = adjRow[static_cast<long long>(i) * adjInputs.strides_[1]];
#pragma unroll
                            for (int i = first; i < first + 16 && i < NUM_INPUTS; ++i)
                                adjRow[static_cast<long long>(i) * adjInputs.strides_[1]] = before[i - first] + adjEncodingInput[i];
                        }
                    }
                }
            }

            // parameter gradients of the grid encodings, scattered by the whole wavefront
            if (!SHARED_TILE || wave == 0) {
$$CALL_ENCODING_SCATTER$$
            }
            if constexpr (SHARED_TILE) __syncthreads();
            else waveLdsSync();
        }
    }
$$FLUSH_LDS_GRADIENTS$$
$$STORE_WEIGHT_GRADIENTS$$
}

QUICKMLP_KERNEL_NAMESPACE_END
