#pragma once
// One fully-connected layer of the adjoint kernel whose workgroup works on a tile of points together
// (network_backward_cooperative.h). Every wavefront runs the layers forward and backward for 32 points of its own,
// activations in registers in the layout of layer.h; the weight gradients, a contraction over the points, are formed
// by the whole workgroup: a wavefront writes the adjoint pre-activations and the input of a layer to LDS, a row of
// channels per point, and owns a block of the 16 x 16 tiles of dW for which it contracts the rows of all wavefronts.
// A wavefront then holds an eighth of the gradient tiles (64 -> 64 x 4 -> 4: 9 of 68, 36 registers), so that networks
// whose tiles exceed its registers need neither stored intermediates nor a weight-update kernel per layer.
//
// The contraction over points needs operands with 4 points of one channel per lane, the rows hold 4 channels of
// one point: ds_read_b64_tr_b16 transposes on the way from LDS (of 16 lanes, lane i supplies 4 halves of the 4 x 16
// block, row i / 4, and receives column i). The same instruction reads W^T from the one row-major copy of the
// weights, which serves both directions. Rows of W + 4 halves: measured with 8 wavefronts on a compute unit, a read of
// 16 rows x 4 pieces of 8 bytes then takes 4.6 cycles, transposed or not, and a write 6.2 (linear addresses: 3.7 - 4.3 and
// 6.2; rows of W + 8 halves: 3.6 - 4.6 and 8.1; rows without padding of 64 halves: 16, 8.2 and 64).

#include <qmlp/kernels/common.h>
#include <qmlp/kernels/layer.h>

QUICKMLP_KERNEL_NAMESPACE_BEGIN

constexpr int COOP_NT = 2;                    // column tiles of 16 points per wavefront: column r of tile nt is point 2r + nt
constexpr int COOP_POINTS = 16 * COOP_NT;     // points per wavefront
constexpr int COOP_PAD = 4;                   // halves behind every row in LDS

/** 4 halves of column (lane & 15) of the 4 x 16 block whose row (lane & 15) / 4, piece (lane & 3) this lane points at. */
__device__ __forceinline__ f16x4 readTransposed(const f16* p)
{
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    return __builtin_bit_cast(f16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p)));
}

/**
 * How the WAVES wavefronts of a workgroup share MT x KT gradient tiles: M x K blocks of tiles, and P shares of the points.
 * Few large blocks need fewer operand reads, many small ones fewer registers: the split of least
 *   matrix instructions + operand reads + REGISTER_WEIGHT / 8 x registers   (per tile of points and wavefront)
 * with the weight that the host found to leave the registers of the whole kernel within their budget
 * (FusedNetwork::cooperativeRegisters repeats this sum). Blocks may overlap the edge (3 tiles in blocks of 2):
 * those beyond it repeat the last tile and are not stored.
 */
template <int MT, int KT, int WAVES, int REGISTER_WEIGHT>
struct TileShare
{
    static constexpr int split(int which)
    {
        int bestM = 1, bestK = 1, best = 1 << 30;
        for (int m = 1; m <= WAVES; m *= 2)
            for (int k = 1; m * k <= WAVES; k *= 2) {
                const int mo = (MT + m - 1) / m, ki = (KT + k - 1) / k;
                const int cost = 8 * m * k * (mo * ki + mo + ki) + REGISTER_WEIGHT * 4 * mo * ki;
                if (cost < best) {
                    best = cost;
                    bestM = m;
                    bestK = k;
                }
            }
        return which == 0 ? bestM : bestK;
    }
    static constexpr int M = split(0), K = split(1), P = WAVES / (M * K);
    static constexpr int MO = (MT + M - 1) / M, KI = (KT + K - 1) / K;   // tiles of a wavefront
};

/**
 * The lane, as a value the compiler knows nothing about: what depends on it (the addresses of a layer in LDS) is computed where
 * it is used. Hoisted out of the loop over the tiles, the addresses of all layers take tens of registers. Passed as the lane
 * by the kernels of networks that need them otherwise.
 */
__device__ __forceinline__ int opaqueLane(int lane)
{
    asm volatile("" : "+v"(lane));
    return lane;
}

template <int CIN, int COUT, bool BIAS, typename Activation, int WAVES, int REGISTER_WEIGHT>
struct CooperativeLayer
{
    static constexpr int KT = CIN / 16, MT = COUT / 16;
    static constexpr int F_KB = (KT + 1) / 2, A_KB = (MT + 1) / 2;   // blocks of 32 contracted channels, forward and adjoint
    static constexpr int W_STRIDE = CIN + COOP_PAD;                 // of the weights in LDS, halves per output channel
    static constexpr int D_STRIDE = COUT + COOP_PAD, X_STRIDE = CIN + COOP_PAD;   // of the rows of a point: adjoint pre-activations and input
    static constexpr int X_OFFSET = COOP_POINTS * D_STRIDE;         // the input rows lie behind the others
    typedef TileShare<MT, KT, WAVES, REGISTER_WEIGHT> Share;
    static constexpr int MO = Share::MO, KI = Share::KI;

    typedef f16x4 input_t[COOP_NT][KT];
    typedef f16x4 output_t[COOP_NT][MT];

    /** Weights into LDS, row-major with padded rows. */
    __device__ static void stageWeights(const f16* __restrict__ W, f16* __restrict__ dst, int tid, int nthreads)
    {
        for (int v = tid; v < COUT * CIN / 8; v += nthreads) {
            const int o = (v * 8) / CIN, k = (v * 8) % CIN;
            const f16x8 w = *reinterpret_cast<const f16x8*>(W + v * 8);
            *reinterpret_cast<f16x4*>(dst + o * W_STRIDE + k) = f16x4{w[0], w[1], w[2], w[3]};
            *reinterpret_cast<f16x4*>(dst + o * W_STRIDE + k + 4) = f16x4{w[4], w[5], w[6], w[7]};
        }
    }

    /** The layer forward: pre-activations only (the same operations as Layer::forward: the same bits). */
    __device__ __forceinline__ static void forward(const f16* __restrict__ w, const f16* __restrict__ bias, const input_t& x, output_t& pre, int lane)
    {
        const int g = lane >> 4, r = lane & 15;
        const f16x4 zero4 = {0, 0, 0, 0};
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            f32x4 acc[COOP_NT];
            f32x4 start = {0.f, 0.f, 0.f, 0.f};
            if constexpr (BIAS) start = __builtin_convertvector(*reinterpret_cast<const f16x4*>(bias + 16 * m + 4 * g), f32x4);
#pragma unroll
            for (int nt = 0; nt < COOP_NT; ++nt) acc[nt] = start;
            const f16* row = w + (16 * m + r) * W_STRIDE + 4 * g;
#pragma unroll
            for (int kb = 0; kb < F_KB; ++kb) {
                const f16x4 lo = *reinterpret_cast<const f16x4*>(row + 32 * kb);
                const f16x4 hi = 2 * kb + 1 < KT ? *reinterpret_cast<const f16x4*>(row + 32 * kb + 16) : zero4;
                const f16x8 a = concat(lo, hi);
#pragma unroll
                for (int nt = 0; nt < COOP_NT; ++nt)
                    acc[nt] = mfma32(a, concat(x[nt][2 * kb], 2 * kb + 1 < KT ? x[nt][2 * kb + 1 < KT ? 2 * kb + 1 : 0] : zero4), acc[nt]);
            }
#pragma unroll
            for (int nt = 0; nt < COOP_NT; ++nt) pre[nt][m] = toF16(acc[nt]);
        }
    }

    // The activation's adjoint follows from its output: kept (output_t pre) is the output then, else the pre-activation.
    static constexpr bool KEEPS_OUTPUT = HasAdjointOfOutput<Activation>::value;

    /** The activation of the layer: y, and in pre what the adjoint needs. */
    __device__ __forceinline__ static void activate(output_t& pre, output_t& y, int lane)
    {
        const int g = lane >> 4;
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int nt = 0; nt < COOP_NT; ++nt) {
                y[nt][m] = activationForwardChannels<Activation>(pre[nt][m], 16 * m + 4 * g);
                if constexpr (KEEPS_OUTPUT) pre[nt][m] = y[nt][m];
            }
    }

    /** dy: from the adjoint of the output to that of the pre-activation, into the rows of this wavefront. valid: all bits set for
     *  a point of the batch; zero: no gradient (whatever the activation makes of a zero adjoint). kept: pre after activate. */
    __device__ __forceinline__ static void adjointActivation(const output_t& kept, output_t& dy, f16* rows, const unsigned (&valid)[COOP_NT], int lane)
    {
        const int g = lane >> 4, r = lane & 15;
#pragma unroll
        for (int nt = 0; nt < COOP_NT; ++nt)
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const u32x2 mask = {valid[nt], valid[nt]};
                if constexpr (KEEPS_OUTPUT) dy[nt][m] = Activation::adjointOfOutput4(kept[nt][m], dy[nt][m], mask);
                else dy[nt][m] = activationAdjointMasked<Activation>(kept[nt][m], dy[nt][m], 16 * m + 4 * g, mask);
                *reinterpret_cast<f16x4*>(rows + (16 * nt + r) * D_STRIDE + 16 * m + 4 * g) = dy[nt][m];
            }
    }

    /** The input of the layer, from what the layer of InputActivation in front kept, into the rows of this wavefront. */
    template <typename InputActivation>
    __device__ __forceinline__ static void stageInput(const input_t& kept, f16* rows, int lane)
    {
        const int g = lane >> 4, r = lane & 15;
#pragma unroll
        for (int t = 0; t < KT; ++t) {
#pragma unroll
            for (int nt = 0; nt < COOP_NT; ++nt) {
                f16x4 x = kept[nt][t];
                if constexpr (!HasAdjointOfOutput<InputActivation>::value) x = activationForwardChannels<InputActivation>(x, 16 * t + 4 * g);
                *reinterpret_cast<f16x4*>(rows + X_OFFSET + (16 * nt + r) * X_STRIDE + 16 * t + 4 * g) = x;
            }
        }
    }

    /** dx = W^T dy (the same operations as Layer::adjoint). */
    __device__ __forceinline__ static void adjointInput(const f16* __restrict__ w, const output_t& dy, input_t& dx, int lane)
    {
        const int g = lane >> 4, i = lane & 15;
        const f16x4 zero4 = {0, 0, 0, 0};
        const f16* at = w + (4 * g + (i >> 2)) * W_STRIDE + 4 * (i & 3);
#pragma unroll
        for (int mi = 0; mi < KT; ++mi) {
            f32x4 acc[COOP_NT];
#pragma unroll
            for (int nt = 0; nt < COOP_NT; ++nt) acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kb = 0; kb < A_KB; ++kb) {
                const f16x4 lo = readTransposed(at + 32 * kb * W_STRIDE + 16 * mi);
                const f16x4 hi = 2 * kb + 1 < MT ? readTransposed(at + (32 * kb + 16) * W_STRIDE + 16 * mi) : zero4;
                const f16x8 a = concat(lo, hi);
#pragma unroll
                for (int nt = 0; nt < COOP_NT; ++nt)
                    acc[nt] = mfma32(a, concat(dy[nt][2 * kb], 2 * kb + 1 < MT ? dy[nt][2 * kb + 1 < MT ? 2 * kb + 1 : 0] : zero4), acc[nt]);
            }
#pragma unroll
            for (int nt = 0; nt < COOP_NT; ++nt) dx[nt][mi] = toF16(acc[nt]);
        }
    }

    /** Gradient tiles of this wavefront; column m of the bias tile holds the sums of its m-th tile of output channels. (A tile that
     *  several layers share saves registers, but its other columns are multiplied by zero: an infinite adjoint in one layer
     *  makes sums of the others NaN.) */
    struct Sums
    {
        f32x4 w[MO][KI];
        f32x4 b;
        __device__ __forceinline__ void zero()
        {
            zeroTiles(w);
            b = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    };

    /**
     * Adds the points of all wavefronts to the tiles of this one. rows: the rows of wavefront 0, those of wavefront i
     * start i * rowsPerWave halves further.
     */
    __device__ __forceinline__ static void weightGradient(const f16* rows, int rowsPerWave, Sums& sums, int wave, int lane)
    {
        const int g = lane >> 4, i = lane & 15;
        const int wm = wave % Share::M, wk = (wave / Share::M) % Share::K, wp = wave / (Share::M * Share::K);
        const f16* d = rows + (4 * g + (i >> 2)) * D_STRIDE + 4 * (i & 3);
        const f16* x = rows + X_OFFSET + (4 * g + (i >> 2)) * X_STRIDE + 4 * (i & 3);
        // channels of the m-th / k-th tile of this wavefront
        auto dChannels = [&](int m) { return 16 * (MT % Share::M == 0 ? wm * MO + m : min(wm * MO + m, MT - 1)); };
        auto xChannels = [&](int k) { return 16 * (KT % Share::K == 0 ? wk * KI + k : min(wk * KI + k, KT - 1)); };
        const f16x8 ones = {1, 1, 1, 1, 1, 1, 1, 1};
        const f16x8 zeros = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll 2
        for (int p = 0; p < WAVES / Share::P; ++p) {
            const int offset = (p * Share::P + wp) * rowsPerWave;
            f16x8 b[KI];
#pragma unroll
            for (int k = 0; k < KI; ++k)
                b[k] = concat(readTransposed(x + offset + xChannels(k)), readTransposed(x + offset + 16 * X_STRIDE + xChannels(k)));
#pragma unroll
            for (int m = 0; m < MO; ++m) {
                const f16x8 a = concat(readTransposed(d + offset + dChannels(m)), readTransposed(d + offset + 16 * D_STRIDE + dChannels(m)));
#pragma unroll
                for (int k = 0; k < KI; ++k) sums.w[m][k] = mfma32(a, b[k], sums.w[m][k]);
                if constexpr (BIAS) {
                    if (p % Share::K == wk) {   // (one of the wavefronts that read these rows)
                        sums.b = mfma32(a, MO == 1 || i == m ? ones : zeros, sums.b);
                    }
                }
            }
        }
    }

    /**
     * After the last tile: the workgroup's sums into slice blockIdx.x of the partial gradients, slices beyond the grid
     * zeroed (as Layer::storeWeightGradient). sAcc: (MT * KT * 256 + WAVES * COUT) floats. All threads call this.
     */
    __device__ __forceinline__ static void storeWeightGradient(const Sums& sums, float* sAcc, float* __restrict__ partialWeights,
                                                               float* __restrict__ partialBias, int numSlices, int sliceStride, int wave, int lane)
    {
        const int g = lane >> 4, r = lane & 15;
        const int wm = wave % Share::M, wk = (wave / Share::M) % Share::K, wp = wave / (Share::M * Share::K);
        float* sBias = sAcc + MT * KT * 256;
        for (int p = 0; p < Share::P; ++p) {
            __syncthreads();   // whatever used this LDS before is done
            if (wp != p) continue;
#pragma unroll
            for (int m = 0; m < MO; ++m)
#pragma unroll
                for (int k = 0; k < KI; ++k) {
                    if (wm * MO + m >= MT || wk * KI + k >= KT) continue;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        float* target = sAcc + (16 * (wm * MO + m) + 4 * g + i) * CIN + 16 * (wk * KI + k) + r;
                        *target = p == 0 ? sums.w[m][k][i] : *target + sums.w[m][k][i];
                    }
                }
        }
        if constexpr (BIAS) {
            if (r < MO && wm * MO + r < MT) {
#pragma unroll
                for (int i = 0; i < 4; ++i) sBias[(wp * Share::K + wk) * COUT + 16 * (wm * MO + r) + 4 * g + i] = sums.b[i];
            }
        }
        __syncthreads();
        for (int e = threadIdx.x; e < COUT * CIN; e += blockDim.x) partialWeights[e] = sAcc[e];
        if constexpr (BIAS) {
            for (int e = threadIdx.x; e < COUT; e += blockDim.x) {
                float sum = sBias[e];
#pragma unroll
                for (int s = 1; s < Share::P * Share::K; ++s) sum += sBias[s * COUT + e];
                partialBias[e] = sum;
            }
        }
        for (int slice = blockIdx.x + gridDim.x; slice < numSlices; slice += gridDim.x) {
            const long long offset = static_cast<long long>(slice - static_cast<int>(blockIdx.x)) * sliceStride;
            for (int e = threadIdx.x; e < COUT * CIN; e += blockDim.x) partialWeights[offset + e] = 0.f;
            if constexpr (BIAS) {
                for (int e = threadIdx.x; e < COUT; e += blockDim.x) partialBias[offset + e] = 0.f;
            }
        }
    }
};

QUICKMLP_KERNEL_NAMESPACE_END
