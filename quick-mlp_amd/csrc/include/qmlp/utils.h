#pragma once

#include "common.h"
#include "tensor.h"

QUICKMLP_NAMESPACE_BEGIN

/**
 * Helper operations that are not part of the network path.
 * Mirrors src_cpp/include/qmlp/utils.h:16-85 of the reference.
 */
class Utils
{
public:
    /**
     * Differentiable inpainting by pull-push: down- and upsampling over an image pyramid with
     * fractional masks (1: pixel is known, 0: pixel is empty, anything in between). All
     * tensors live on the GPU and are float or double.
     *
     * \param mask (Batch, Height, Width)
     * \param data (Batch, Channels, Height, Width), at most 15 channels like the reference
     * \param output the inpainted data, (Batch, Channels, Height, Width)
     */
    static void fractionalPullpush(const Tensor& mask, const Tensor& data, Tensor& output, stream_t stream);

    /** Bytes of device memory that the image pyramid of 'data' and its gradients take (both may be 0). */
    static void pullpushMemory(const Tensor& data, size_t& pyramidBytes, size_t& gradientBytes);

    /**
     * As above, with the image pyramid in memory of the caller (pullpushMemory(), aligned to 16 bytes), which an
     * adjoint call on the same mask and data may take over.
     */
    static void fractionalPullpush(const Tensor& mask, const Tensor& data, Tensor& output, void* pyramid, stream_t stream);

    /**
     * Adjoint of fractionalPullpush (runs the forward pass again to get the pyramid).
     * \param adjOutput gradient of the output, (Batch, Channels, Height, Width)
     * \param adjMask gradient of the mask, (Batch, Height, Width); accumulated, zero it first
     * \param adjData gradient of the data, (Batch, Channels, Height, Width); accumulated
     */
    static void adjointFractionalPullpush(const Tensor& mask, const Tensor& data, const Tensor& adjOutput,
                                          Tensor& adjMask, Tensor& adjData, stream_t stream);

    /**
     * As above, with memory of the caller (pullpushMemory(), aligned to 16 bytes).
     * \param accumulate add to adjMask and adjData; false: overwrite them
     * \param pyramidReady the pyramid is the one that the forward pass on this mask and data left; false: it is computed
     */
    static void adjointFractionalPullpush(const Tensor& mask, const Tensor& data, const Tensor& adjOutput, Tensor& adjMask,
                                          Tensor& adjData, bool accumulate, void* pyramid, bool pyramidReady, void* gradients,
                                          stream_t stream);

    /** Compiles the pull-push kernels of one precision into the kernel cache; needs no GPU. */
    static void precompile(Tensor::Precision precision);
};

QUICKMLP_NAMESPACE_END
