import ctypes

import torch

from . import _lib
from ._lib import check, current_stream, desc, lib


def _check_device(*tensors):
    for t in tensors:
        if not t.is_cuda:
            raise ValueError("pullpush works on GPU tensors only")


def _memory(data, which):
    """Device memory for the image pyramid (which = 0) or for its gradients (1) of images like data: from torch's
    allocator, so that it is reused in the order of the stream."""
    sizes = ctypes.c_size_t(), ctypes.c_size_t()
    check(lib.qmlp_utils_pullpush_memory(desc(data), ctypes.byref(sizes[0]), ctypes.byref(sizes[1])))
    return torch.empty((max(sizes[which].value, 16),), dtype=torch.uint8, device=data.device)


def _forward(mask, data):
    _check_device(mask, data)
    output = torch.empty_like(data)
    pyramid = _memory(data, 0)
    check(lib.qmlp_utils_pullpush_forward_in(desc(mask), desc(data), desc(output), pyramid.data_ptr(), current_stream(data.device)))
    return output, pyramid


def _backward(mask, data, adj_output, pyramid):
    _check_device(mask, data, adj_output)
    adj_mask = torch.empty_like(mask)
    adj_data = torch.empty_like(data)
    ready = pyramid is not None
    if not ready:
        pyramid = _memory(data, 0)
    gradients = _memory(data, 1)
    check(lib.qmlp_utils_pullpush_adjoint_in(desc(mask), desc(data), desc(adj_output), desc(adj_mask), desc(adj_data), 0,
                                             pyramid.data_ptr(), 1 if ready else 0, gradients.data_ptr(),
                                             current_stream(data.device)))
    return adj_mask, adj_data


def pullpush_forward(mask: torch.Tensor, data: torch.Tensor) -> torch.Tensor:
    """The inpainted data without autograd (``utils.pullpush_forward`` of the reference's
    torch bindings, src_cpp/pytorch-bindings/src/bind_utils.cpp:9-20)."""
    return _forward(mask, data)[0]


def pullpush_backward(mask: torch.Tensor, data: torch.Tensor, adj_output: torch.Tensor):
    """Gradients (adj_mask, adj_data) of the inpainting (``utils.pullpush_backward``,
    src_cpp/pytorch-bindings/src/bind_utils.cpp:22-40)."""
    return _backward(mask, data, adj_output, None)


def precompile(dtype: torch.dtype = torch.float32) -> None:
    """Compiles the pull-push kernels of one dtype into the kernel cache; needs no GPU."""
    check(lib.qmlp_utils_pullpush_precompile(_lib._PRECISION_OF[dtype]))


class _PullPushFunction(torch.autograd.Function):
    """src_cpp/pytorch-bindings/src/bind_utils.cpp:48-66; the image pyramid of the forward pass is kept for the
    backward pass (twice the planes of the low-res levels, about three quarters of the images' own memory)."""

    @staticmethod
    def forward(ctx, mask, data):
        output, pyramid = _forward(mask, data)
        ctx.save_for_backward(mask, data, pyramid)
        return output

    @staticmethod
    def backward(ctx, grad_output):
        mask, data, pyramid = ctx.saved_tensors
        return _backward(mask, data, grad_output, pyramid)


def pullpush(mask: torch.Tensor, data: torch.Tensor) -> torch.Tensor:
    """
    Performs differentiable inpainting via the Pull-Push algorithm.

    All tensors must reside on the GPU and are of type float or double.
    The mask is defined as 1: non-empty pixel, 0: empty pixel, and any fraction in between.

    :param mask: the mask of shape (Batch, Height, Width)
    :param data: the data of shape (Batch, Channels, Height, Width), fewer than 16 channels
    :return: the inpainted data of shape (Batch, Channels, Height, Width)

    Mirrors src_py/qmlp/pullpush.py:8-25 of the reference.
    """
    return _PullPushFunction.apply(mask, data)
