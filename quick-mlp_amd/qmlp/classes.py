"""Python counterparts of the custom classes the reference registers as
``torch.classes.qmlp_cu.{QuickMLP, Network, Encoding, Activation}``
(src_cpp/pytorch-bindings/src/bindings.cpp:102-122, bind_network.cpp:346-411,
bind_encoding.cpp:165-197, bind_activation.cpp:80-98), same method names and
argument meaning, implemented on the C ABI of libqmlp.so. torch only provides
device memory, the current stream and autograd bookkeeping here.
"""
import ctypes
import json

import torch

from . import _lib
from . import _native   # the per-batch calls in C++; like libqmlp.so there is no fallback
from ._lib import (GRADIENTS_INPUT, GRADIENTS_INPUT_ENCODINGS, GRADIENTS_NETWORK_WEIGHTS,
                   QMLP_GRADIENTS, QMLP_INFERENCE, check, current_stream, desc, lib)


def _device_of(t):
    if not t.is_cuda:
        raise RuntimeError("QuickMLP tensors must live on the GPU")
    return t.device


def _create_output(input, channels):
    if input.dim() != 2:
        raise RuntimeError("input must be a tensor with 2 dimensions (batch, channels)")
    return torch.empty((input.shape[0], channels), dtype=input.dtype, device=input.device)


class QuickMLP:
    """Global settings (bindings.cpp:104-113)."""

    @staticmethod
    def set_compile_debug_mode(enable):
        check(lib.qmlp_set_compile_debug_mode(1 if enable else 0))

    @staticmethod
    def is_compile_debug_mode():
        return bool(_lib.get_int(lib.qmlp_is_compile_debug_mode))

    @staticmethod
    def set_log_level(level):
        _lib.set_log_level(level)

    @staticmethod
    def is_cuda_available():
        return bool(_lib.get_int(lib.qmlp_is_gpu_available))

    is_gpu_available = is_cuda_available


# ---------------------------------------------------------------------------- activation
class _ActivationFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, input, activ):
        ctx.save_for_backward(input)
        ctx.activ = activ
        return activ.inference(input)

    @staticmethod
    def backward(ctx, grad_output):
        (input,) = ctx.saved_tensors
        return ctx.activ.adjoint(input, grad_output.contiguous()), None


class Activation:
    """A built-in activation id or an inline JSON specification; half tensors only."""

    def __init__(self, cfg):
        self._cfg = cfg
        self._handle = ctypes.c_void_p()
        check(lib.qmlp_activation_create(cfg.encode(), ctypes.byref(self._handle)))

    def __del__(self):
        if getattr(self, "_handle", None):
            lib.qmlp_activation_destroy(self._handle)
            self._handle = None

    def cfg(self):
        return self._cfg

    def to_json(self):
        return _lib.get_string(lib.qmlp_activation_to_json, self._handle)

    def precompile(self):
        """Compiles the standalone kernels into the kernel cache; needs no GPU."""
        check(lib.qmlp_activation_precompile(self._handle))

    def inference(self, input):
        _device_of(input)
        output = torch.empty_like(input)
        check(lib.qmlp_activation_forward(self._handle, desc(input), desc(output), current_stream(input.device)))
        return output

    def adjoint(self, input, adj_output):
        adj_input = torch.empty_like(input)
        check(lib.qmlp_activation_adjoint(self._handle, desc(input), desc(adj_output), desc(adj_input),
                                          current_stream(input.device)))
        return adj_input

    def forward(self, input):
        return _ActivationFunction.apply(input, self)

    def __getstate__(self):
        return self._cfg

    def __setstate__(self, state):
        self.__init__(state)


# ---------------------------------------------------------------------------- encoding
class _RecordedEncoding(torch.autograd.Function):
    """A call of an encoding while torch.jit.trace records: what it records, and plays later, is a call of this function.
    Everywhere else the autograd node in C++ does the same with less work on the host."""

    @staticmethod
    def forward(ctx, native, input, parameter):
        ctx.native = native
        ctx.flags = (1 if ctx.needs_input_grad[1] else 0) | (2 if ctx.needs_input_grad[2] else 0)
        ctx.save_for_backward(input, parameter)
        return native.inference(input, parameter)

    @staticmethod
    def backward(ctx, grad_output):
        input, parameter = ctx.saved_tensors
        if ctx.flags == 0:
            return None, None, None
        adj_input, adj_parameter = ctx.native.adjoint_pass(input, parameter, grad_output.contiguous(), ctx.flags)
        return None, adj_input, None if adj_parameter is None else adj_parameter.to(parameter.dtype)


class Encoding:
    """One input encoding, standalone (fp32 in, fp32 out)."""

    def __init__(self, cfg=None, _borrowed=None, _owner=None):
        self._owner = _owner          # keeps the network alive for borrowed handles
        self._borrowed = _borrowed is not None
        if _borrowed is not None:
            self._handle = _borrowed
            self._cfg = self.to_json()
        else:
            self._cfg = cfg
            self._handle = ctypes.c_void_p()
            check(lib.qmlp_encoding_create(cfg.encode(), ctypes.byref(self._handle)))
        # owns the handle, unless a network does, together with the autograd graphs of its calls
        self._native = _native.Encoding(self._handle.value, _owner._native if self._borrowed else None)

    def cfg(self):
        return self._cfg

    def to_json(self):
        return _lib.get_string(lib.qmlp_encoding_to_json, self._handle)

    def id(self):
        return _lib.get_string(lib.qmlp_encoding_id, self._handle)

    def max_input_channel(self):
        return _lib.get_int(lib.qmlp_encoding_max_input_channel, self._handle)

    def num_output_channels(self):
        return _lib.get_int(lib.qmlp_encoding_num_output_channels, self._handle)

    def has_parameters(self):
        # fixed by the specification: asked once (this sits on the per-call path of the network)
        if getattr(self, "_has_parameters", None) is None:
            self._has_parameters = bool(_lib.get_int(lib.qmlp_encoding_has_parameters, self._handle))
        return self._has_parameters

    def num_parameters(self):
        return _lib.get_int(lib.qmlp_encoding_parameter_count, self._handle)

    def parameter_dtype(self, gradients=False):
        p = _lib.get_int(lib.qmlp_encoding_parameter_precision, self._handle,
                         QMLP_GRADIENTS if gradients else QMLP_INFERENCE)
        return _lib.DTYPE_OF[p]

    def create_inference_parameters(self, device="cuda"):
        if not self.has_parameters():
            raise RuntimeError("the encoding has no parameters")
        return torch.empty((self.num_parameters(),), dtype=self.parameter_dtype(False), device=device)

    def create_gradient_parameters(self, device="cuda"):
        if not self.has_parameters():
            raise RuntimeError("the encoding has no parameters")
        return torch.empty((self.num_parameters(),), dtype=self.parameter_dtype(True), device=device)

    def set_parameter(self, tensor, gradients=False):
        if not gradients:
            # binding the same memory again changes nothing: skipped, unless the encoding belongs to a network,
            # whose own calls bind it as well
            # (a native call on a table of its own leaves the encoding without one)
            key = None if tensor is None else (tensor.data_ptr(), tensor.numel(), tensor.dtype, self._native.calls)
            if key is not None and not self._borrowed and key == getattr(self, "_bound_inference", None):
                return
            self._bound_inference = key
        check(lib.qmlp_encoding_set_parameter(self._handle, desc(tensor),
                                              QMLP_GRADIENTS if gradients else QMLP_INFERENCE))

    def precompile(self, adjoint_mode=3):
        """Compiles the standalone kernels into the kernel cache (needs no GPU)."""
        with self._native:
            check(lib.qmlp_encoding_precompile(self._handle, int(adjoint_mode)))

    def hashgrid_levels(self):
        """[(resolution, hashed, memory_offset, hash_grid_size)] of a HashGrid encoding."""
        n = ctypes.c_int()
        cap = 64
        arrs = [(ctypes.c_int * cap)() for _ in range(4)]
        check(lib.qmlp_encoding_hashgrid_levels(self._handle, cap, ctypes.byref(n), *arrs))
        off, res, hs, hashed = arrs
        return [(res[l], bool(hashed[l]), off[l], hs[l]) for l in range(n.value)]

    def hashgrid_corners(self, input, mode=0):
        """Device-computed table offsets and weights, shape (N, levels, 2^dim). mode 0: the index
        function; 1: what the gathers of the fused forward kernels use (bind a table first);
        2: what the gradient scatter of the fused backward kernel adds to; 3: what the gradient
        records of large batches (sums per slice of the table) stand for; 4: the elements behind the
        sums of the column kernel (single dense levels whose batches train sorted by slab)."""
        if input is None:      # compile the kernel of this mode into the kernel cache, nothing runs
            with self._native:
                check(lib.qmlp_encoding_hashgrid_trace(self._handle, None, int(mode), None, None, None))
            return None
        levels = self.hashgrid_levels()
        dim = int(json.loads(self.to_json())["n_in"])
        n = input.shape[0]
        idx = torch.full((n, len(levels), 1 << dim), -1, dtype=torch.int32, device=input.device)
        w = torch.full((n, len(levels), 1 << dim), float("nan"), dtype=torch.float32, device=input.device)
        with self._native:
            check(lib.qmlp_encoding_hashgrid_trace(self._handle, desc(input), int(mode), idx.data_ptr(), w.data_ptr(),
                                                   current_stream(input.device)))
        return idx, w

    def inference(self, input):
        if self.has_parameters():
            raise RuntimeError("Encoding has parameters, call the variation of 'inference' with parameters")
        return self._native.inference(input, None)

    def inference_with_parameter(self, input, parameter_forward):
        if not self.has_parameters():
            raise RuntimeError("Encoding doesn't have parameters, call the variation of 'inference' without parameters")
        # the native call binds the table for its own duration and leaves the encoding unbound
        self._bound_inference = None
        return self._native.inference(input, parameter_forward)

    def adjoint(self, input, adj_output):
        if self.has_parameters():
            raise RuntimeError("Encoding has parameters, call the variation of 'adjoint' with parameters")
        adj_input = torch.zeros_like(input)
        with self._native:
            check(lib.qmlp_encoding_adjoint(self._handle, desc(input), desc(adj_output), desc(adj_input),
                                            current_stream(input.device), None, None, 3))
        return adj_input

    def adjoint_with_parameter(self, input, parameter_forward, adj_output):
        return self.adjoint_with_parameter_and_flags(input, parameter_forward, adj_output, 3)

    def adjoint_with_parameter_and_flags(self, input, parameter_forward, adj_output, flags):
        if not self.has_parameters():
            raise RuntimeError("Encoding doesn't have parameters, call the variation of 'adjoint' without parameters")
        adj_input = torch.zeros_like(input)
        adj_param = torch.zeros(parameter_forward.shape, dtype=self.parameter_dtype(True),
                                device=parameter_forward.device)
        size = ctypes.c_size_t()
        check(lib.qmlp_encoding_adjoint_memory(self._handle, input.shape[0], int(flags), ctypes.byref(size)))
        memory = torch.empty((size.value,), dtype=torch.uint8, device=input.device) if size.value else None
        with self._native:
            check(lib.qmlp_encoding_adjoint_in(self._handle, desc(input), desc(adj_output), desc(adj_input),
                                               current_stream(input.device), desc(parameter_forward), desc(adj_param),
                                               int(flags), memory.data_ptr() if size.value else None))
        self._bound_inference = None   # as in inference_with_parameter
        return adj_input, adj_param.to(parameter_forward.dtype)

    def forward(self, input):
        if self.has_parameters():
            raise RuntimeError("Encoding has parameters, call the variation of 'forward' with parameters")
        return self._native.forward(input, None)

    def forward_with_parameter(self, input, parameter):
        if not self.has_parameters():
            raise RuntimeError("Encoding doesn't have parameters, call the variation of 'forward' without parameters")
        if parameter is None:
            raise RuntimeError("Encoding has parameters, but none are given")
        return self._native.forward(input, parameter)

    def __getstate__(self):
        return self._cfg

    def __setstate__(self, state):
        self.__init__(state)


# ---------------------------------------------------------------------------- network
class _RecordedNetwork(torch.autograd.Function):
    """As _RecordedEncoding, for networks; tables: None for encodings without parameters."""

    @staticmethod
    def forward(ctx, native, input, network_parameters, *tables):
        needs = ctx.needs_input_grad[1:]
        flags = ((GRADIENTS_INPUT if needs[0] else 0) | (GRADIENTS_NETWORK_WEIGHTS if needs[1] else 0)
                 | (GRADIENTS_INPUT_ENCODINGS if any(needs[2:]) else 0))
        if flags == 0:
            return native.inference(input, network_parameters, list(tables))
        half = network_parameters.to(torch.float16)
        output, memory, contents = native.forward_pass(input, half, list(tables), flags)
        ctx.native, ctx.flags, ctx.contents, ctx.dtype = native, flags, contents, network_parameters.dtype
        ctx.save_for_backward(input, half, memory, *tables)
        return output

    @staticmethod
    def backward(ctx, grad_output):
        input, half, memory, *tables = ctx.saved_tensors
        adj_input, adj_network, adj_tables = ctx.native.adjoint_pass(input, half, tables, memory, ctx.contents,
                                                                     grad_output.contiguous(), ctx.flags)
        adj_tables = [g.to(t.dtype) if g is not None and ctx.needs_input_grad[3 + i] else None
                      for i, (g, t) in enumerate(zip(adj_tables, tables))]
        return (None, adj_input, None if adj_network is None else adj_network.to(ctx.dtype), *adj_tables)


class Network:
    """The fused network of a JSON configuration (bind_network.h:16-95)."""

    def __init__(self, cfg, parent="."):
        self._cfg = cfg
        self._parent = parent
        self._handle = ctypes.c_void_p()
        check(lib.qmlp_network_create(cfg.encode(), parent.encode(), ctypes.byref(self._handle)))
        self._native = _native.Network(self._handle.value)   # owns the handle, together with the autograd graphs of its calls
        self._mutex = self._native    # (one call of the native network at a time)
        self._encodings = {}

    def cfg(self):
        return self._cfg

    def parent(self):
        return self._parent

    @staticmethod
    def MatrixSize():
        return _lib.get_int(lib.qmlp_network_matrix_size)

    @staticmethod
    def WarpSize():
        return _lib.get_int(lib.qmlp_network_warp_size)

    @staticmethod
    def MaxSharedMemoryBytes():
        return _lib.get_int(lib.qmlp_network_max_shared_memory_bytes)

    def is_parallel_streams(self):
        return bool(_lib.get_int(lib.qmlp_network_is_parallel_streams, self._handle))

    def set_parallel_streams(self, enabled):
        with self._mutex:
            check(lib.qmlp_network_set_parallel_streams(self._handle, 1 if enabled else 0))

    def num_encodings(self):
        if getattr(self, "_num_encodings", None) is None:
            self._num_encodings = _lib.get_int(lib.qmlp_network_num_encodings, self._handle)
        return self._num_encodings

    def encoding(self, idx):
        if idx not in self._encodings:
            h = ctypes.c_void_p()
            check(lib.qmlp_network_encoding(self._handle, idx, ctypes.byref(h)))
            self._encodings[idx] = Encoding(_borrowed=h, _owner=self)
        return self._encodings[idx]

    def channels_in(self):
        return _lib.get_int(lib.qmlp_network_channels_in, self._handle)

    def channels_out(self):
        if getattr(self, "_channels_out", None) is None:
            self._channels_out = _lib.get_int(lib.qmlp_network_channels_out, self._handle)
        return self._channels_out

    def num_layers(self):
        return _lib.get_int(lib.qmlp_network_num_layers, self._handle)

    def num_network_parameters(self):
        return _lib.get_int(lib.qmlp_network_parameter_count, self._handle)

    def create_inference_parameters(self, device="cuda"):
        """Uninitialized fp16 tensor of shape (num_network_parameters(),)."""
        return torch.empty((self.num_network_parameters(),), dtype=torch.float16, device=device)

    def initialize_inference_parameters(self, dst):
        """Default (torch.nn.Linear style) initialization of the fp16 tensor 'dst'."""
        with self._mutex:
            check(lib.qmlp_network_set_parameter(self._handle, desc(dst), QMLP_INFERENCE))
            seed = int(torch.randint(2 ** 31 - 1, (1,)).item())
            check(lib.qmlp_network_initialize_inference_parameters(self._handle, seed))

    def parameter_view(self, layer, bias, parameters):
        """Read-write view of the weight matrix / bias vector of 'layer' inside 'parameters'."""
        if parameters.dtype not in (torch.float32, torch.float16):
            raise RuntimeError("parameters must be float or half")
        if parameters.dim() != 1 or parameters.shape[0] != self.num_network_parameters():
            raise RuntimeError("The tensor must be of shape (num_parameters, )")
        view = _lib.TensorDesc()
        prec = _lib.QMLP_FLOAT if parameters.dtype == torch.float32 else _lib.QMLP_HALF
        check(lib.qmlp_network_parameter_view(self._handle, int(layer), 1 if bias else 0,
                                              ctypes.c_void_p(parameters.data_ptr()), prec, ctypes.byref(view)))
        if view.ndim == 0:
            return None
        offset = (view.data - parameters.data_ptr()) // parameters.element_size()
        sizes = [view.sizes[i] for i in range(view.ndim)]
        strides = [view.strides[i] for i in range(view.ndim)]
        return torch.as_strided(parameters, sizes, strides, parameters.storage_offset() + offset)

    def forward_memory(self, num_elements, flags):
        n = ctypes.c_size_t()
        check(lib.qmlp_network_forward_memory(self._handle, int(num_elements), int(flags), ctypes.byref(n)))
        return n.value

    def adjoint_memory(self, num_elements, flags):
        n = ctypes.c_size_t()
        check(lib.qmlp_network_adjoint_memory(self._handle, int(num_elements), int(flags), ctypes.byref(n)))
        return n.value

    def precompile(self, adjoint_flags=7):
        with self._mutex:
            check(lib.qmlp_network_precompile(self._handle, int(adjoint_flags)))

    def prepare(self, num_elements, adjoint_flags=0):
        """Loads the kernels and allocates the workspace that calls on a batch of this size need,
        so that those calls only enqueue kernels (e.g. under graph capture)."""
        with self._mutex:
            check(lib.qmlp_network_prepare(self._handle, int(num_elements), int(adjoint_flags)))

    def generated_source(self, kind, adjoint_flags=0):
        with self._mutex:
            return _lib.get_string(lib.qmlp_network_generated_source, self._handle, kind.encode(), int(adjoint_flags))

    def _set_network_parameters(self, network_parameters, encoding_parameters):
        self._native.bind(network_parameters, list(encoding_parameters))

    def inference(self, input, network_parameters, encoding_parameters=()):
        return self._native.inference(input, network_parameters, list(encoding_parameters))

    def inference_noalloc(self, input, output, network_parameters, encoding_parameters=()):
        """inference() into a tensor of the caller through the entry point of the C ABI that
        allocates no device memory (for code under HIP graph capture and the like): the kernels must
        have been loaded by an inference() call on a batch of the same size, the parameters are
        fp16 already, and a batch that is ordered by grid slab has to fit the library's static
        48 MiB workspace. Calls that overlap on one GPU race on that workspace."""
        _device_of(input)
        if network_parameters.dtype != torch.float16:
            raise RuntimeError("inference_noalloc takes fp16 network parameters (a conversion would allocate)")
        with self._mutex:
            self._set_network_parameters(network_parameters, list(encoding_parameters))
            check(lib.qmlp_network_inference_noalloc(self._handle, desc(input), desc(output), current_stream(input.device)))
        return output

    def forward_raw(self, input, network_parameters, encoding_parameters=(), flags=7, contents=False):
        """forward() of the C ABI without autograd: returns (output, tmp_forward). With contents=True the pass leaves no
        more in tmp_forward than an adjoint pass with these flags reads, and what it left is the third value returned:
        the 'contents' of adjoint_raw."""
        _device_of(input)
        output = _create_output(input, self.channels_out())
        nbytes = self.forward_memory(input.shape[0], flags)
        tmp_forward = torch.empty((max(nbytes, 16),), dtype=torch.uint8, device=input.device)
        left = ctypes.c_int()
        with self._mutex:
            self._set_network_parameters(network_parameters, list(encoding_parameters))
            if contents:
                check(lib.qmlp_network_forward_for(self._handle, desc(input), desc(output), int(flags),
                                                   ctypes.c_void_p(tmp_forward.data_ptr()), ctypes.byref(left),
                                                   current_stream(input.device)))
            else:
                check(lib.qmlp_network_forward(self._handle, desc(input), desc(output),
                                               ctypes.c_void_p(tmp_forward.data_ptr()), current_stream(input.device)))
        return (output, tmp_forward, left.value) if contents else (output, tmp_forward)

    def adjoint_raw(self, input, adj_output, flags, tmp_forward, network_parameters, encoding_parameters=(),
                    grad_network=None, grad_encodings=None, adj_input=None, contents=None):
        """adjoint() of the C ABI without autograd. Gradient tensors that are passed in are
        accumulated into (+=); missing ones are created zero-filled. contents: what forward_raw
        reported of tmp_forward, if it was asked to.
        Returns (adj_input, grad_network, grad_encodings)."""
        encoding_parameters = list(encoding_parameters)
        if flags & GRADIENTS_INPUT and adj_input is None:
            adj_input = torch.zeros_like(input)
        if flags & GRADIENTS_NETWORK_WEIGHTS and grad_network is None:
            grad_network = torch.zeros((self.num_network_parameters(),), dtype=torch.float32, device=input.device)
        if grad_encodings is None:
            grad_encodings = [None] * self.num_encodings()
        grad_encodings = list(grad_encodings)
        if flags & GRADIENTS_INPUT_ENCODINGS:
            for i in range(self.num_encodings()):
                enc = self.encoding(i)
                if enc.has_parameters() and grad_encodings[i] is None:
                    grad_encodings[i] = torch.zeros((enc.num_parameters(),), dtype=torch.float32, device=input.device)
        nbytes = self.adjoint_memory(input.shape[0], flags)
        tmp_adjoint = torch.empty((max(nbytes, 16),), dtype=torch.uint8, device=input.device)
        with self._mutex:
            self._set_network_parameters(network_parameters, encoding_parameters)
            if flags & GRADIENTS_NETWORK_WEIGHTS:
                check(lib.qmlp_network_set_parameter(self._handle, desc(grad_network), QMLP_GRADIENTS))
            if flags & GRADIENTS_INPUT_ENCODINGS:
                for i, g in enumerate(grad_encodings):
                    if g is not None:
                        self.encoding(i).set_parameter(g, gradients=True)
            adj = desc(adj_input if flags & GRADIENTS_INPUT else None)
            if contents is None:
                check(lib.qmlp_network_adjoint(self._handle, desc(input), desc(adj_output), int(flags), adj,
                                               ctypes.c_void_p(tmp_forward.data_ptr()),
                                               ctypes.c_void_p(tmp_adjoint.data_ptr()), current_stream(input.device)))
            else:
                check(lib.qmlp_network_adjoint_for(self._handle, desc(input), desc(adj_output), int(flags), 0, adj,
                                                   ctypes.c_void_p(tmp_forward.data_ptr()), int(contents),
                                                   ctypes.c_void_p(tmp_adjoint.data_ptr()), current_stream(input.device)))
            check(lib.qmlp_network_set_parameter(self._handle, None, QMLP_GRADIENTS))
            for i, g in enumerate(grad_encodings):
                if g is not None and self.encoding(i).has_parameters():
                    self.encoding(i).set_parameter(None, gradients=True)
        return adj_input, grad_network, grad_encodings

    def forward(self, input, network_parameters, encoding_parameters=()):
        """Differentiable forward pass; gradients flow to every argument that requires them."""
        return self._native.forward(input, network_parameters, list(encoding_parameters))

    def __getstate__(self):
        return (self._cfg, self._parent)

    def __setstate__(self, state):
        self.__init__(*state)
