// qmlp._native: the calls that a training or rendering loop makes once per batch (FusedNetwork.forward, a standalone
// encoding, and their backward passes), from Python straight into C++. A call on a small batch is bound by the host:
// inference on 1000 points takes 8 us beside a kernel of 3.4 us, a train step on 513 points 60 us beside kernels of 20 us;
// through ctypes and a Python autograd function they took 13 and 143 us. Everything else of the Python package stays on ctypes.
//
// Like the torch custom classes (qmlp_torch.cpp) this is written on the C ABI of libqmlp.so; the autograd node
// replaces the one of the reference's binding (src_cpp/pytorch-bindings/src/bind_network.cpp:189-319).
#include <torch/extension.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/Exceptions.h>
#include <ATen/FuncTorchTLS.h>
#include <ATen/TracerMode.h>
#include <c10/hip/HIPStream.h>

#include "qmlp_capi.h"

#include <atomic>
#include <cstdint>
#include <memory>
#include <mutex>
#include <vector>

namespace {

using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

/** A failed call of the C ABI, as the exception class of the Python package (qmlp.QmlpError with its code). */
struct Failure
{
    int code;
    std::string message;
};
void check(int rc)
{
    if (rc != 0) throw Failure{rc, qmlp_last_error()};
}
void setError(const Failure& f)
{
    py::object cls = py::module_::import("qmlp._lib").attr("QmlpError");
    PyErr_SetObject(cls.ptr(), cls(f.code, f.message).ptr());
}
[[noreturn]] void raise(const Failure& f)
{
    py::gil_scoped_acquire gil;
    setError(f);
    throw py::error_already_set();
}
/** The exception in flight out of a backward pass: in the form in which the threads of the autograd engine hand on exceptions of Python. */
[[noreturn]] void raiseFromBackward()
{
    auto persist = [] {
        python_error e;
        e.persist();
        throw e;
    };
    try {
        throw;
    } catch (const Failure& f) {
        py::gil_scoped_acquire gil;
        setError(f);
        persist();
    } catch (const py::builtin_exception& e) {
        py::gil_scoped_acquire gil;
        e.set_error();
        persist();
    }
    throw std::logic_error("unreachable");
}

qmlp_tensor wrap(const at::Tensor& t)
{
    qmlp_tensor d{};
    if (!t.defined()) return d;
    const auto dim = t.dim();
    if (dim < 1 || dim > 4) throw py::value_error("tensors must have 1 to 4 dimensions");
    switch (t.scalar_type()) {
        case at::kFloat: d.precision = QMLP_FLOAT; break;
        case at::kHalf: d.precision = QMLP_HALF; break;
        case at::kDouble: d.precision = QMLP_DOUBLE; break;
        default: throw py::type_error("unsupported dtype " + std::string(c10::toString(t.scalar_type())));
    }
    d.data = t.data_ptr();
    d.ndim = static_cast<int32_t>(dim);
    const auto sizes = t.sizes(), strides = t.strides();
    for (int i = 0; i < d.ndim; ++i) {
        if (sizes[i] > INT32_MAX || strides[i] > INT32_MAX) throw py::value_error("sizes and strides of tensors must fit into 32 bits");
        d.sizes[i] = static_cast<int32_t>(sizes[i]);
        d.strides[i] = static_cast<int32_t>(strides[i]);
    }
    return d;
}

void* currentStream(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

at::Tensor bytesOn(const at::Tensor& like, size_t bytes)
{
    return at::empty({static_cast<int64_t>(std::max<size_t>(bytes, 16))}, like.options().dtype(at::kByte).requires_grad(false));
}

/**
 * A network of the C ABI with what its calls need, kept alive by the Python object and by the autograd graph. The
 * native network keeps the parameter tensors of the call in progress: one call at a time (lock / unlock; the lock is
 * never waited for, nor held across a wait, with the interpreter lock in hand).
 */
struct Network
{
    qmlp_network_t handle;
    std::mutex mutex;
    int channelsOut = 0;
    struct Encoding
    {
        qmlp_encoding_t handle = nullptr;
        bool hasParameters = false;
    };
    std::vector<Encoding> encodings;

    explicit Network(uintptr_t h) : handle(reinterpret_cast<qmlp_network_t>(h))
    {
        int n = 0;
        check(qmlp_network_channels_out(handle, &channelsOut));
        check(qmlp_network_num_encodings(handle, &n));
        encodings.resize(n);
        for (int i = 0; i < n; ++i) {
            int has = 0;
            check(qmlp_network_encoding(handle, i, &encodings[i].handle));
            check(qmlp_encoding_has_parameters(encodings[i].handle, &has));
            encodings[i].hasParameters = has != 0;
        }
    }
    ~Network() { qmlp_network_destroy(handle); }

    /** Binds the inference parameters of the network and of its encodings (under the lock). */
    void bind(const qmlp_tensor& network, const std::vector<qmlp_tensor>& tables)
    {
        check(qmlp_network_set_parameter(handle, &network, QMLP_INFERENCE));
        for (size_t i = 0; i < std::min(tables.size(), encodings.size()); ++i)
            if (tables[i].ndim > 0 && encodings[i].hasParameters)
                check(qmlp_encoding_set_parameter(encodings[i].handle, &tables[i], QMLP_INFERENCE));
    }
};
using Network_ptr = std::shared_ptr<Network>;

/** The tensors of a list; None: an undefined tensor. */
std::vector<at::Tensor> tensorsOf(const py::list& list)
{
    std::vector<at::Tensor> tensors;
    tensors.reserve(list.size());
    for (const auto& item : list) {
        if (item.is_none()) tensors.emplace_back();
        else tensors.push_back(item.cast<at::Tensor>());
    }
    return tensors;
}

std::vector<qmlp_tensor> wrapAll(const Network& net, const std::vector<at::Tensor>& tables)
{
    std::vector<qmlp_tensor> wrapped(std::min(tables.size(), net.encodings.size()));
    for (size_t i = 0; i < wrapped.size(); ++i)
        if (net.encodings[i].hasParameters) wrapped[i] = wrap(tables[i]);
    return wrapped;
}

at::Tensor createOutput(const at::Tensor& input, int channels)
{
    if (!input.is_cuda()) throw std::runtime_error("QuickMLP tensors must live on the GPU");
    if (input.dim() != 2) throw std::runtime_error("input must be a tensor with 2 dimensions (batch, channels)");
    return at::empty({input.size(0), channels}, input.options().requires_grad(false));
}

/**
 * The nodes below know reverse mode only, and calls below the dispatcher look at the memory of a tensor and at nothing else:
 * transforms of torch.func and tensors with a tangent are refused, as torch refuses them for functions without rules for them.
 */
void refuseOtherModes(at::TensorList tensors)
{
    if (const auto& functorch = at::functorch::functorchTLSAccessor()) functorch->checkSupportsCppAutogradFunction();
    for (const auto& t : tensors) {
        if (!t.defined() || !t._fw_grad(0).defined()) continue;
        PyErr_SetString(PyExc_NotImplementedError, "forward-mode AD is not implemented for networks and encodings");
        throw py::error_already_set();
    }
}

at::Tensor inference(const Network_ptr& net, const at::Tensor& input, const at::Tensor& parameters, const std::vector<at::Tensor>& tables)
{
    try {
        at::AutoDispatchBelowADInplaceOrView guard;
        auto output = createOutput(input, net->channelsOut);
        const auto p16 = parameters.scalar_type() == at::kHalf ? parameters : parameters.to(at::kHalf);
        const auto wrappedTables = wrapAll(*net, tables);
        const qmlp_tensor p = wrap(p16), in = wrap(input), out = wrap(output);
        void* stream = currentStream(input);
        {
            py::gil_scoped_release release;
            std::lock_guard<std::mutex> lock(net->mutex);
            net->bind(p, wrappedTables);
            check(qmlp_network_inference(net->handle, &in, &out, stream));
        }
        return output;
    } catch (const Failure& f) {
        raise(f);
    }
}

/** What a forward pass leaves for its adjoint pass, beside its inputs. */
struct ForwardPass
{
    at::Tensor output, memory;
    int contents = 0;   // of the memory
};

/** parameters: in half precision; tables: undefined for encodings without parameters */
ForwardPass forwardPass(const Network_ptr& net, const at::Tensor& input, const at::Tensor& parameters, const std::vector<at::Tensor>& tables, int flags)
{
    ForwardPass pass;
    pass.output = createOutput(input, net->channelsOut);
    at::AutoDispatchBelowADInplaceOrView guard;
    const auto wrappedTables = wrapAll(*net, tables);
    const qmlp_tensor p = wrap(parameters), in = wrap(input), out = wrap(pass.output);
    void* stream = currentStream(input);
    py::gil_scoped_release release;
    std::lock_guard<std::mutex> lock(net->mutex);
    size_t bytes = 0;
    check(qmlp_network_forward_memory(net->handle, in.sizes[0], flags, &bytes));
    pass.memory = bytesOn(input, bytes);
    net->bind(p, wrappedTables);
    check(qmlp_network_forward_for(net->handle, &in, &out, flags, pass.memory.data_ptr(), &pass.contents, stream));
    return pass;
}

/** Gradients of the input, the network parameters and the tables, those of parameters in floats; undefined where flags do not ask for them. */
struct Gradients
{
    at::Tensor input, network;
    std::vector<at::Tensor> tables;
};

Gradients adjointPass(const Network_ptr& net, const at::Tensor& input, const at::Tensor& parameters, const std::vector<at::Tensor>& tables,
                      const at::Tensor& memory, int contents, const at::Tensor& adjOutput, int flags)
{
    const size_t n = net->encodings.size();
    // (memory: may have been elsewhere in between, see saved-tensor hooks)
    TORCH_CHECK(input.is_cuda() && memory.device() == input.device() && memory.is_contiguous(), "saved tensors came back on another device");
    at::AutoDispatchBelowADInplaceOrView guard;
    Gradients g;
    g.tables.resize(n);
    // zeroed only where the kernels add to them
    int overwriteTables = 0;
    if (flags & QMLP_GRADIENTS_INPUT_ENCODINGS) {
        {
            std::lock_guard<std::mutex> lock(net->mutex);
            check(qmlp_network_overwritable_tables(net->handle, wrap(input).sizes[0], flags, &overwriteTables));
        }
        // the kernel adds the gradients of every encoding with parameters: a frozen one gets a zero tensor as
        // well, which the callers drop (bind_network.cpp:277-290)
        for (size_t i = 0; i < n; ++i)
            if (net->encodings[i].hasParameters) {
                const auto options = tables.at(i).options().dtype(at::kFloat);
                g.tables[i] = overwriteTables ? at::empty(tables[i].sizes(), options) : at::zeros(tables[i].sizes(), options);
            }
    }
    void* stream = currentStream(input);
    const auto wrappedTables = wrapAll(*net, tables);
    const qmlp_tensor p = wrap(parameters), in = wrap(input), adjOut = wrap(adjOutput);
    std::vector<qmlp_tensor> adjEnc(n);
    for (size_t i = 0; i < n; ++i) adjEnc[i] = wrap(g.tables[i]);
    std::lock_guard<std::mutex> lock(net->mutex);
    size_t bytes = 0;
    check(qmlp_network_adjoint_memory(net->handle, in.sizes[0], flags, &bytes));
    const at::Tensor scratch = bytesOn(input, bytes);
    net->bind(p, wrappedTables);
    int overwrite = 0;
    check(qmlp_network_overwritable_gradients(net->handle, in.sizes[0], flags, nullptr, &overwrite));
    if (overwriteTables) overwrite |= QMLP_GRADIENTS_INPUT_ENCODINGS;
    if (flags & QMLP_GRADIENTS_INPUT) g.input = overwrite & QMLP_GRADIENTS_INPUT ? at::empty_like(input) : at::zeros_like(input);
    if (flags & QMLP_GRADIENTS_NETWORK_WEIGHTS) {
        const auto options = parameters.options().dtype(at::kFloat);
        g.network = overwrite & QMLP_GRADIENTS_NETWORK_WEIGHTS ? at::empty(parameters.sizes(), options) : at::zeros(parameters.sizes(), options);
    }
    const qmlp_tensor adjIn = wrap(g.input), adjNet = wrap(g.network);
    struct Unbind   // no dangling gradient bindings, whatever happens
    {
        Network& net;
        bool tables;
        ~Unbind()
        {
            qmlp_network_set_parameter(net.handle, nullptr, QMLP_GRADIENTS);
            for (const auto& e : net.encodings)
                if (tables && e.hasParameters) qmlp_encoding_set_parameter(e.handle, nullptr, QMLP_GRADIENTS);
        }
    } unbind{*net, (flags & QMLP_GRADIENTS_INPUT_ENCODINGS) != 0};
    if (g.network.defined()) check(qmlp_network_set_parameter(net->handle, &adjNet, QMLP_GRADIENTS));
    for (size_t i = 0; i < n; ++i)
        if (g.tables[i].defined()) check(qmlp_encoding_set_parameter(net->encodings[i].handle, &adjEnc[i], QMLP_GRADIENTS));
    check(qmlp_network_adjoint_for(net->handle, &in, &adjOut, flags, overwrite, &adjIn, memory.data_ptr(), contents, scratch.data_ptr(), stream));
    return g;
}

/** The backward pass of one forward call: outputs are the gradients of (input, network parameters, tables ...). */
struct FusedBackward : torch::autograd::Node
{
    Network_ptr net;
    int flags = 0;
    SavedVariable input, p16, memory;
    std::vector<SavedVariable> tables;
    int contents = 0;   // of the memory
    at::ScalarType parameterType = at::kHalf;

    std::string name() const override { return "QmlpFusedBackward"; }
    void release_variables() override
    {
        std::lock_guard<std::mutex> lock(mutex_);   // (as generated nodes do: two threads may run backward on one graph)
        input.reset_data();
        p16.reset_data();
        for (auto& t : tables) t.reset_data();
        memory.reset_data();
    }

    variable_list apply(variable_list&& gradOutputs) override
    {
        std::lock_guard<std::mutex> lock(mutex_);
        const size_t n = net->encodings.size();
        variable_list grads(2 + n);
        if (!gradOutputs[0].defined()) return grads;
        const at::Tensor x = input.unpack(), parameters = p16.unpack();
        std::vector<at::Tensor> unpacked(n);
        for (size_t i = 0; i < n; ++i)
            if (net->encodings[i].hasParameters) unpacked[i] = tables[i].unpack();
        Gradients g;
        try {
            g = adjointPass(net, x, parameters, unpacked, memory.unpack(), contents, gradOutputs[0].contiguous(), flags);
        } catch (...) {
            raiseFromBackward();
        }
        at::AutoDispatchBelowADInplaceOrView guard;
        if (g.input.defined() && task_should_compute_output(0)) grads[0] = g.input;
        if (g.network.defined() && task_should_compute_output(1)) grads[1] = g.network.to(parameterType);
        for (size_t i = 0; i < n; ++i)
            if (g.tables[i].defined() && task_should_compute_output(2 + i)) grads[2 + i] = g.tables[i].to(unpacked[i].scalar_type());
        return grads;
    }
};

at::Tensor halves(const at::Tensor& parameters)
{
    at::AutoDispatchBelowADInplaceOrView guard;
    return parameters.scalar_type() == at::kHalf ? parameters : parameters.to(at::kHalf);
}

/** Differentiable forward pass; gradients flow to every argument that requires them. */
at::Tensor forward(const Network_ptr& net, const at::Tensor& input, const at::Tensor& parameters, const std::vector<at::Tensor>& tables)
{
    const size_t n = net->encodings.size();
    int flags = 0;
    if (at::GradMode::is_enabled()) {
        if (input.requires_grad()) flags |= QMLP_GRADIENTS_INPUT;
        if (parameters.requires_grad()) flags |= QMLP_GRADIENTS_NETWORK_WEIGHTS;
        for (size_t i = 0; i < std::min(n, tables.size()); ++i)
            if (net->encodings[i].hasParameters && tables[i].defined() && tables[i].requires_grad()) flags |= QMLP_GRADIENTS_INPUT_ENCODINGS;
    }
    if (flags == 0) return inference(net, input, parameters, tables);
    std::vector<at::Tensor> positions(n);   // of encodings without parameters: undefined
    for (size_t i = 0; i < n; ++i) {
        if (!net->encodings[i].hasParameters) continue;
        if (i < tables.size()) positions[i] = tables[i];
        if (!positions[i].defined()) raise(Failure{2, "encoding " + std::to_string(i) + " has parameters, but none are given"});
    }
    refuseOtherModes({input, parameters});
    refuseOtherModes(positions);
    const at::Tensor p16 = halves(parameters);
    ForwardPass pass;
    try {
        pass = forwardPass(net, input, p16, positions, flags);
    } catch (const Failure& f) {
        raise(f);
    }
    auto node = std::shared_ptr<FusedBackward>(new FusedBackward(), torch::autograd::deleteNode);
    node->set_next_edges(torch::autograd::collect_next_edges(input, parameters, at::TensorList(positions)));
    node->net = net;
    node->flags = flags;
    node->input = SavedVariable(input, false);
    node->p16 = SavedVariable(p16, false);
    node->tables.reserve(n);
    for (const auto& t : positions) node->tables.emplace_back(t, false);
    node->memory = SavedVariable(pass.memory, false);
    node->contents = pass.contents;
    node->parameterType = parameters.scalar_type();
    torch::autograd::set_history(pass.output, node);
    return pass.output;
}

// ------------------------------------------------------------------------------------------------ standalone encodings
/** An encoding of the C ABI, of its own or of a network (which it keeps alive), one call at a time. */
struct Encoding
{
    qmlp_encoding_t handle;
    Network_ptr network;
    std::mutex ownMutex;
    std::mutex& mutex;
    int channelsOut = 0;
    std::atomic<long long> calls{0};   // each leaves the native encoding without a bound table

    Encoding(uintptr_t h, Network_ptr net)
        : handle(reinterpret_cast<qmlp_encoding_t>(h)), network(std::move(net)), mutex(network ? network->mutex : ownMutex)
    {
        check(qmlp_encoding_num_output_channels(handle, &channelsOut));
    }
    ~Encoding() { if (!network) qmlp_encoding_destroy(handle); }
};
using Encoding_ptr = std::shared_ptr<Encoding>;

/** parameter: undefined for encodings without parameters */
at::Tensor encode(const Encoding_ptr& enc, const at::Tensor& input, const at::Tensor& parameter)
{
    try {
        at::AutoDispatchBelowADInplaceOrView guard;
        auto output = createOutput(input, enc->channelsOut);
        const qmlp_tensor in = wrap(input), out = wrap(output), par = wrap(parameter);
        void* stream = currentStream(input);
        {
            py::gil_scoped_release release;
            std::lock_guard<std::mutex> lock(enc->mutex);
            ++enc->calls;
            check(qmlp_encoding_forward(enc->handle, &in, &out, stream, parameter.defined() ? &par : nullptr));
        }
        return output;
    } catch (const Failure& f) {
        raise(f);
    }
}

/** Gradients of input and parameter (in float); undefined where they were not asked for or there are none. */
std::pair<at::Tensor, at::Tensor> encodeAdjoint(Encoding& enc, const at::Tensor& input, const at::Tensor& parameter, const at::Tensor& adjOutput, int flags)
{
    at::AutoDispatchBelowADInplaceOrView guard;
    // (the native call wants the tensor in any case: without input gradients it is not written)
    at::Tensor adjInput = flags & QMLP_ENCODING_INPUT_GRADIENTS ? at::zeros_like(input) : at::Tensor();
    std::lock_guard<std::mutex> lock(enc.mutex);
    ++enc.calls;
    size_t bytes = 0;
    check(qmlp_encoding_adjoint_memory(enc.handle, wrap(input).sizes[0], flags, &bytes));
    at::Tensor memory;
    if (bytes > 0) memory = bytesOn(input, bytes);
    at::Tensor adjParameter;
    if (parameter.defined() && (flags & QMLP_ENCODING_PARAM_GRADIENTS)) {
        // with the memory the table's gradients are written, without it added to
        const auto options = parameter.options().dtype(at::kFloat);
        adjParameter = bytes > 0 ? at::empty(parameter.sizes(), options) : at::zeros(parameter.sizes(), options);
    }
    const qmlp_tensor in = wrap(input), adjOut = wrap(adjOutput), adjIn = adjInput.defined() ? wrap(adjInput) : in, par = wrap(parameter),
                      adjPar = wrap(adjParameter);
    auto* adjoint = bytes > 0 && adjParameter.defined() ? qmlp_encoding_adjoint_overwriting : qmlp_encoding_adjoint_in;
    check(adjoint(enc.handle, &in, &adjOut, &adjIn, currentStream(input), parameter.defined() ? &par : nullptr,
                  adjParameter.defined() ? &adjPar : nullptr, flags, bytes > 0 ? memory.data_ptr() : nullptr));
    return {adjInput, adjParameter};
}

struct EncodingBackward : torch::autograd::Node
{
    Encoding_ptr enc;
    int flags = 0;
    SavedVariable input, parameter;

    std::string name() const override { return "QmlpEncodingBackward"; }
    void release_variables() override
    {
        std::lock_guard<std::mutex> lock(mutex_);   // (as generated nodes do: two threads may run backward on one graph)
        input.reset_data();
        parameter.reset_data();
    }
    variable_list apply(variable_list&& gradOutputs) override
    {
        std::lock_guard<std::mutex> lock(mutex_);
        variable_list grads(2);
        if (!gradOutputs[0].defined()) return grads;
        const at::Tensor x = input.unpack(), table = parameter.unpack();
        try {
            auto [adjInput, adjParameter] = encodeAdjoint(*enc, x, table, gradOutputs[0].contiguous(), flags);
            if (adjInput.defined() && task_should_compute_output(0)) grads[0] = adjInput;
            if (adjParameter.defined() && task_should_compute_output(1)) grads[1] = adjParameter.to(table.scalar_type());
        } catch (...) {
            raiseFromBackward();
        }
        return grads;
    }
};

at::Tensor encodeForward(const Encoding_ptr& enc, const at::Tensor& input, const at::Tensor& parameter)
{
    refuseOtherModes({input, parameter});
    int flags = 0;
    if (at::GradMode::is_enabled()) {
        if (input.requires_grad()) flags |= QMLP_ENCODING_INPUT_GRADIENTS;
        if (parameter.defined() && parameter.requires_grad()) flags |= QMLP_ENCODING_PARAM_GRADIENTS;
    }
    auto output = encode(enc, input, parameter);
    if (flags == 0) return output;
    auto node = std::shared_ptr<EncodingBackward>(new EncodingBackward(), torch::autograd::deleteNode);
    node->set_next_edges(torch::autograd::collect_next_edges(input, parameter));
    node->enc = enc;
    node->flags = flags;
    node->input = SavedVariable(input, false);
    node->parameter = SavedVariable(parameter, false);
    torch::autograd::set_history(output, node);
    return output;
}

at::Tensor tensorOrNone(const py::object& o) { return o.is_none() ? at::Tensor() : o.cast<at::Tensor>(); }
py::object noneOr(const at::Tensor& t) { return t.defined() ? py::cast(t) : py::none(); }

/**
 * While torch.jit.trace records, a call goes through the function of the Python package that it can record: of what is done
 * here it would see the allocation of the output and nothing else.
 */
bool recording() { return at::tracer::impl::is_dispatch_enabled(); }
py::object recorded(const char* function) { return py::module_::import("qmlp.classes").attr(function).attr("apply"); }

} // namespace

PYBIND11_MODULE(_native, m)
{
    py::register_exception_translator([](std::exception_ptr p) {
        try {
            if (p) std::rethrow_exception(p);
        } catch (const Failure& f) {
            setError(f);
        }
    });
    py::class_<Network, Network_ptr>(m, "Network")
        .def(py::init<uintptr_t>())   // takes the handle over
        // as a context manager: the lock of the native network
        .def("__enter__", [](const Network_ptr& net) { py::gil_scoped_release release; net->mutex.lock(); })
        .def("__exit__", [](const Network_ptr& net, const py::args&) { net->mutex.unlock(); })
        .def("bind",
             [](const Network_ptr& net, const at::Tensor& parameters, const py::list& tables) {
                 net->bind(wrap(parameters), wrapAll(*net, tensorsOf(tables)));
             },
             "Binds inference parameters (with the lock held).")
        .def("inference", [](const Network_ptr& net, const at::Tensor& input, const at::Tensor& parameters,
                             const py::list& tables) { return inference(net, input, parameters, tensorsOf(tables)); })
        .def("forward", [](const Network_ptr& net, const at::Tensor& input, const at::Tensor& parameters, const py::list& tables) {
            if (!recording()) return forward(net, input, parameters, tensorsOf(tables));
            py::list positions;
            for (size_t i = 0; i < net->encodings.size(); ++i)
                positions.append(net->encodings[i].hasParameters && i < tables.size() ? py::object(tables[i]) : py::object(py::none()));
            return recorded("_RecordedNetwork")(net, input, parameters, *py::tuple(positions)).cast<at::Tensor>();
        })
        .def("forward_pass",
             [](const Network_ptr& net, const at::Tensor& input, const at::Tensor& parameters, const py::list& tables, int flags) {
                 const auto pass = forwardPass(net, input, parameters, tensorsOf(tables), flags);
                 return py::make_tuple(pass.output, pass.memory, pass.contents);
             },
             "(output, memory, contents) without autograd; parameters: in half precision.")
        .def("adjoint_pass",
             [](const Network_ptr& net, const at::Tensor& input, const at::Tensor& parameters, const py::list& tables, const at::Tensor& memory,
                int contents, const at::Tensor& adjOutput, int flags) {
                 const auto unwrapped = tensorsOf(tables);
                 Gradients g;
                 {
                     py::gil_scoped_release release;
                     g = adjointPass(net, input, parameters, unwrapped, memory, contents, adjOutput, flags);
                 }
                 py::list adjTables;
                 for (const auto& t : g.tables) adjTables.append(noneOr(t));
                 return py::make_tuple(noneOr(g.input), noneOr(g.network), adjTables);
             },
             "Gradients (input, parameters, [tables]), those of parameters in floats; None where flags do not ask for them.");
    py::class_<Encoding, Encoding_ptr>(m, "Encoding")
        .def(py::init<uintptr_t, Network_ptr>())   // handle, the network it belongs to (None: it is taken over)
        // as a context manager: the lock of the native encoding, of its network if it belongs to one
        .def("__enter__", [](const Encoding_ptr& enc) { py::gil_scoped_release release; enc->mutex.lock(); })
        .def("__exit__", [](const Encoding_ptr& enc, const py::args&) { enc->mutex.unlock(); })
        .def_property_readonly("calls", [](const Encoding_ptr& enc) { return enc->calls.load(); })
        .def("inference", [](const Encoding_ptr& enc, const at::Tensor& input, const py::object& parameter) {
            return encode(enc, input, tensorOrNone(parameter));
        })
        .def("forward", [](const Encoding_ptr& enc, const at::Tensor& input, const py::object& parameter) {
            if (recording()) return recorded("_RecordedEncoding")(enc, input, parameter).cast<at::Tensor>();
            return encodeForward(enc, input, tensorOrNone(parameter));
        })
        .def("adjoint_pass",
             [](const Encoding_ptr& enc, const at::Tensor& input, const py::object& parameter, const at::Tensor& adjOutput, int flags) {
                 const at::Tensor p = tensorOrNone(parameter);
                 std::pair<at::Tensor, at::Tensor> g;
                 {
                     py::gil_scoped_release release;
                     g = encodeAdjoint(*enc, input, p, adjOutput, flags);
                 }
                 return py::make_tuple(noneOr(g.first), noneOr(g.second));
             },
             "Gradients (input, parameter), the latter in floats; None where flags do not ask for them.");
}
