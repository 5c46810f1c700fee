"""Networks and encodings under what PyTorch offers beside plain reverse mode: refused or recorded, as for any function without
rules of its own."""
import json
import threading

import pytest
import torch
from torch.autograd import forward_ad

import qmlp
from helpers import identity_cfg, warm_cache

pytestmark = pytest.mark.gpu

GRID = {"id": "HashGrid", "start_in": 0, "n_in": 3, "n_levels": 4, "n_features_per_level": 2, "log2_hashmap_size": 10, "min_resolution": 4,
        "max_resolution": 64, "combination_mode": "concat", "bounding_box_min": [0.0] * 3, "bounding_box_size": [1.0] * 3,
        "parameter_precision": "float"}
NETWORK = dict(identity_cfg(3, [32, 2], ["relu", "identity"], [True, False]), encodings=[GRID, {"id": "Identity", "start_in": 0, "n_in": 3}])


@pytest.fixture
def modules():
    warm_cache(NETWORK)
    network = qmlp.FusedNetwork(json.dumps(NETWORK), weight_dtype=torch.float32)
    encoding = qmlp.FusedEncoding(json.dumps(GRID))
    table = torch.nn.Parameter(encoding.create_parameter_tensor())
    with torch.no_grad():
        network.encoding_parameters[0].copy_(table)
    return network, encoding, table


def test_tangents_and_function_transforms_are_refused(modules):
    network, encoding, table = modules
    x = torch.rand(100, 3, device="cuda")
    calls = [network, lambda v: encoding(v, table), lambda v: encoding(v, table.detach())]
    for call in calls:
        with forward_ad.dual_level():
            with pytest.raises(NotImplementedError):
                call(forward_ad.make_dual(x, torch.ones_like(x)))
            call(x)
        with pytest.raises(RuntimeError):
            torch.func.vmap(call)(x[None])
        with pytest.raises(RuntimeError):
            torch.func.grad(lambda v: call(v).sum())(x)
    with forward_ad.dual_level(), pytest.raises(NotImplementedError):
        encoding(x, forward_ad.make_dual(table.detach(), torch.ones_like(table)))


def test_errors_of_a_backward_pass_are_those_of_the_native_library(modules):
    """Provoked by a hook that hands saved tensors of the wrong shape back: refused before anything is launched."""
    network, encoding, table = modules
    x = torch.rand(100, 3, device="cuda", requires_grad=True)
    for call in (network, lambda v: encoding(v, table)):
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t[:, :2] if t.dim() == 2 else t):
            out = call(x).sum()
        with pytest.raises(qmlp.QmlpError) as error:
            out.backward()
        assert error.value.code != 0
    call(x).sum().backward()


def test_a_differentiable_call_wants_the_parameters_of_every_encoding(modules):
    """... and does not take those that an earlier call has left bound."""
    network, encoding, _ = modules
    x = torch.rand(100, 3, device="cuda", requires_grad=True)
    table = network.encoding_parameters[0]
    network._network.forward(x, network.weights, [table, None]).sum().backward()
    for tables in ([], [None, None]):
        with pytest.raises(qmlp.QmlpError, match="encoding 0"):
            network._network.forward(x, network.weights, tables)
    with pytest.raises(RuntimeError, match="none are given"):
        encoding._encoding.forward_with_parameter(x, None)


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.filterwarnings("ignore")   # (of the tracer, about Python values)
def test_traced_modules_call_the_kernels_when_they_are_played(modules, grad):
    network, encoding, table = modules
    x = torch.rand(100, 3, device="cuda")
    with torch.set_grad_enabled(grad):
        calls = [(network, torch.jit.trace(network, x, check_trace=False), ()),
                 (encoding, torch.jit.trace(encoding, (x, table), check_trace=False), (table,))]
    for module, traced, more in calls:
        for n in (100, 777):
            x = torch.rand(n, 3, device="cuda", requires_grad=True)
            want, got = module(x, *more), traced(x, *more)
            assert torch.equal(got, want) and float(want.abs().max()) > 0
            leaves = [x, *more, *(p for p in module.parameters() if p.requires_grad)]
            g = torch.randn_like(want)
            for a, b in zip(torch.autograd.grad(got, leaves, g), torch.autograd.grad(want, leaves, g)):
                torch.testing.assert_close(a, b, rtol=0.0, atol=1e-5 * float(b.abs().max()))


def test_threads_run_backward_on_one_graph(modules):
    network, encoding, table = modules
    x = torch.rand(500, 3, device="cuda", requires_grad=True)
    leaves = {network: [x, network.weights], encoding: [x, table]}
    for module, call in ((network, network), (encoding, lambda v: encoding(v, table))):
        out = call(x)
        g = torch.randn_like(out)
        want = torch.autograd.grad(out, leaves[module], g, retain_graph=True)
        results = []

        def run():
            for i in range(50):
                results.append(torch.autograd.grad(out, leaves[module], g, retain_graph=True))

        threads = [threading.Thread(target=run) for _ in range(4)]
        [t.start() for t in threads]
        [t.join() for t in threads]
        assert len(results) == 200
        for got in results:
            for a, b in zip(got, want):
                torch.testing.assert_close(a, b, rtol=0.0, atol=1e-5 * float(b.abs().max()))


def test_tables_that_were_replaced_keep_their_place(modules):
    """A table that passes through a parametrization comes back at the end of its list's dict."""
    cfg = dict(identity_cfg(3, [32, 2], ["relu", "identity"], [True, False]), encodings=[GRID, GRID])
    warm_cache(cfg)
    network = qmlp.FusedNetwork(json.dumps(cfg), weight_dtype=torch.float32)
    for p in network.encoding_parameters:
        p.data.uniform_(-1, 1)
    x = torch.rand(200, 3, device="cuda")
    want = network(x)
    torch.nn.utils.parametrize.register_parametrization(network.encoding_parameters, "0", torch.nn.Identity())
    assert torch.equal(network(x), want)
    torch.nn.utils.parametrize.remove_parametrizations(network.encoding_parameters, "0")
    assert list(network.encoding_parameters._parameters) == ["1", "0"]
    assert torch.equal(network(x), want)
