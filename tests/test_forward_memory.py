"""The memory that a training pass leaves for the adjoint pass, moved in between: what it holds is told by the caller
(qmlp_network_forward_for, qmlp_network_adjoint_for) and not looked up by its address."""
import json

import pytest
import torch

import qmlp
from helpers import identity_cfg, warm_cache

pytestmark = pytest.mark.gpu


def behind_grid(n_in, levels, features, log2_size, options, encodings=()):
    grid = {"id": "HashGrid", "start_in": 0, "n_in": 3, "n_levels": levels, "n_features_per_level": features, "log2_hashmap_size": log2_size,
            "min_resolution": 8 if levels > 1 else 64, "max_resolution": 64, "combination_mode": "concat", "bounding_box_min": [0.0] * 3,
            "bounding_box_size": [1.0] * 3, "parameter_precision": "float"}
    return {"num_inputs": n_in, "num_outputs": 2, "activation_specification": ["qmlp/builtin-activations.json"],
            "encodings": [*encodings, grid], "options": options,
            "network": [{"n_out": 32, "bias": True, "activation": "relu"}, {"n_out": 2, "bias": False, "activation": "identity"}]}


# nothing stored; the encoded input only; all intermediates; position derivatives of the levels; rows in sorted order
SPECS = [
    (identity_cfg(4, [64] * 4 + [3], ["relu"] * 4 + ["identity"], [False] * 5), 9001),
    (identity_cfg(4, [16, 2], ["relu", "identity"], [True, True]), 700),
    (identity_cfg(4, [128, 128, 2], ["relu", "relu", "identity"], [True] * 3), 300),
    (behind_grid(3, 4, 2, 10, {"slice_gradients": 1}), 3001),
    (behind_grid(4, 1, 8, -1, {"sort_points": 1, "slice_gradients": 1}, [{"id": "Identity", "start_in": 3, "n_in": 1}]), 9001),
]


def problem(spec, points):
    net = qmlp.Network(json.dumps(spec))
    gen = torch.Generator(device="cuda").manual_seed(17)
    x = torch.rand(points, spec["num_inputs"], device="cuda", generator=gen)
    g = torch.randn(points, spec["num_outputs"], device="cuda", generator=gen)
    params = (torch.rand(net.num_network_parameters(), device="cuda", generator=gen) - 0.5)
    tables = [torch.rand(net.encoding(i).num_parameters(), device="cuda", generator=gen) if net.encoding(i).has_parameters() else None
              for i in range(net.num_encodings())]
    return net, x, g, params, tables


def close(got, want):
    # (records and points of one slab come in any order: the sums differ by rounding)
    for a, b in zip(got, want):
        torch.testing.assert_close(a, b, rtol=0.0, atol=1e-5 * float(b.abs().max()))


def elsewhere():
    """Hooks that keep saved tensors in host memory and bring them back at another address than they had."""
    kept = []

    def unpack(packed):
        kept.append(torch.zeros_like(packed, device="cuda"))     # (takes the place that was given back)
        return packed.cuda()

    return torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), unpack), kept


@pytest.mark.parametrize("spec,points", SPECS)
def test_saved_tensors_that_come_back_elsewhere(spec, points):
    warm_cache(spec)
    net, x, g, params, tables = problem(spec, points)

    def gradients():
        leaves = [t.clone().requires_grad_(True) for t in [x, params, *tables] if t is not None]
        rest = iter(leaves[2:])
        out = net.forward(leaves[0], leaves[1], [next(rest) if t is not None else None for t in tables])
        return torch.autograd.grad(out, leaves, g)

    want = gradients()
    hooks, kept = elsewhere()
    with hooks:
        got = gradients()
    assert len(kept) >= 3                                        # input, weights and the memory of the forward pass
    close(got, want)


@pytest.mark.parametrize("spec,points", SPECS)
@pytest.mark.parametrize("told", [False, True])
def test_a_copy_of_the_forward_memory(spec, points, told):
    """Of the pass that stores everything, and of the pass that was told which gradients follow; those and others."""
    warm_cache(spec)
    net, x, g, params, tables = problem(spec, points)
    half = params.half()
    every = 7 if any(t is not None for t in tables) else 3
    for flags in (every, 2, 1):
        out, memory, *contents = net.forward_raw(x, half, tables, flags, contents=True)
        want = net.adjoint_raw(x, g, flags, memory, half, tables, contents=contents[0])
        again, memory, *contents = net.forward_raw(x, half, tables, every, contents=told)
        assert torch.equal(again, out)
        copy = memory.clone()
        memory.fill_(255)                                        # NaN wherever it is read as halves or floats
        got = net.adjoint_raw(x, g, flags, copy, half, tables, **({"contents": contents[0]} if told else {}))
        pairs = [(got[0], want[0])] if flags & 1 else []
        pairs += [(got[1], want[1])] if flags & 2 else []
        pairs += [(a, b) for a, b in zip(got[2], want[2]) if flags & 4 and a is not None]
        assert pairs and all(float(b.abs().max()) > 0 for _, b in pairs)
        for a, b in pairs:
            # (position derivatives are halves, 2^-11 each; without them the grids are gathered from again)
            torch.testing.assert_close(a, b, rtol=0.0, atol=(2e-3 if told is False else 1e-5) * float(b.abs().max()))


@pytest.mark.parametrize("spec,points", SPECS[:2])
def test_saved_tensors_of_the_torch_custom_class_that_come_back_elsewhere(spec, points):
    warm_cache(spec)
    module = qmlp.FusedNetwork(json.dumps(spec), weight_dtype=torch.float32, scriptable=True)
    _, x, g, _, _ = problem(spec, points)
    x.requires_grad_(True)
    want = torch.autograd.grad(module(x), [x, module.weights], g)
    hooks, kept = elsewhere()
    with hooks:
        got = torch.autograd.grad(module(x), [x, module.weights], g)
    assert len(kept) >= 3
    close(got, want)
