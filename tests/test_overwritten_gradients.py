"""Gradients of the input and of the weights that the adjoint pass writes instead of adding to them
(qmlp_network_adjoint_overwriting): every element, whatever the tensor held."""
import ctypes
import json

import pytest
import torch

import qmlp
from helpers import identity_cfg, warm_cache
from qmlp._lib import QMLP_GRADIENTS, QMLP_INFERENCE, check, lib
from qmlp.classes import current_stream, desc

pytestmark = pytest.mark.gpu

GRID = {"id": "HashGrid", "start_in": 0, "n_in": 3, "n_levels": 1, "n_features_per_level": 8, "log2_hashmap_size": -1,
        "min_resolution": 64, "max_resolution": 64, "combination_mode": "concat", "bounding_box_min": [0.0] * 3,
        "bounding_box_size": [1.0] * 3, "parameter_precision": "float"}


def behind_grid(num_inputs, encodings, options):
    return {"num_inputs": num_inputs, "num_outputs": 2, "activation_specification": ["qmlp/builtin-activations.json"],
            "encodings": encodings, "options": options,
            "network": [{"n_out": 32, "bias": True, "activation": "relu"}, {"n_out": 2, "bias": False, "activation": "identity"}]}


PARTIAL = identity_cfg(3, [48, 2], ["relu", "identity"], [True, True])
PARTIAL = dict(PARTIAL, num_inputs=5, encodings=[{"id": "Identity", "start_in": 1, "n_in": 3}])
IDENTITY = {"id": "Identity", "start_in": 0, "n_in": 2}
# specification, batch, gradients (1: input, 2: weights) that may be overwritten
SPECS = [
    (identity_cfg(4, [64, 48, 3], ["sine", "celu", "identity"], [True] * 3), 8192 + 33, 3),   # the rows of the input themselves
    (identity_cfg(3, [64, 48, 3], ["sine", "celu", "identity"], [True] * 3), 70001, 3),
    (PARTIAL, 8192 + 33, 2),                                                                  # channels that no encoding reads
    (identity_cfg(4, [16, 2], ["relu", "identity"], [True] * 2), 100, 2),                     # stored intermediates
    (behind_grid(3, [IDENTITY, GRID], {"sort_points": 1, "slice_gradients": 1}), 70001, 3),   # sorted; two encodings
    (behind_grid(4, [IDENTITY, GRID], {"sort_points": 1, "slice_gradients": 1}), 70001, 3),   # sorted; rows of four
    (behind_grid(3, [GRID], {"sort_points": 1, "slice_gradients": 1}), 70001, 3),             # sorted; no encoding in the backward kernel
    (behind_grid(3, [GRID], {"sort_points": 1, "slice_gradients": 0}), 70001, 3),             # sorted; atomics in the backward kernel
    (behind_grid(3, [IDENTITY, GRID], {"sort_points": 0, "slice_gradients": 1, "cooperative_backward": 1}), 9000, 3),
]


@pytest.mark.parametrize("spec,points,expected", SPECS)
def test_overwritten_gradients(spec, points, expected):
    warm_cache(spec)
    net = qmlp.Network(json.dumps(spec))
    gen = torch.Generator(device="cuda").manual_seed(3)
    x = torch.rand(points, spec["num_inputs"], device="cuda", generator=gen)
    g = torch.randn(points, spec["num_outputs"], device="cuda", generator=gen)
    params = (torch.rand(net.num_network_parameters(), device="cuda", generator=gen) - 0.5).to(torch.float16)
    check(lib.qmlp_network_set_parameter(net._handle, desc(params), QMLP_INFERENCE))
    flags, tables = 3, []
    for i, e in enumerate(spec["encodings"]):
        if e["id"] == "HashGrid":
            flags = 7
            table = torch.rand(net.encoding(i).num_parameters(), device="cuda", generator=gen)
            tables += [table, torch.zeros_like(table)]
            net.encoding(i).set_parameter(table)
            net.encoding(i).set_parameter(tables[-1], gradients=True)
    stream = current_stream(x.device)
    size = ctypes.c_size_t()
    out = torch.empty(points, spec["num_outputs"], device="cuda")
    results = []
    for overwriting in (False, True):
        check(lib.qmlp_network_forward_memory(net._handle, points, flags, ctypes.byref(size)))
        forward = torch.empty(max(size.value, 16), dtype=torch.uint8, device="cuda")
        check(lib.qmlp_network_adjoint_memory(net._handle, points, flags, ctypes.byref(size)))
        scratch = torch.full((max(size.value, 16),), 255, dtype=torch.uint8, device="cuda")   # NaN wherever it is read as floats
        check(lib.qmlp_network_forward(net._handle, desc(x), desc(out), forward.data_ptr(), stream))
        mask = ctypes.c_int()
        check(lib.qmlp_network_overwritable_gradients(net._handle, points, flags, forward.data_ptr(), ctypes.byref(mask)))
        assert mask.value == expected
        overwrite = mask.value if overwriting else 0
        adj_x = torch.full_like(x, float("nan") if overwrite & 1 else 0.0)
        adj_params = torch.full((params.numel(),), float("nan") if overwrite & 2 else 0.0, device="cuda")
        check(lib.qmlp_network_set_parameter(net._handle, desc(adj_params), QMLP_GRADIENTS))
        check(lib.qmlp_network_adjoint_overwriting(net._handle, desc(x), desc(g), flags, overwrite, desc(adj_x), forward.data_ptr(),
                                                   scratch.data_ptr(), stream))
        results.append((adj_x, adj_params))
    assert float(results[0][0].abs().sum()) > 0 and float(results[0][1].abs().sum()) > 0
    assert torch.equal(results[0][0], results[1][0])
    # (points of one slab are sorted in any order: the sums over the batch differ by rounding)
    rounding = 1e-5 * float(results[0][1].abs().max()) if spec.get("options", {}).get("sort_points") else 0.0
    torch.testing.assert_close(results[1][1], results[0][1], rtol=0.0, atol=rounding)
    if expected != 3:
        with pytest.raises(qmlp.QmlpError, match="asked to overwrite"):
            check(lib.qmlp_network_adjoint_overwriting(net._handle, desc(x), desc(g), flags, 3, desc(results[0][0]), forward.data_ptr(),
                                                       scratch.data_ptr(), stream))
