"""Table gradients that the slice kernels write instead of adding to a zeroed tensor: every element, whatever the tensor held,
and the sum that adding gives. Batches at the edges of regions (1024 to 128 points), tables whose slices end inside a dense
level, points outside of the box, all points in one cell (long segments), adjoints of zero."""
import ctypes
import json

import pytest
import torch

import qmlp
from helpers import require_gpu, warm_cache
from qmlp._lib import QMLP_INFERENCE, check, lib
from qmlp.classes import current_stream, desc

pytestmark = pytest.mark.gpu


def grid(levels, features, log2_size, precision, dims=3, resolution=(5, 200)):
    return {"id": "HashGrid", "start_in": 0, "n_in": dims, "n_levels": levels, "n_features_per_level": features,
            "log2_hashmap_size": log2_size, "min_resolution": resolution[0], "max_resolution": resolution[1],
            "combination_mode": "concat", "bounding_box_min": [0.0] * dims, "bounding_box_size": [1.0] * dims,
            "parameter_precision": precision}


GRIDS = [grid(8, 2, 13, "float"), grid(9, 1, 14, "half"), grid(11, 4, 12, "float", 2),
         grid(8, 2, 16, "float", 2, (100, 20000)),   # hashed, more cells along a coordinate than a slice has entries
         grid(8, 3, 18, "float", 3, (8, 60))]        # dense levels of several slices, entries that are no power of two


def points_of(kind, count, dims, gen):
    x = torch.rand(count, dims, device="cuda", generator=gen)
    if kind == "outside":
        x[::7] = x[::7] * 1.02 - 0.01
    elif kind == "one cell":
        x = 0.731 + 1e-4 * x
    return x


def assert_same(kind, written, added, adjoints):
    """Float additions come in any order (all of them of the atomic path; else coarse levels, first entries of slices,
    exceptions): each rounds with a standard deviation of at most 2^-24 / sqrt(3) of the running sum, a random walk (adjoints of both
    signs) that ends within the largest sum of the table, or for points outside within the largest term: weights there (0.01
    beyond the box, two of 200 cells) reach 3 per coordinate. Two sums of k terms differ by sqrt(2 k / 3) 2^-24 of that, here by six
    of these, and no entry gets more terms than there are points."""
    largest = max(float(added.abs().max()), 27.0 * float(adjoints.abs().max()) if kind == "outside" else 0.0)
    torch.testing.assert_close(written, added, rtol=1e-5, atol=6 * (2 * adjoints.shape[0] / 3) ** 0.5 * 2.0 ** -24 * largest)


@pytest.mark.parametrize("cfg", GRIDS)
@pytest.mark.parametrize("count", [1 << 14, (1 << 15) + 1, 3 * 1024 * 16 - 1])
@pytest.mark.parametrize("kind", ["even", "outside", "one cell"])
def test_encoding(cfg, count, kind):
    if kind == "outside" and cfg["max_resolution"] > 200:
        pytest.skip("weights of a point outside grow with the resolution")
    require_gpu(cfg, (2,))
    enc = qmlp.Encoding(json.dumps(cfg))
    gen = torch.Generator(device="cuda").manual_seed(count)
    x = points_of(kind, count, cfg["n_in"], gen)
    table = (torch.rand(enc.num_parameters(), device="cuda", generator=gen) - 0.5).to(enc.parameter_dtype())
    g = torch.randn(count, enc.num_output_channels(), device="cuda", generator=gen)
    size = ctypes.c_size_t()
    check(lib.qmlp_encoding_adjoint_memory(enc._handle, count, 2, ctypes.byref(size)))
    results = []
    for call, fill, adj in ((lib.qmlp_encoding_adjoint_in, 0.0, g), (lib.qmlp_encoding_adjoint_overwriting, float("nan"), g),
                            (lib.qmlp_encoding_adjoint_overwriting, float("nan"), torch.zeros_like(g))):
        memory = torch.full((size.value,), 255, dtype=torch.uint8, device="cuda")
        out = torch.full((enc.num_parameters(),), fill, device="cuda")
        check(call(enc._handle, desc(x), desc(adj), desc(x), current_stream(x.device), desc(table), desc(out), 2, memory.data_ptr()))
        results.append(out)
    assert float(results[0].abs().sum()) > 0 and float(results[2].abs().sum()) == 0
    assert_same(kind, results[1], results[0], g)
    # against float atomics
    expected = torch.zeros_like(results[0])
    check(lib.qmlp_encoding_adjoint(enc._handle, desc(x), desc(g), desc(x), current_stream(x.device), desc(table), desc(expected), 2))
    assert_same(kind, results[0], expected, g)
    with pytest.raises(qmlp.QmlpError, match="asked to overwrite"):
        check(lib.qmlp_encoding_adjoint_overwriting(enc._handle, desc(x), desc(g), desc(x), current_stream(x.device), desc(table),
                                                    desc(expected), 2, None))


@pytest.mark.parametrize("precision", ["half", "float"])
@pytest.mark.parametrize("count", [70001, 1 << 16])
@pytest.mark.parametrize("second", [False, True])
def test_network(precision, count, second):
    """A network behind one grid, whose input gradients are written as well, or behind two encodings."""
    first = grid(9, 2, 15, precision)
    cfg = {"num_inputs": 3, "num_outputs": 2, "activation_specification": ["qmlp/builtin-activations.json"],
           "encodings": [first] + ([grid(2, 2, 12, precision)] if second else []),
           "network": [{"n_out": 32, "bias": False, "activation": "relu"}, {"n_out": 2, "bias": False, "activation": "identity"}]}
    warm_cache(cfg)
    net = qmlp.Network(json.dumps(cfg))
    gen = torch.Generator(device="cuda").manual_seed(7)
    x = points_of("outside", count, 3, gen)
    g = torch.randn(count, 2, device="cuda", generator=gen)
    params = (torch.rand(net.num_network_parameters(), device="cuda", generator=gen) - 0.5).to(torch.float16)
    check(lib.qmlp_network_set_parameter(net._handle, desc(params), QMLP_INFERENCE))
    tables = []
    for i in range(len(cfg["encodings"])):
        tables.append((torch.rand(net.encoding(i).num_parameters(), device="cuda", generator=gen) - 0.5).to(net.encoding(i).parameter_dtype()))
        net.encoding(i).set_parameter(tables[-1])
    stream, size, flags = current_stream(x.device), ctypes.c_size_t(), 5
    mask, yes = ctypes.c_int(), ctypes.c_int()
    check(lib.qmlp_network_overwritable_gradients(net._handle, count, flags, None, ctypes.byref(mask)))
    check(lib.qmlp_network_overwritable_tables(net._handle, count, flags, ctypes.byref(yes)))
    assert yes.value == 1 and mask.value == (0 if second else 1)
    out = torch.empty(count, 2, device="cuda")
    results = []
    for overwrite in (0, mask.value | 4):
        check(lib.qmlp_network_forward_memory(net._handle, count, flags, ctypes.byref(size)))
        forward = torch.empty(size.value, dtype=torch.uint8, device="cuda")
        check(lib.qmlp_network_adjoint_memory(net._handle, count, flags, ctypes.byref(size)))
        scratch = torch.full((size.value,), 255, dtype=torch.uint8, device="cuda")
        check(lib.qmlp_network_forward(net._handle, desc(x), desc(out), forward.data_ptr(), stream))
        adj_tables = [torch.full(t.shape, float("nan") if overwrite else 0.0, device="cuda") for t in tables]
        for i, t in enumerate(adj_tables):
            net.encoding(i).set_parameter(t, gradients=True)
        adj_x = torch.full_like(x, float("nan") if overwrite & 1 else 0.0)
        check(lib.qmlp_network_adjoint_overwriting(net._handle, desc(x), desc(g), flags, overwrite, desc(adj_x), forward.data_ptr(),
                                                   scratch.data_ptr(), stream))
        results.append((adj_x, adj_tables))
    assert torch.equal(results[0][0], results[1][0]) and float(results[0][0].abs().sum()) > 0
    for added, written in zip(results[0][1], results[1][1]):
        torch.testing.assert_close(written, added, rtol=1e-5, atol=1e-5 * float(added.abs().max()))
    # small batches add with atomics
    check(lib.qmlp_network_overwritable_tables(net._handle, 4096, flags, ctypes.byref(yes)))
    assert yes.value == 0
