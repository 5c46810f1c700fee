"""Input gradients of batches whose table gradients go by slices: computed beside the records or by workgroups of their own, from the
entries of all corners or from stored derivatives, for one level and several, at every number of points per workgroup; against the pass
without temporary memory (float atomics), which computes them in the same order of operations, and its time against that pass's."""
import json

import pytest
import torch

import qmlp
from helpers import require_gpu, warm_cache
from qmlp._lib import check, lib
from qmlp.classes import current_stream, desc
from test_gradient_exceptions import adjoint_call, check_sums, time_of
from test_overwritten_tables import grid

pytestmark = pytest.mark.gpu

GRIDS = {"one, many values": grid(1, 8, -1, "half", 4, (20, 20)), "one": grid(1, 2, 18, "float", 3, (300, 300)), "two": grid(2, 2, 16, "float", 2, (9, 500)),
         "nine, half": grid(9, 2, 14, "half", 3), "eight of four floats": grid(8, 4, 14, "float", 3), "sixteen": grid(16, 1, 13, "float", 3)}


@pytest.mark.parametrize("name", GRIDS)
@pytest.mark.parametrize("count", [(1 << 16) + 1, 100003, (1 << 17) + 63, 300001])   # 128 to 1024 points per workgroup
def test_from_entries(name, count):
    cfg = GRIDS[name]
    require_gpu(cfg, (3,))
    enc = qmlp.Encoding(json.dumps(cfg))
    print("input gradients from entries", name, count, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(count)
    x = torch.rand(count, cfg["n_in"], device="cuda", generator=gen)
    x[::101] = 1.0 + 0.5 / cfg["max_resolution"] * x[::101]      # some outside, within a cell of the border
    table = (torch.rand(enc.num_parameters(), device="cuda", generator=gen) - 0.5).to(enc.parameter_dtype())
    g = torch.randn(count, enc.num_output_channels(), device="cuda", generator=gen)
    expected, tables = torch.zeros_like(x), torch.zeros(enc.num_parameters(), device="cuda")
    check(lib.qmlp_encoding_adjoint(enc._handle, desc(x), desc(g), desc(expected), current_stream(x.device), desc(table), desc(tables), 3))
    got = torch.zeros_like(x)
    run, tables = adjoint_call(enc, x, table, g, mode=3, adj_x=got)
    run()
    # (the products of a level are those of the other pass; what a compiler contracts of them may differ: a few roundings of the largest)
    torch.testing.assert_close(got, expected, rtol=1e-5, atol=1e-5 * float(expected.abs().max()))
    check_sums(enc, cfg, x, g, tables)


@pytest.mark.parametrize("name", GRIDS)
@pytest.mark.parametrize("count", [1 << 16, 100003, 270001])
def test_from_stored_derivatives(name, count):
    """A network keeps the derivatives of its encoded features where they are few (options.input_derivatives)."""
    cfg = {"num_inputs": GRIDS[name]["n_in"], "num_outputs": 1, "activation_specification": ["qmlp/builtin-activations.json"], "encodings": [GRIDS[name]],
           "network": [{"n_out": 16, "bias": False, "activation": "relu"}, {"n_out": 1, "bias": False, "activation": "identity"}]}
    cfgs = [dict(cfg, options=o) for o in ({"sort_training": False}, {"sort_training": False, "input_derivatives": 0}, {"sort_training": False, "slice_gradients": 0})]
    warm_cache(*cfgs)
    print("input gradients of a network", name, count, flush=True)
    results = []
    for c in cfgs:
        net = qmlp.Network(json.dumps(c))
        gen = torch.Generator(device="cuda").manual_seed(count)
        x = torch.rand(count, net.channels_in(), device="cuda", generator=gen)
        params = (torch.rand(net.num_network_parameters(), device="cuda", generator=gen) - 0.5).to(torch.float16)
        table = (torch.rand(net.encoding(0).num_parameters(), device="cuda", generator=gen) - 0.5).to(net.encoding(0).parameter_dtype())
        adj = torch.randn(count, 1, device="cuda", generator=gen)
        _, tmp = net.forward_raw(x, params, [table], 5)
        results.append(net.adjoint_raw(x, adj, 5, tmp, params, [table])[0])
    largest = float(results[2].abs().max())
    assert largest > 0
    # from entries: the same operations as the backward kernel's; from derivatives in the precision of the table: 2^-11 each of halves
    torch.testing.assert_close(results[1], results[2], rtol=1e-5, atol=1e-5 * largest)
    torch.testing.assert_close(results[0], results[2], rtol=2e-3, atol=(1e-3 if GRIDS[name]["parameter_precision"] == "half" else 1e-5) * largest)


def test_slices_with_input_gradients_are_not_slower_than_atomics():
    """16 levels, 2^15 points: left to one workgroup per region of 1024 points, the entries of all corners were gathered by 32 of 256
    compute units, and the pass by slices took longer (177 us) than the pass with atomics (150 us; by slices 89 us now)."""
    cfg = grid(16, 2, 19, "float", 3, (16, 4096))
    require_gpu(cfg, (3,))
    enc = qmlp.Encoding(json.dumps(cfg))
    gen = torch.Generator(device="cuda").manual_seed(1)
    x = torch.rand(1 << 15, 3, device="cuda", generator=gen)
    table = torch.rand(enc.num_parameters(), device="cuda", generator=gen) - 0.5
    g = torch.randn(x.shape[0], enc.num_output_channels(), device="cuda", generator=gen)
    by_slices = time_of(adjoint_call(enc, x, table, g, mode=3)[0])
    adj_x, out = torch.zeros_like(x), torch.zeros(enc.num_parameters(), device="cuda")
    descs = [desc(t) for t in (x, g, adj_x, table, out)]
    with_atomics = time_of(lambda: check(lib.qmlp_encoding_adjoint(enc._handle, descs[0], descs[1], descs[2], current_stream(x.device),
                                                                   descs[3], descs[4], 3)))
    print("by slices", by_slices, "with atomics", with_atomics, flush=True)
    assert by_slices < with_atomics
