"""The standalone adjoint pass of a grid with temporary memory (records and sums per slice of the table, adjoints in
floats) against the same pass without (float atomics), and the forward pass by groups of levels against whole rows."""
import ctypes
import json

import pytest
import torch

import qmlp
from helpers import require_gpu
from qmlp._lib import check, lib
from qmlp.classes import current_stream, desc

pytestmark = pytest.mark.gpu


def grid(levels, features, log2_size, precision, dims=3):
    return json.dumps({"id": "HashGrid", "start_in": 0, "n_in": dims, "n_levels": levels, "n_features_per_level": features,
                       "log2_hashmap_size": log2_size, "min_resolution": 5, "max_resolution": 200, "combination_mode": "concat",
                       "bounding_box_min": [0.0] * dims, "bounding_box_size": [1.0] * dims, "parameter_precision": precision})


GRIDS = [grid(8, 2, 13, "float"), grid(9, 1, 14, "half"), grid(11, 4, 12, "float", 2)]


def adjoint(enc, x, table, g, flags, with_memory):
    size = ctypes.c_size_t()
    check(lib.qmlp_encoding_adjoint_memory(enc._handle, x.shape[0], flags, ctypes.byref(size)))
    assert (size.value > 0) == (x.shape[0] >= (1 << 14) + (flags & 1))
    memory = torch.empty(max(size.value, 256), dtype=torch.uint8, device="cuda")
    adj_x, adj_table = torch.zeros_like(x), torch.zeros(table.shape, device="cuda")
    check(lib.qmlp_encoding_adjoint_in(enc._handle, desc(x), desc(g), desc(adj_x), current_stream(x.device), desc(table),
                                       desc(adj_table), flags, memory.data_ptr() if with_memory else None))
    return adj_x, adj_table


@pytest.mark.parametrize("cfg", GRIDS)
@pytest.mark.parametrize("points", [(1 << 14) - 1, 1 << 14, 50001])
def test_gradients_by_slices(cfg, points):
    require_gpu(json.loads(cfg), (2, 3))
    enc = qmlp.Encoding(cfg)
    gen = torch.Generator(device="cuda").manual_seed(points)
    x = torch.rand(points, enc.max_input_channel() + 1, device="cuda", generator=gen)
    x[:20] = x[20]                                                    # one cell
    x[points // 2:points // 2 + 40] = 1.0 + 0.01 * x[:40]                # outside of the box
    table = (torch.rand(enc.num_parameters(), device="cuda", generator=gen) - 0.5).to(enc.parameter_dtype())
    g = torch.randn(points, enc.num_output_channels(), device="cuda", generator=gen)
    for flags in (2, 3):
        expected_x, expected = adjoint(enc, x, table, g, flags, False)
        adj_x, adj_table = adjoint(enc, x, table, g, flags, True)
        torch.testing.assert_close(adj_x, expected_x, rtol=1e-5, atol=1e-5 * float(expected_x.abs().max()))
        # (points outside of the box: large weights of both signs that cancel)
        torch.testing.assert_close(adj_table, expected, rtol=1e-4, atol=3e-5 * float(expected.abs().max()))

    # adjoints of very different magnitude: the small ones keep their relative precision
    inside = torch.rand(points, x.shape[1], device="cuda", generator=gen)
    scale = torch.ones(points, 1, device="cuda")
    inside[0] = 0.99
    near = ((inside - inside[0]).abs().max(dim=1).values < 0.3)
    scale[near] = 1e12
    _, expected = adjoint(enc, inside, table, g * scale, 2, False)
    _, adj_table = adjoint(enc, inside, table, g * scale, 2, True)
    small = expected.abs() < 1e4
    assert small.any() and torch.equal(expected == 0, adj_table == 0)
    # Float additions (the expected sums, and those of coarse levels) come in any order: each rounds with a standard deviation of at
    # most 2^-24 / sqrt(3) of the running sum, a random walk that ends within the largest of these sums. Two sums of k terms differ
    # by sqrt(2 k / 3) 2^-24 of that, here by six of these (12 609 terms, sums up to 76: 2.5e-3; 1.9e-4 seen in 20 repetitions).
    corners = enc.hashgrid_corners(inside)[0]
    order = 6 * (2 * int(torch.bincount(corners.flatten()).max()) / 3) ** 0.5 * 2.0 ** -24 * float(expected[small].abs().max())
    torch.testing.assert_close(adj_table[small], expected[small], rtol=1e-4, atol=order)

    # NaN and infinity reach the gradients
    g[7, 0], g[points - 1, 1] = float("nan"), float("inf")
    _, expected = adjoint(enc, inside, table, g, 2, False)
    _, adj_table = adjoint(enc, inside, table, g, 2, True)
    assert not torch.isfinite(adj_table).all() and torch.equal(torch.isfinite(expected), torch.isfinite(adj_table))


@pytest.mark.parametrize("cfg", GRIDS)
def test_forward_by_groups_of_levels_gives_the_same_bits(cfg):
    require_gpu(json.loads(cfg), (2, 3))
    enc = qmlp.Encoding(cfg)
    gen = torch.Generator(device="cuda").manual_seed(1)
    x = torch.rand(3 << 14, enc.max_input_channel() + 1, device="cuda", generator=gen) * 1.2 - 0.1
    table = (torch.rand(enc.num_parameters(), device="cuda", generator=gen) - 0.5).to(enc.parameter_dtype())
    whole = enc.inference_with_parameter(x, table)
    for points in (1, 63, 65, 257, 5000, (3 << 14) - 1):
        assert torch.equal(enc.inference_with_parameter(x[:points], table), whole[:points]), points


@pytest.mark.parametrize("levels, features, precision", [(11, 4, "half"), (16, 2, "half"), (9, 3, "float"), (24, 1, "float"), (16, 8, "half")])
def test_forward_by_levels_gives_the_same_bits(levels, features, precision):
    # tables of 20 to 60 MB: the dies share out the levels of larger batches. Rows with gaps, and positions in the rows' memory, take the
    # kernel of whole rows.
    cfg = json.loads(grid(levels, features, 19, precision))
    cfg["max_resolution"] = 2000
    require_gpu(cfg, (2, 3))
    enc = qmlp.Encoding(json.dumps(cfg))
    gen = torch.Generator(device="cuda").manual_seed(1)
    channels = enc.num_output_channels()
    table = (torch.rand(enc.num_parameters(), device="cuda", generator=gen) - 0.5).to(enc.parameter_dtype())
    for points in ((3 << 14) - 1, 3 << 14, 50001, (7 << 14) + 1, (1 << 17) + 63, (1 << 18) + 65):
        x = torch.rand(points, 4, device="cuda", generator=gen) * 1.2 - 0.1
        padded = torch.zeros(points, channels + 1, device="cuda")
        check(lib.qmlp_encoding_forward(enc._handle, desc(x), desc(padded), current_stream(x.device), desc(table)))
        assert torch.equal(enc.inference_with_parameter(x, table), padded[:, :channels]), points
        if channels > 62 or points < 3 << 14:
            continue   # (rows that are written as they come, and in pieces)
        shared = torch.empty(points, channels, device="cuda")
        shared[:, :3] = x[:, :3]
        check(lib.qmlp_encoding_forward(enc._handle, desc(shared[:, :3]), desc(shared), current_stream(x.device), desc(table)))
        assert torch.equal(shared, padded[:, :channels]), points
