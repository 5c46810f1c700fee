"""The kernels for small batches, whose wavefronts share the grid levels of a tile. Forward: the same bits as the shapes with
a tile per wavefront, for the results and for what the training pass leaves to the adjoint pass. Backward: the same
gradients but for rounding."""
import json

import pytest
import torch

import qmlp
from helpers import require_gpu, warm_cache
from qmlp._lib import check, lib
from qmlp.classes import current_stream, desc

pytestmark = pytest.mark.gpu


def grid(levels, features, start, mode="concat", precision="half"):
    return {"id": "HashGrid", "start_in": start, "n_in": 2, "n_levels": levels, "n_features_per_level": features,
            "log2_hashmap_size": 10, "min_resolution": 4, "max_resolution": 100, "combination_mode": mode,
            "bounding_box_min": [0.0, 0.0], "bounding_box_size": [1.0, 1.0], "parameter_precision": precision}


def spec(*encodings, slices=1):
    return {"num_inputs": 3, "num_outputs": 3, "activation_specification": ["qmlp/builtin-activations.json"],
            "encodings": list(encodings), "options": {"slice_gradients": slices},
            "network": [{"n_out": 32, "bias": True, "activation": "relu"}, {"n_out": 3, "bias": False, "activation": "identity"}]}


IDENTITY = {"id": "Identity", "start_in": 1, "n_in": 2}
# 8 wavefronts (levels that do not divide among them), 4 wavefronts, grids without levels of their own beside them
SPECS = [spec(IDENTITY, grid(9, 2, 0)), spec(grid(5, 1, 1, precision="float"), grid(6, 2, 0, "add")), spec(grid(12, 4, 0))]


@pytest.mark.parametrize("cfg", SPECS)
def test_small_batches_give_the_bits_of_large_ones(cfg):
    warm_cache(cfg)
    net = qmlp.Network(json.dumps(cfg))
    assert any(s["shape"] == "shared" for s in json.loads(net.generated_source("shapes")))
    gen = torch.Generator(device="cuda").manual_seed(5)
    rand = lambda *shape: torch.rand(shape, device="cuda", generator=gen)  # noqa: E731
    x, g = rand(40000, 3) * 1.2 - 0.1, rand(40000, 3) - 0.5
    params = (rand(net.num_network_parameters()) - 0.5).half()
    tables = [(rand(net.encoding(i).num_parameters()) - 0.5).to(net.encoding(i).parameter_dtype())
              if net.encoding(i).has_parameters() else None for i in range(len(cfg["encodings"]))]

    def train(n):
        out, memory = net.forward_raw(x[:n], params, tables, 7)
        adj_x, _, _ = net.adjoint_raw(x[:n], g[:n], 7, memory, params, tables)
        return out, adj_x

    large = net.inference(x, params, tables)
    large_out, large_adj = train(len(x))
    for n in (1, 63, 65, 1000, 448 * 64, 448 * 64 + 1):
        assert torch.equal(net.inference(x[:n], params, tables), large[:n]), n
        out, adj_x = train(n)
        assert torch.equal(out, large_out[:n]) and torch.equal(adj_x, large_adj[:n]), n


# three levels in no wavefront, levels added up and many features stay with the first wavefront
BACKWARD = [(IDENTITY, grid(9, 2, 0)), (grid(5, 1, 1, precision="float"), grid(6, 2, 0, "add")), (grid(4, 4, 0), grid(4, 3, 1))]


@pytest.mark.parametrize("encodings", BACKWARD)
@pytest.mark.parametrize("flags", [1, 4, 6, 7])
def test_small_batches_are_differentiated_like_large_ones(encodings, flags):
    cfg, sliced = spec(*encodings, slices=0), spec(*encodings, slices=1)
    warm_cache(cfg, sliced)
    gen = torch.Generator(device="cuda").manual_seed(5)
    rand = lambda *shape: torch.rand(shape, device="cuda", generator=gen)  # noqa: E731
    x, g = rand(20000, 3) * 1.2 - 0.1, rand(20000, 3) - 0.5
    nets = [qmlp.Network(json.dumps(c)) for c in (cfg, sliced)]
    params = (rand(nets[0].num_network_parameters()) - 0.5).half()
    tables = [(rand(nets[0].encoding(i).num_parameters()) - 0.5).to(nets[0].encoding(i).parameter_dtype())
              if nets[0].encoding(i).has_parameters() else None for i in range(len(encodings))]

    def train(net, n):
        _, memory = net.forward_raw(x[:n], params, tables, flags)
        return net.adjoint_raw(x[:n], g[:n], flags, memory, params, tables)

    large, _, _ = train(nets[0], len(x))
    for n in (1, 63, 65, 1000, 256 * 64, 256 * 64 + 1):
        adj_x, weights, adj_tables = train(nets[0], n)
        if flags & 1:
            # (the same operations, multiplications and additions contracted differently here and there)
            torch.testing.assert_close(adj_x, large[:n], rtol=1e-5, atol=1e-6 * float(large.abs().max()))
        _, expected_weights, expected_tables = train(nets[1], n)
        pairs = [(weights, expected_weights)] if flags & 2 else []
        pairs += [(a, b) for a, b in zip(adj_tables, expected_tables) if a is not None] if flags & 4 else []
        for a, b in pairs:
            assert float(b.abs().max()) > 0
            torch.testing.assert_close(a, b, rtol=1e-3, atol=1e-4 * float(b.abs().max()))


@pytest.mark.parametrize("encoding", [grid(9, 2, 0), grid(5, 1, 1, precision="float"), grid(4, 4, 0)])
def test_standalone_adjoint_of_small_batches(encoding):
    """Against a batch that is too large for the kernel, whose further rows have no adjoint."""
    require_gpu(encoding, (1, 2, 3))
    enc = qmlp.Encoding(json.dumps(encoding))
    gen = torch.Generator(device="cuda").manual_seed(7)
    x = torch.rand((20000, 3), device="cuda", generator=gen) * 1.02 - 0.01
    g = torch.rand((20000, enc.num_output_channels()), device="cuda", generator=gen) - 0.5
    table = (torch.rand(enc.num_parameters(), device="cuda", generator=gen) - 0.5).to(enc.parameter_dtype())

    def adjoint(x, g, flags):
        adj_x, adj_table = torch.ones_like(x), torch.zeros(table.shape, device="cuda")
        check(lib.qmlp_encoding_adjoint(enc._handle, desc(x), desc(g), desc(adj_x), current_stream(x.device), desc(table),
                                        desc(adj_table), flags))
        return adj_x, adj_table

    for n in (1, 63, 65, 1000, 256 * 64):
        front = g.clone()
        front[n:] = 0
        for flags in (1, 2, 3):
            for a, b in zip(adjoint(x[:n], g[:n], flags), adjoint(x, front, flags)):
                b = b[:n] if b.dim() == 2 else b
                torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-5 * float(b.abs().max()))
