"""Rows that the backward kernels read a group of tiles ahead, without branches for lanes: numbers of channels of which a lane's four are all, some or
none in a row, rows with gaps, columns that are not next to each other, batches whose last points are repeated for lanes without one."""
import numpy as np
import pytest
import torch

from helpers import FLAG_INPUT, FLAG_WEIGHTS, Case, check_gradients, identity_cfg, random_parameters, warm_cache

pytestmark = pytest.mark.gpu


def laid_out(values, layout):
    """A tensor of these values: rows side by side, rows with a gap (of 4 and of 3 floats), channels apart from each other."""
    n, c = values.shape
    x = torch.from_numpy(values).cuda()
    if layout == "dense":
        return x
    if layout == "columns":
        return x.t().contiguous().t()
    gap = {"gap4": 4, "gap3": 3}[layout]
    wide = torch.full((n, c + gap), float("nan"), device="cuda")
    wide[:, :c] = x
    return wide[:, :c]


@pytest.mark.parametrize("n_in,n_out", [(1, 1), (3, 2), (4, 4), (5, 3), (8, 8), (16, 16), (17, 20), (20, 7), (32, 33)])
def test_rows_of_any_layout_give_the_same_gradients(n_in, n_out):
    """The kernel that does not cooperate reads the same rows: the same bits in the input gradients, the same sums in another order."""
    base = identity_cfg(n_in, [48, 32, n_out], ["relu", "celu", "identity"], [True, False, True])
    on, off = dict(base, options={"cooperative_backward": 1}), dict(base, options={"cooperative_backward": 0})
    warm_cache(on, off)
    cases = [Case(on), Case(off)]
    rng = np.random.default_rng(n_in * 64 + n_out)
    params = random_parameters(cases[0].oracle, rng)
    for c in cases:
        c.set_parameters(params)
    assert "CooperativeLayer<" in cases[0].net.generated_source("backward_cooperative", 3)
    for N in (1, 33, 200, 70001):
        X, adj = rng.uniform(-1, 1, (N, n_in)).astype(np.float32), rng.uniform(-1, 1, (N, n_out)).astype(np.float32)
        reference = cases[1].gpu_train(X, adj, FLAG_INPUT | FLAG_WEIGHTS)
        scale = float(np.abs(reference["grads"]).max())
        for layout in ("dense", "gap4", "gap3", "columns"):
            print("rows", n_in, n_out, N, layout, flush=True)
            c = cases[0]
            x, a = laid_out(X, layout), laid_out(adj, layout)
            out, tmp = c.net.forward_raw(x, c.params, [None], FLAG_INPUT | FLAG_WEIGHTS)
            adj_x, grads, _ = c.net.adjoint_raw(x, a, FLAG_INPUT | FLAG_WEIGHTS, tmp, c.params, [None])
            assert np.array_equal(out.cpu().numpy(), reference["out"])
            assert np.array_equal(adj_x.cpu().numpy(), reference["adj_x"])
            np.testing.assert_allclose(grads.cpu().numpy() / scale, reference["grads"] / scale, rtol=1e-3, atol=1e-5)


@pytest.mark.parametrize("options", [{"cooperative_backward": 0}, {"cooperative_backward": 0, "recompute_intermediates": 0},
                                     {"cooperative_backward": 0, "fused_weight_update": 0}])
@pytest.mark.parametrize("n_out", [1, 2, 3, 4, 8, 20])
def test_rows_of_any_layout_in_the_other_backward_kernels(options, n_out):
    """Rows in any layout hold the same numbers: the same bits in the same kernel."""
    cfg = dict(identity_cfg(6, [32, 16, n_out], ["relu", "sine", "identity"], [True, False, True]), options=options)
    warm_cache(cfg)
    c = Case(cfg)
    rng = np.random.default_rng(n_out)
    c.set_parameters(random_parameters(c.oracle, rng))
    for N in (1, 65, 200, 9001):
        X, adj = rng.uniform(-1, 1, (N, 6)).astype(np.float32), rng.uniform(-1, 1, (N, n_out)).astype(np.float32)
        reference = c.gpu_train(X, adj, FLAG_INPUT | FLAG_WEIGHTS)
        if N == 200:
            check_gradients(c, X, adj, FLAG_INPUT | FLAG_WEIGHTS, reference, kinks=True)
        for layout in ("gap4", "gap3", "columns"):
            print("rows", options, n_out, N, layout, flush=True)
            x, a = laid_out(X, layout), laid_out(adj, layout)
            _, tmp = c.net.forward_raw(x, c.params, [None], FLAG_INPUT | FLAG_WEIGHTS)
            adj_x, grads, _ = c.net.adjoint_raw(x, a, FLAG_INPUT | FLAG_WEIGHTS, tmp, c.params, [None])
            assert np.array_equal(adj_x.cpu().numpy(), reference["adj_x"]) and np.array_equal(grads.cpu().numpy(), reference["grads"])
