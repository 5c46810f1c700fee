"""Pull-push levels that one launch walks through (trees): tiles with borders of odd sizes at every level, tiles that end inside the
image, fewer levels per launch for many channels, against the CPU oracle at the tolerances of test_pullpush_gpu.py."""
import numpy as np
import pytest
import torch

import pullpush_oracle as ppo
from qmlp import pullpush as qpp
from qmlp.pullpush import pullpush
from test_pullpush_gpu import ADJ_TOL, FWD_TOL, _gpu_or_warm, gpu, make_case  # noqa: F401

pytestmark = pytest.mark.gpu

# 511, 255, 127 ..: odd on every level; 514 x 258: a tile of two pixels at the end; 300 x 515: odd on some; long and narrow; many channels
SHAPES = [(1, 4, 511, 255), (2, 1, 514, 258), (1, 3, 300, 515), (1, 2, 1025, 33), (1, 1, 40, 700), (1, 15, 190, 130), (1, 5, 257, 256)]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("shape", SHAPES)
def test_trees_against_oracle(shape, dtype):
    mask, data, adj = make_case(sum(shape), *shape, dtype)
    print("pullpush trees", shape, dtype, flush=True)
    m64, d64, a64 = (x.astype(np.float64) for x in (mask, data, adj))
    out = pullpush(gpu(mask, dtype), gpu(data, dtype))
    np.testing.assert_allclose(out.cpu().numpy().astype(np.float64), ppo.pullpush(m64, d64), **FWD_TOL[dtype])
    gm, gd = qpp.pullpush_backward(gpu(mask, dtype), gpu(data, dtype), gpu(adj, dtype))
    wm, wd = ppo.pullpush_adjoint(m64, d64, a64)
    np.testing.assert_allclose(gd.cpu().numpy().astype(np.float64), wd, **ADJ_TOL[dtype])
    np.testing.assert_allclose(gm.cpu().numpy().astype(np.float64), wm, **ADJ_TOL[dtype])


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("shape", [(26, 2, 259, 517), (100, 1, 259, 517), (90, 1, 515, 261), (40, 3, 300, 400)])
def test_large_tiles_against_small_ones(shape, dtype):
    """Many images fill the chip with tiles of 32 and 64 pixels, a single one with tiles of 16: the same pixels, of odd sizes and even ones.
    (Single images against the oracle: above.)"""
    print("pullpush tiles", shape, dtype, flush=True)
    mask, data, adj = (gpu(x, dtype) for x in make_case(sum(shape), *shape, dtype))
    out = pullpush(mask, data)
    gm, gd = qpp.pullpush_backward(mask, data, adj)
    for i in (0, 7, shape[0] - 1):
        one = slice(i, i + 1)
        torch.testing.assert_close(out[one], pullpush(mask[one].contiguous(), data[one].contiguous()), **FWD_TOL[dtype])
        om, od = qpp.pullpush_backward(mask[one].contiguous(), data[one].contiguous(), adj[one].contiguous())
        torch.testing.assert_close(gd[one], od, **ADJ_TOL[dtype])
        torch.testing.assert_close(gm[one], om, **ADJ_TOL[dtype])
