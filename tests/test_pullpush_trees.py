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
