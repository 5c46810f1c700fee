"""The cooperative backward kernel of networks with wide rows: the rows that are asked for ahead cost registers, the kernel spills, and is still
the one that batches take."""
import json

import numpy as np
import pytest

from helpers import FLAG_INPUT, FLAG_WEIGHTS, Case, identity_cfg, random_parameters, warm_cache

pytestmark = pytest.mark.gpu


# wavefronts of 512 registers, workgroups of 8 wavefronts; rows of eight tiles of channels, and of some that are not full
@pytest.mark.parametrize("n_in,widths,act,bias", [(128, [64, 64, 128], "sine", False), (128, [64, 64, 128], "sine", True),
                                                  (128, [128, 128], "sine", True), (128, [32, 96, 128], "relu", False),
                                                  (128, [64, 64, 64], "relu", True), (113, [48, 97], "celu", True)])
def test_wide_rows_take_the_cooperative_kernel(n_in, widths, act, bias):
    base = identity_cfg(n_in, widths, [act] * (len(widths) - 1) + ["identity"], [bias] * len(widths))
    on, off = dict(base, options={"cooperative_backward": 1}), dict(base, options={"cooperative_backward": 0})
    warm_cache(on, off)
    cases = [Case(on), Case(off)]
    rng = np.random.default_rng(n_in + len(widths))
    params = random_parameters(cases[0].oracle, rng)
    for c in cases:
        c.set_parameters(params)
    for flags in (FLAG_WEIGHTS, FLAG_INPUT | FLAG_WEIGHTS):
        resources = [json.loads(c.net.generated_source("backward_resources", flags)) for c in cases]
        print("wide rows", n_in, widths, resources[0], flush=True)
        assert resources[0]["cooperative"] and not resources[1]["cooperative"]
    for N in (1, 33, 1000, 20011):
        print("wide rows", n_in, widths, N, flush=True)
        X, adj = rng.uniform(-1, 1, (N, n_in)).astype(np.float32), rng.uniform(-1, 1, (N, widths[-1])).astype(np.float32)
        a, b = (c.gpu_train(X, adj, FLAG_INPUT | FLAG_WEIGHTS) for c in cases)
        # the same operations forward and for the input gradients; the products of the weight gradients summed in another order
        assert np.array_equal(a["out"], b["out"]) and np.array_equal(a["adj_x"], b["adj_x"])
        scale = float(np.abs(b["grads"]).max())
        np.testing.assert_allclose(a["grads"] / scale, b["grads"] / scale, rtol=1e-3, atol=1e-5)
