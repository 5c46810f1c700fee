"""Bias sums of the cooperative backward kernel: the layers share tiles of 16 columns (kernels/layer_cooperative.h), a column per
tile of output channels of a wavefront."""
import numpy as np
import pytest

from helpers import FLAG_INPUT, FLAG_WEIGHTS, Case, identity_cfg, random_parameters, warm_cache

pytestmark = pytest.mark.gpu


# more than 16 columns; layers with and without a bias in turn; a wavefront with several tiles of output channels
@pytest.mark.parametrize("widths,biases", [([16] * 18 + [3], [True] * 19), ([48, 16, 64, 5], [True, False, True, True]),
                                           ([112, 32, 16], [False, True, False])])
def test_shared_bias_tiles_match_the_kernels_that_sum_by_themselves(widths, biases):
    """The same products summed in another order: single-precision sums of halves."""
    base = identity_cfg(6, widths, ["celu"] * (len(widths) - 1) + ["identity"], biases)
    on, off = dict(base, options={"cooperative_backward": 1}), dict(base, options={"cooperative_backward": 0})
    warm_cache(on, off)
    cases = [Case(on), Case(off)]
    rng = np.random.default_rng(len(widths))
    params = random_parameters(cases[0].oracle, rng, 0.4)
    for c in cases:
        c.set_parameters(params)
    assert "CooperativeLayer<" in cases[0].net.generated_source("backward_cooperative", 3)
    for N in (1, 40, 1000, 40001):
        X = rng.uniform(-1, 1, (N, 6)).astype(np.float32)
        adj = rng.uniform(-1, 1, (N, widths[-1])).astype(np.float32)
        print("bias tiles", widths, N, flush=True)
        a, b = (c.gpu_train(X, adj, FLAG_INPUT | FLAG_WEIGHTS) for c in cases)
        assert np.array_equal(a["adj_x"], b["adj_x"])
        for l in cases[0].oracle.layers:
            parts = [slice(l["w_start"], l["w_start"] + l["cin"] * l["cout"])]
            if l["bias"]:
                parts.append(slice(l["b_start"], l["b_start"] + l["cout"]))
            for p in parts:
                scale = max(float(np.abs(b["grads"][p]).max()), 1e-20)
                np.testing.assert_allclose(a["grads"][p] / scale, b["grads"][p] / scale, rtol=1e-3, atol=1e-5)
