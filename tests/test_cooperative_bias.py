"""Bias sums of the cooperative backward kernel: every layer has a tile of its own, a column per tile of output channels of a
wavefront (kernels/layer_cooperative.h)."""
import numpy as np
import pytest

import qmlp_oracle as qo
from helpers import FLAG_INPUT, FLAG_WEIGHTS, Case, identity_cfg, random_parameters, warm_cache

pytestmark = pytest.mark.gpu


# more than 16 tiles of output channels; layers with and without a bias in turn; a wavefront with several tiles of output channels
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


STEEP = {"id": "steep", "forward": "z = x", "adjoint": "adjx = __hmul(__float2half(3000.0f), adjz)"}


@pytest.mark.parametrize("widths,biases", [([32, 48, 5], [True, True, True]), ([16, 16, 64, 3], [True, False, True, True])])
def test_an_adjoint_that_overflows_stays_in_its_layer(widths, biases):
    """One unit of the first layer has an infinite adjoint. The sums of all other layers are finite and those of the other kernel; in its own
    layer a tile's sums are multiplied by ones and zeros, which reaches at most the units 16, 32 .. channels away."""
    base = identity_cfg(6, widths, ["steep"] + ["identity"] * (len(widths) - 1), biases, extra_acts=[STEEP])
    on, off = dict(base, options={"cooperative_backward": 1}), dict(base, options={"cooperative_backward": 0})
    warm_cache(on, off)
    cases = [Case(c, {"steep": qo.BUILTIN_ACTIVATIONS["identity"]}) for c in (on, off)]
    rng = np.random.default_rng(len(widths))
    params = random_parameters(cases[0].oracle, rng, 0.1)
    first, second = cases[0].oracle.layers[:2]
    unit = 5
    into_second = params[second["w_start"]:second["w_start"] + second["cin"] * second["cout"]].reshape(second["cout"], second["cin"])
    into_second[:] = np.float16(0.001) * np.sign(into_second)
    into_second[:, unit] = 256.0
    for c in cases:
        c.set_parameters(params)
    assert "CooperativeLayer<" in cases[0].net.generated_source("backward_cooperative", 3)
    for N in (40, 1000, 40001):
        X = rng.uniform(-1, 1, (N, 6)).astype(np.float32)
        adj = rng.uniform(1, 2, (N, widths[-1])).astype(np.float32)
        print("overflow", widths, N, flush=True)
        a, b = (c.gpu_train(X, adj, FLAG_WEIGHTS)["grads"] for c in cases)
        own = a[first["b_start"]:first["b_start"] + first["cout"]]
        away = np.arange(first["cout"]) % 16 != unit
        assert np.isfinite(own[away]).all() and not np.isfinite(own[unit])
        for l in cases[0].oracle.layers[1:]:
            p = slice(l["w_start"], l["w_start"] + l["cin"] * l["cout"])
            parts = [p] + ([slice(l["b_start"], l["b_start"] + l["cout"])] if l["bias"] else [])
            for p in parts:
                assert np.isfinite(a[p]).all()
                scale = float(np.abs(b[p]).max())
                np.testing.assert_allclose(a[p] / scale, b[p] / scale, rtol=1e-3, atol=1e-5)
