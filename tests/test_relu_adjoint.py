"""ReLU's packed adjoint (Activation::adjointOfOutput4, two instructions for two values) where its integer arithmetic could go
wrong: pre-activations that are zero, minus zero, the smallest denormal, infinite or NaN, in every form of the backward kernel."""
import numpy as np
import pytest

from helpers import FLAG_INPUT, FLAG_WEIGHTS, Case, identity_cfg, warm_cache

pytestmark = pytest.mark.gpu

TINY = 2.0 ** -24                       # the smallest positive half
OPTIONS = [{"cooperative_backward": 1}, {"cooperative_backward": 0}, {"cooperative_backward": 0, "recompute_intermediates": 0},
           {"cooperative_backward": 0, "fused_weight_update": 0}]
FINITE = [0.0, 0.25, -0.25, 1.0, -1.0, 3.0, -3.0, 1024.0, -1024.0, 2048.0, -2048.0]
SPECIAL = [np.inf, -np.inf, np.nan, -np.nan]


@pytest.mark.parametrize("options", OPTIONS)
@pytest.mark.parametrize("special", [False, True])
def test_adjoint_of_relu_is_the_adjoint_or_zero(options, special):
    """x = 2^-24 times weights: products of 0.25 round to zero, of -0.25 to minus zero, of 1 to the smallest denormal. The second
    layer hands every unit the same adjoint, so that the units whose pre-activation is positive receive it and all others zero:
    sums of few bits, exact in single precision. Batches whose last tile is not full."""
    cfg = dict(identity_cfg(16, [16, 16], ["relu", "identity"], [False, False]), options=options)
    warm_cache(cfg)
    c = Case(cfg)
    values = np.array((FINITE + SPECIAL if special else FINITE) + [0.5] * 16, dtype=np.float32)[:16]
    first, second = np.zeros((16, 16), np.float32), np.zeros((16, 16), np.float32)
    first[:, 0] = values
    second[0, :] = 1.0
    params = np.zeros(c.oracle.num_parameters, np.float32)
    for layer, w in zip(c.oracle.layers, (first, second)):
        params[layer["w_start"]:layer["w_start"] + 256] = w.ravel()
    c.set_parameters(params)
    for N, x in ((1, TINY), (33, TINY), (70, 1.0), (130, -1.0)):
        X = np.zeros((N, 16), np.float32)
        X[:, 0] = x
        adj = np.zeros((N, 16), np.float32)
        adj[:, 0] = 1.0
        print("relu", options, special, N, x, flush=True)
        out = c.gpu_train(X, adj, FLAG_INPUT | FLAG_WEIGHTS)
        with np.errstate(invalid="ignore"):
            pre = (values * np.float32(x)).astype(np.float16)
        on = np.where(pre > 0, 1.0, 0.0).astype(np.float32)
        start = c.oracle.layers[0]["w_start"]
        assert np.array_equal(out["grads"][start:start + 256].reshape(16, 16)[:, 0], on * np.float32(x) * N)
        if not special:
            expected = np.float16(np.sum(on.astype(np.float64) * values))
            assert np.array_equal(out["adj_x"][:, 0], np.full(N, expected, np.float32))
