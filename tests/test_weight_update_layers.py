"""The weight gradients of the layers of a small batch in one launch: the bits of a launch per layer (which
options.parallel_weight_update asks for)."""
import numpy as np
import pytest

from helpers import FLAG_INPUT, FLAG_WEIGHTS, Case, identity_cfg, random_parameters, warm_cache

pytestmark = pytest.mark.gpu

# layers that split into several blocks of tiles, odd numbers of tiles, biases on some of the layers
NETWORKS = [(16, [64] * 4 + [4], [False] * 5), (5, [128, 96, 48, 80, 20], [True, False, True, False, True])]


@pytest.mark.parametrize("n_in,widths,biases", NETWORKS)
def test_all_layers_in_one_launch(n_in, widths, biases):
    base = identity_cfg(n_in, widths, ["relu"] * (len(widths) - 1) + ["identity"], biases)
    together, apart = (dict(base, options={"cooperative_backward": 0, "parallel_weight_update": p}) for p in (False, True))
    warm_cache(together, apart)
    cases = [Case(together), Case(apart)]
    rng = np.random.default_rng(1)
    params = random_parameters(cases[0].oracle, rng)
    for c in cases:
        c.set_parameters(params)
    for n in (1, 64, 65, 1000, 8191, 70001):
        x = rng.uniform(-1, 1, (n, n_in)).astype(np.float32)
        adj = (rng.uniform(-1, 1, (n, widths[-1])) / np.sqrt(n)).astype(np.float32)
        a, b = (c.gpu_train(x, adj, FLAG_INPUT | FLAG_WEIGHTS) for c in cases)
        assert np.abs(a["grads"]).max() > 0 and np.array_equal(a["grads"], b["grads"]), n
