"""The backward kernel whose workgroups share the gradient tiles (options.cooperative_backward, kernels/
network_backward_cooperative.h) against the kernels it replaces and the oracles."""
import numpy as np
import pytest

from helpers import FLAG_ENC, FLAG_INPUT, FLAG_WEIGHTS, Case, check_gradients, identity_cfg, random_parameters, warm_cache

pytestmark = pytest.mark.gpu

# one layer; tiles that do not divide among the wavefronts (3, 5, 7 of them); many small layers; workgroups of 8 wavefronts
# (96 wide), of 4 with 512 registers (128 wide); biases, per-channel widths that need padding
NETWORKS = [
    (3, [5], ["identity"], [True]),
    (7, [48, 48, 3], ["celu", "relu", "identity"], [True, False, True]),
    (16, [80, 112, 16], ["relu", "sine", "identity"], [False, True, False]),
    (5, [32] * 6 + [2], ["relu"] * 6 + ["identity"], [True] * 7),
    (4, [128, 64, 48, 4], ["sine", "sine", "celu", "identity"], [True] * 4),
    (16, [64] * 4 + [4], ["relu"] * 4 + ["identity"], [False] * 5),
    (20, [96] * 3 + [7], ["relu", "celu", "relu", "relu"], [True] * 4),
    (16, [128, 128, 33], ["relu", "relu", "identity"], [False, True, True]),
]


@pytest.mark.parametrize("n_in,widths,acts,biases", NETWORKS)
def test_cooperative_backward_matches_the_stored_intermediates_and_the_oracle(n_in, widths, acts, biases):
    """Same operations forward and for the input gradients: the same bits. The weight gradients are the same products
    summed in another order. Batches around the 32 points of a wavefront, the tile of a workgroup and one pass of the
    grid, a single point, and strided rows."""
    base = identity_cfg(n_in, widths, acts, biases)
    on, off = dict(base, options={"cooperative_backward": 1}), dict(base, options={"cooperative_backward": 0})
    warm_cache(on, off)
    cases = [Case(on), Case(off)]
    rng = np.random.default_rng(len(widths) + n_in)
    params = random_parameters(cases[0].oracle, rng)
    for c in cases:
        c.set_parameters(params)
    assert "CooperativeLayer<" in cases[0].net.generated_source("backward_cooperative", 3)
    for N in (1, 31, 33, 129, 257, 4099, 66001):
        X = rng.uniform(-1, 1, (N, n_in)).astype(np.float32)
        adj = (rng.uniform(-1, 1, (N, widths[-1])) / np.sqrt(N)).astype(np.float32)
        for flags in (FLAG_WEIGHTS, FLAG_INPUT | FLAG_WEIGHTS):
            print("cooperative", n_in, widths, N, flags, flush=True)
            a, b = (c.gpu_train(X, adj, flags) for c in cases)
            assert np.array_equal(a["out"], b["out"])
            if flags & FLAG_INPUT:
                assert np.array_equal(a["adj_x"], b["adj_x"])
            scale = float(np.abs(b["grads"]).max())
            np.testing.assert_allclose(a["grads"] / scale, b["grads"] / scale, rtol=1e-3, atol=1e-5)
        if N == 257:
            check_gradients(cases[0], X, adj, FLAG_INPUT | FLAG_WEIGHTS, a, kinks=True)


def test_cooperative_backward_behind_grids_and_beside_an_identity():
    """The encoded input from the forward memory, the adjoint of the encoded rows for the kernels of the gradient slices,
    and the identity's share of the input gradients."""
    grid = {"id": "HashGrid", "start_in": 1, "n_in": 2, "n_levels": 6, "n_features_per_level": 2, "log2_hashmap_size": 10,
            "min_resolution": 4, "max_resolution": 64, "combination_mode": "concat", "bounding_box_min": [0.0, 0.0],
            "bounding_box_size": [1.0, 1.0], "parameter_precision": "half"}
    base = {"num_inputs": 3, "num_outputs": 3, "activation_specification": ["qmlp/builtin-activations.json"],
            "encodings": [{"id": "Identity", "start_in": 0, "n_in": 3}, grid],
            "network": [{"n_out": 64, "bias": True, "activation": "celu"}, {"n_out": 64, "bias": False, "activation": "relu"},
                        {"n_out": 3, "bias": True, "activation": "identity"}]}
    on = dict(base, options={"cooperative_backward": 1, "slice_gradients": 1})
    off = dict(base, options={"cooperative_backward": 0, "slice_gradients": 1})
    warm_cache(on, off)
    cases = [Case(on), Case(off)]
    rng = np.random.default_rng(3)
    params = random_parameters(cases[0].oracle, rng)
    table = rng.uniform(-1, 1, cases[0].oracle.encodings[1][1].n_params)
    for c in cases:
        c.set_parameters(params)
        c.set_table(1, table)
    for N in (50, 1000, 9001):
        X = rng.uniform(0, 1, (N, 3)).astype(np.float32)
        adj = (rng.uniform(-1, 1, (N, 3)) / 16).astype(np.float32)
        flags = FLAG_INPUT | FLAG_WEIGHTS | FLAG_ENC
        print("cooperative grid", N, flush=True)
        a, b = (c.gpu_train(X, adj, flags) for c in cases)
        assert np.array_equal(a["out"], b["out"]) and np.array_equal(a["adj_x"], b["adj_x"])
        for key, x, y in (("grads", a["grads"], b["grads"]), ("table", a["table_grads"][1], b["table_grads"][1])):
            scale = float(np.abs(y).max())
            np.testing.assert_allclose(x / scale, y / scale, rtol=1e-3, atol=1e-5, err_msg=key)
