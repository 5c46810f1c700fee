"""Networks behind a grid of one table take one tile per wavefront, and four for whole steps of a training pass in slab order
(FusedNetwork::forwardKernelFor): batches on both sides of the steps, cut into two launches, and small ones."""
import numpy as np
import pytest
import torch

from helpers import FLAG_ENC, FLAG_INPUT, FLAG_WEIGHTS, Case, random_parameters, warm_cache

pytestmark = pytest.mark.gpu


def configuration(dim, features, resolution, log2, options):
    return {"num_inputs": dim, "num_outputs": 2, "activation_specification": ["qmlp/builtin-activations.json"],
            "encodings": [{"id": "HashGrid", "start_in": 0, "n_in": dim, "n_levels": 1, "n_features_per_level": features,
                           "log2_hashmap_size": log2, "min_resolution": resolution, "max_resolution": resolution,
                           "combination_mode": "concat", "bounding_box_min": [0.0] * dim, "bounding_box_size": [1.0] * dim,
                           "parameter_precision": "half"}],
            "network": [{"n_out": 16, "bias": True, "activation": "relu"}, {"n_out": 2, "bias": False, "activation": "identity"}],
            "options": options}


# ordered by slab from 2^19 points on; a table that stays in the L2, never ordered; hashed entries
@pytest.mark.parametrize("dim,features,resolution,log2,sizes", [
    (4, 8, 32, -1, (1, 65, 300007, 1 << 19, (1 << 19) + 1, 700001, (1 << 20) + 30011, 1 << 21, (1 << 22) + 6403)),
    (2, 4, 64, -1, (1, 4097, 300007, 1 << 19)), (3, 2, 128, 12, (63, 70001, 600011))])
def test_shapes_give_the_bits_of_one_tile_per_wavefront(dim, features, resolution, log2, sizes):
    free, pinned = configuration(dim, features, resolution, log2, {}), configuration(dim, features, resolution, log2, {"points_per_lane": 1, "sort_points": 0})
    warm_cache(free, pinned)
    cases = [Case(free), Case(pinned)]
    rng = np.random.default_rng(dim)
    params = random_parameters(cases[0].oracle, rng)
    table = rng.uniform(-1, 1, cases[0].oracle.encodings[0][1].n_params)
    for c in cases:
        c.set_parameters(params)
        c.set_table(0, table)
    for N in sizes:
        print("single table", dim, N, flush=True)
        X = rng.uniform(0, 1, (N, dim)).astype(np.float32)
        outputs = [c.gpu_inference(X) for c in cases]
        assert np.array_equal(outputs[0], outputs[1])
        trained = [c.net.forward_raw(torch.from_numpy(X).cuda(), c.params, c.encoding_parameters(), FLAG_INPUT | FLAG_WEIGHTS | FLAG_ENC)[0] for c in cases]
        assert np.array_equal(trained[0].cpu().numpy(), outputs[1]) and np.array_equal(trained[1].cpu().numpy(), outputs[1])

