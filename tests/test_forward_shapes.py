"""Which shapes of the forward kernel batches behind one table are launched with: a tile per wavefront, but where entries are as wide as half a
line, and never a training pass in slab order with a kernel of four tiles that spills."""
import json

import numpy as np
import pytest
import torch

from helpers import FLAG_ENC, FLAG_INPUT, FLAG_WEIGHTS, Case, random_parameters, warm_cache

pytestmark = pytest.mark.gpu


def grid(dim, features, resolution, precision):
    return {"id": "HashGrid", "start_in": 0, "n_in": dim, "n_levels": 1, "n_features_per_level": features, "log2_hashmap_size": -1,
            "min_resolution": resolution, "max_resolution": resolution, "combination_mode": "concat", "bounding_box_min": [0.0] * dim,
            "bounding_box_size": [1.0] * dim, "parameter_precision": precision}


def configuration(encoding, inputs, **options):
    return {"num_inputs": inputs, "num_outputs": 2, "activation_specification": ["qmlp/builtin-activations.json"], "encodings": [encoding],
            "network": [{"n_out": 32, "bias": True, "activation": "relu"}, {"n_out": 2, "bias": False, "activation": "identity"}],
            "options": options}


def line(child):
    return {"id": "LineIntegration", "start_in": 0, "n_in": 3, "volume": child, "stepsize": 0.2, "blending": "additive"}


# (encoding, inputs, kind of pass, points, one tile per wavefront throughout)
@pytest.mark.parametrize("encoding,inputs,kind,points,narrow", [
    (grid(3, 16, 64, "float"), 3, "inference", 100003, False), (grid(3, 16, 64, "half"), 3, "inference", 100003, True),
    (grid(2, 16, 64, "float"), 2, "inference", 100003, True), (line(grid(3, 4, 32, "half")), 6, "inference", 100003, True),
    (grid(4, 8, 32, "half"), 4, "forward", 1 << 21, False), (grid(4, 8, 32, "half"), 4, "forward", 1 << 20, True),
    (grid(4, 16, 24, "half"), 4, "forward", 1 << 21, True)])
def test_launches_of_a_batch_behind_one_table(encoding, inputs, kind, points, narrow):
    free, pinned = configuration(encoding, inputs), configuration(encoding, inputs, points_per_lane=1, sort_points=0)
    warm_cache(free, pinned)
    cases = [Case(free), Case(pinned)]
    launches = json.loads(cases[0].net.generated_source(kind + "_launches", points))
    print(kind, points, launches, flush=True)
    assert sum(l["tiles"] for l in launches) == -(-points // 64)
    assert all(l["tiles_per_wave"] == 1 for l in launches) == narrow
    if not narrow and kind == "forward":
        assert all(l["scratch_bytes"] == 0 for l in launches)
    rng = np.random.default_rng(inputs)
    params, table = random_parameters(cases[0].oracle, rng), None
    for c in cases:
        c.set_parameters(params)
        table = rng.uniform(-1, 1, c.net.encoding(0).num_parameters()) if table is None else table
        c.set_table(0, table)
    X = rng.uniform(0, 1, (points, inputs)).astype(np.float32)
    flags = FLAG_INPUT | FLAG_WEIGHTS | FLAG_ENC
    a, b = (c.gpu_inference(X) if kind == "inference"
            else c.net.forward_raw(torch.from_numpy(X).cuda(), c.params, c.encoding_parameters(), flags)[0].cpu().numpy() for c in cases)
    assert np.array_equal(a, b)
