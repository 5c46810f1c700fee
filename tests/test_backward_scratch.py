"""Scratch memory of the backward kernels that read stored intermediates: what goes through it costs their batches up to a fifth of their time."""
import json

import pytest

import qmlp
from helpers import FLAG_ENC, FLAG_INPUT, FLAG_WEIGHTS, identity_cfg, warm_cache

pytestmark = pytest.mark.gpu

STORED = {"cooperative_backward": 0, "recompute_intermediates": 0}


def dense_grid_cfg():
    grid = {"id": "HashGrid", "start_in": 0, "n_in": 4, "n_levels": 1, "n_features_per_level": 8, "log2_hashmap_size": -1, "min_resolution": 32,
            "max_resolution": 32, "combination_mode": "concat", "bounding_box_min": [0.0] * 4, "bounding_box_size": [1.0] * 4,
            "parameter_precision": "half"}
    cfg = identity_cfg(4, [32, 32, 32, 2], ["relu"] * 4, [True] * 4)
    return dict(cfg, encodings=[grid] + cfg["encodings"])


CASES = [
    # the adjoint of an activation: ReLU in several layers, behind a grid, other activations
    (identity_cfg(16, [64] * 4 + [4], ["relu"] * 4 + ["identity"], [False] * 5), FLAG_INPUT | FLAG_WEIGHTS),
    (identity_cfg(16, [64] * 4 + [4], ["sine"] * 4 + ["identity"], [True] * 5), FLAG_INPUT | FLAG_WEIGHTS),
    (dense_grid_cfg(), FLAG_ENC),
    # input gradients of wide rows, added to what the rows hold
    (identity_cfg(128, [64, 64, 64], ["sine", "sine", "identity"], [False] * 3), FLAG_INPUT | FLAG_WEIGHTS),
]


@pytest.mark.parametrize("cfg,flags", CASES)
def test_stored_intermediates_take_no_scratch_memory(cfg, flags):
    cfg = dict(cfg, options=STORED)
    warm_cache(cfg)
    resources = json.loads(qmlp.Network(json.dumps(cfg)).generated_source("backward_resources", flags))
    print(resources, flush=True)
    assert not resources["recompute"] and resources["scratch_bytes"] == 0
