"""The counting sort in front of a network (kernels/point_order.h): rows of every number of channels and layout that its loads
tell apart, batches at the ends of its chunks of 4096 points, all points in one slab. A point is evaluated on its own, so
the sorted batch gives the bits of the batch as given."""
import numpy as np
import pytest
import torch

from helpers import require_gpu, warm_cache
from test_gpu_parity import FLAG_ENC, FLAG_INPUT, Case, random_parameters

pytestmark = pytest.mark.gpu


# (grid dimensions, input channels, the grid's first one): rows that move as one vector, element by element, and too wide to wait in LDS
@pytest.mark.parametrize("dims,channels,start", [(2, 2, 0), (3, 3, 0), (3, 4, 1), (2, 4, 2), (2, 5, 3), (3, 12, 7)])
def test_sorted_rows_of_all_layouts_give_the_bits_of_the_order_given(dims, channels, start):
    require_gpu()
    grid = {"id": "HashGrid", "start_in": start, "n_in": dims, "n_levels": 1, "n_features_per_level": 4 if dims == 2 else 2,
            "log2_hashmap_size": -1, "min_resolution": 1000 if dims == 2 else 128, "max_resolution": 1000 if dims == 2 else 128,
            "combination_mode": "concat", "bounding_box_min": [0.0] * dims, "bounding_box_size": [1.0] * dims, "parameter_precision": "half"}
    base = {"num_inputs": channels, "num_outputs": 2, "activation_specification": ["qmlp/builtin-activations.json"],
            "encodings": [{"id": "Identity", "start_in": 0, "n_in": channels}, grid],
            "network": [{"n_out": 2, "bias": False, "activation": "identity"}]}
    specs = [dict(base, options={"sort_points": mode}) for mode in (1, 0)]
    warm_cache(*specs)
    given = []
    rng = np.random.default_rng(4)
    for spec in specs:
        case = Case(spec)
        if not given:
            parameters = random_parameters(case.oracle, rng)
            table = rng.uniform(-1, 1, case.oracle.encodings[1][1].n_params)
        case.set_parameters(parameters)
        case.set_table(1, table)
        given.append(case)

    def outputs(x):
        return [c.net.inference(x, c.params, c.encoding_parameters()) for c in given]

    wide = torch.rand((12289, channels + 3), device="cuda", generator=torch.Generator(device="cuda").manual_seed(5))
    one_slab = wide * 1e-3 + 0.4
    one_slab[::5, start] = float("nan")
    for points in (1, 4095, 4096, 4097, 12289):
        for rows in (wide, one_slab):
            x = rows[:points]
            column = torch.empty((channels, points), device="cuda").t()
            column.copy_(x[:, :channels])
            # dense, at every distance from a multiple of 16 bytes, rows further apart, column by column
            for layout in (x[:, :channels].contiguous(), x[:, 1:1 + channels], x[:, 2:2 + channels], x[:, 3:3 + channels], column):
                a, b = outputs(layout)
                assert torch.equal(torch.nan_to_num(a, nan=7.0), torch.nan_to_num(b, nan=7.0)), (points, layout.stride())
    assert float(a[torch.isfinite(a)].abs().max()) > 0.01


# chunks of 4096 points: 8 dies share them out, of 512 and more a thread of the scan adds up more than it holds
@pytest.mark.parametrize("chunks", [7, 9, 37, 517])
def test_batches_of_many_chunks_give_the_bits_of_the_order_given(chunks):
    require_gpu()
    points = chunks * 4096 - 1001
    base = {"num_inputs": 4, "num_outputs": 2, "activation_specification": ["qmlp/builtin-activations.json"],
            "encodings": [{"id": "HashGrid", "start_in": 0, "n_in": 3, "n_levels": 1, "n_features_per_level": 2, "log2_hashmap_size": -1,
                           "min_resolution": 128, "max_resolution": 128, "combination_mode": "concat", "bounding_box_min": [0.0] * 3,
                           "bounding_box_size": [1.0] * 3, "parameter_precision": "half"}],
            "network": [{"n_out": 2, "bias": False, "activation": "identity"}]}
    specs = [dict(base, options={"sort_points": mode, "slice_gradients": 1}) for mode in (1, 0)]
    warm_cache(*specs)
    rng = np.random.default_rng(chunks)
    x = rng.uniform(0, 1, (points, 4)).astype(np.float32)
    adj = rng.uniform(-1, 1, (points, 2)).astype(np.float32)
    results = []
    for spec in specs:
        case = Case(spec)
        if not results:
            parameters = random_parameters(case.oracle, rng)
            table = rng.uniform(-1, 1, case.oracle.encodings[0][1].n_params)
        case.set_parameters(parameters)
        case.set_table(0, table)
        out = case.net.inference(torch.from_numpy(x).cuda(), case.params, case.encoding_parameters())
        results.append((out, case.gpu_train(x, adj, FLAG_ENC | FLAG_INPUT)["adj_x"]))
    assert torch.equal(results[0][0], results[1][0])
    assert np.array_equal(results[0][1], results[1][1]) and np.abs(results[0][1]).max() > 0.01
