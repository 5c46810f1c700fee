"""Table gradients summed by columns (kernels/grid_gradient_columns.h) where their loops end: runs of points around the 64 of a
tile and the 512 of a workgroup, points on and beyond the upper border of the coordinates that are not sorted, entries of one,
three, four and eight features, rows of four floats and others."""
import json

import numpy as np
import pytest
import torch

import qmlp
from helpers import require_gpu, warm_cache
from test_gpu_parity import FLAG_ENC, FLAG_INPUT, Case, random_parameters

pytestmark = pytest.mark.gpu

# (dimensions, features, resolution, precision, input channels in front of the grid's): tables of 4 MB and more
GRIDS = [(4, 8, 32, "half", 0), (4, 4, 32, "float", 1), (3, 3, 128, "half", 0), (3, 1, 128, "float", 0), (2, 1, 2048, "half", 1)]


@pytest.mark.parametrize("dims,features,resolution,precision,start", GRIDS)
def test_columns_at_the_ends_of_runs_and_on_the_upper_border(dims, features, resolution, precision, start):
    require_gpu()
    grid = {"id": "HashGrid", "start_in": start, "n_in": dims, "n_levels": 1, "n_features_per_level": features,
            "log2_hashmap_size": -1, "min_resolution": resolution, "max_resolution": resolution, "combination_mode": "concat",
            "bounding_box_min": [0.0] * dims, "bounding_box_size": [1.0] * dims, "parameter_precision": precision}
    base = {"num_inputs": start + dims, "num_outputs": 2, "activation_specification": ["qmlp/builtin-activations.json"],
            "encodings": [{"id": "Identity", "start_in": 0, "n_in": 1}, grid],
            "network": [{"n_out": 2, "bias": False, "activation": "identity"}]}
    options = {"columns": {"sort_points": 1, "slice_gradients": 1}, "atomics": {"sort_points": 0, "slice_gradients": 0},
               "records": {"sort_points": 1, "slice_gradients": 1, "column_gradients": 0}}
    warm_cache(*[dict(base, options=o) for o in options.values()])
    cases = {k: Case(dict(base, options=o)) for k, o in options.items()}
    rng = np.random.default_rng(3)
    count = len(random_parameters(cases["columns"].oracle, rng))
    table = rng.uniform(-1, 1, cases["columns"].oracle.encodings[1][1].n_params)
    for c in cases.values():
        c.set_parameters(np.full(count, 0.5))   # with positive adjoints: all terms of a sum are positive
        c.set_table(1, table)
    probe = qmlp.Encoding(json.dumps(grid))
    probe.set_parameter(torch.zeros(probe.num_parameters(), device="cuda", dtype=probe.parameter_dtype()))
    cell = 1.0 / (resolution - 1)
    for points in (1, 63, 65, 513, 1100, 3001, 9001):   # up to one, two, six and eighteen loads of a lane for the largest adjoint
        x = rng.uniform(0, 1, (points, start + dims))
        x[:, start:start + 2] = 0.5 + cell * rng.uniform(-2, 2, (points, 2))      # a few slabs
        for d in range(2, dims):
            border = rng.integers(0, 4, points)
            x[:, start + d] = np.choose(border, [x[:, start + d], 1.0, 1 - 0.5 * cell, 1 + 0.5 * cell])
        x = x.astype(np.float32)
        adj = rng.uniform(0.01, 0.05, (points, 2)).astype(np.float32)
        adj[rng.integers(0, points)] *= 500       # which the scale of the sums has to go by, wherever it lies
        for flags in (FLAG_ENC, FLAG_ENC | FLAG_INPUT):
            got = {k: cases[k].gpu_train(x, adj, flags) for k in ("columns", "atomics")}
            a, b = got["columns"]["table_grads"][1], got["atomics"]["table_grads"][1]
            # k positive terms in any order in single precision: k units of the last place of the sum, and a few for the weights,
            # which the two paths round differently beyond the border; the fixed point of the columns keeps 2^-40 of a term
            corners = probe.hashgrid_corners(torch.from_numpy(x).cuda())[0].cpu().numpy().astype(np.int64).ravel()
            k = int(np.bincount(corners).max())
            error = np.abs(a.astype(np.float64) - b)
            bound = (k + 8) * 2.0 ** -24 * np.abs(b) + k * 2.0 ** -40 * float(adj.max())
            worst = int(np.argmax(error - bound))
            assert b.max() > 0 and (error <= bound).all(), (points, flags, worst, a[worst], b[worst], k)
            if flags & FLAG_INPUT:
                # (the same operations on the same sorted batch; the path with atomics rounds features to halves on the way)
                records = cases["records"].gpu_train(x, adj, flags)
                assert np.array_equal(got["columns"]["adj_x"], records["adj_x"]), (points, flags)
