"""Which batches of a standalone grid the dies share out by levels, and that they did: from 10 levels on, not at the end of the second step of a workgroup
per compute unit, wide entries behind the first, never where the rows are not free to hold other points' values."""
import json

import pytest
import torch

import qmlp
from helpers import require_gpu
from qmlp import _lib
from qmlp._lib import check, lib
from qmlp.classes import current_stream, desc

pytestmark = pytest.mark.gpu


def grid(levels, features, precision, dims=3):
    return {"id": "HashGrid", "start_in": 0, "n_in": dims, "n_levels": levels, "n_features_per_level": features, "log2_hashmap_size": 19,
            "min_resolution": 16, "max_resolution": 1000, "combination_mode": "concat", "bounding_box_min": [0.0] * dims,
            "bounding_box_size": [1.0] * dims, "parameter_precision": precision}


def kernel(enc, x, rows):
    return _lib.get_string(lib.qmlp_encoding_forward_kernel, enc._handle, desc(x), desc(rows))


# batches in workgroups of 256 points per compute unit, whether they go by levels
@pytest.mark.parametrize("cfg,steps", [
    (grid(16, 2, "float"), {0.5: False, 0.75: True, 1: True, 1.75: True, 1.76: False, 2: False, 2.01: True, 4: True}),
    (grid(8, 8, "float"), {0.75: False, 1.5: False, 4: False}),
    (grid(12, 8, "half"), {0.75: False, 1: False, 1.01: True, 2: False, 3: True}),
    (grid(16, 1, "float"), {1.5: False, 3.99: False, 4: True}),
    (grid(16, 2, "half", 2), {1: False})])   # (a small grid: its tables fit)
def test_batches_by_levels(cfg, steps):
    require_gpu(cfg, (2, 3))
    enc = qmlp.Encoding(json.dumps(cfg))
    step = 256 * torch.cuda.get_device_properties(0).multi_processor_count
    channels, dims = enc.num_output_channels(), enc.max_input_channel() + 1
    table = (torch.rand(enc.num_parameters(), device="cuda", generator=torch.Generator(device="cuda").manual_seed(2)) - 0.5).to(enc.parameter_dtype())
    for factor, by_levels in steps.items():
        points = int(factor * step)
        print(cfg["n_levels"], cfg["n_features_per_level"], points, flush=True)
        x = torch.rand(points, dims, device="cuda") * 1.2 - 0.1
        rows, gaps = torch.zeros(points, channels, device="cuda"), torch.zeros(points, channels + 1, device="cuda")
        assert kernel(enc, x, rows) == ("EncodingLevelsKernel" if by_levels else "EncodingForwardKernel")
        assert kernel(enc, x, gaps) == "EncodingForwardKernel"
        for target in (rows, gaps):
            check(lib.qmlp_encoding_forward(enc._handle, desc(x), desc(target), current_stream(x.device), desc(table)))
        assert torch.equal(rows, gaps[:, :channels])


def test_positions_in_the_rows_or_beside_them():
    cfg = grid(16, 2, "half")
    require_gpu(cfg, (2, 3))
    enc = qmlp.Encoding(json.dumps(cfg))
    points = 60000
    memory = torch.zeros(points * (32 + 3), device="cuda")
    rows = memory[3 * points:].view(points, 32)
    assert kernel(enc, memory[:3 * points].view(points, 3), rows) == "EncodingLevelsKernel"
    assert kernel(enc, memory[:3 * points].view(3, points).t(), rows) == "EncodingLevelsKernel"
    assert kernel(enc, memory[3:3 + 3 * points].view(points, 3), rows) == "EncodingForwardKernel"
    assert kernel(enc, rows[:, :3], rows) == "EncodingForwardKernel"
    assert kernel(enc, torch.zeros(1, 3, device="cuda").expand(points, 3), rows) == "EncodingLevelsKernel"
