"""Temporary memory of networks whose large batches take the cooperative backward kernel: a slice of partial weight gradients per workgroup."""
import json

import pytest

import baseline_configs as bc
import qmlp
from helpers import identity_cfg


# three workgroups per compute unit of a chip of 256 without tables, where a lane holds at most 120 registers over a tile; else two
@pytest.mark.parametrize("widths,bias,per_compute_unit", [([64, 64, 4], False, 3), ([64, 64, 4], True, 2), ([32] * 4 + [4], True, 3)])
def test_slices_of_partial_weight_gradients(widths, bias, per_compute_unit):
    cfg = identity_cfg(16, widths, ["relu"] * (len(widths) - 1) + ["identity"], [bias] * len(widths))
    net = qmlp.Network(json.dumps(cfg))
    slice_bytes = 4 * net.num_network_parameters()
    assert net.adjoint_memory(1000000, 2) == per_compute_unit * 256 * slice_bytes
    assert net.adjoint_memory(65536, 2) == 512 * slice_bytes      # two half tiles of 64 points per wavefront of four
    assert net.adjoint_memory(1000, 2) == 4 * slice_bytes


def test_networks_behind_tables_keep_two_workgroups_per_compute_unit():
    grid = json.loads(json.dumps(bc.CONFIGS[3]["cfg"]))["encodings"][0]
    cfg = dict(identity_cfg(3, [64, 64, 4], ["relu", "relu", "identity"], [False] * 3), encodings=[grid])
    net = qmlp.Network(json.dumps(cfg))
    assert net.adjoint_memory(1000000, 2) == 512 * 4 * net.num_network_parameters()
