"""What a forward kernel does for batches sorted by slab is in the kernels of networks that sort some batch, and in no other."""
import json

import pytest

import baseline_configs as bc
import qmlp
from helpers import identity_cfg


@pytest.mark.parametrize("cfg,sorts", [
    (bc.CONFIGS[5]["cfg"], True),                                                         # a dense 4-D grid beyond the L2
    (dict(bc.CONFIGS[5]["cfg"], options={"sort_points": 0}), False),
    (bc.CONFIGS[2]["cfg"], False),                                                        # 16 levels
    (identity_cfg(3, [16, 1], ["relu", "identity"], [False, False]), False)])
def test_kernels_of_networks_that_never_sort_have_no_code_for_it(cfg, sorts):
    net = qmlp.Network(json.dumps(cfg))
    for kind in ("inference", "forward"):
        assert ("constexpr bool SORTED_BATCHES = %s;" % ("true" if sorts else "false")) in net.generated_source(kind)
