"""Table gradients of points that have no record (GridGradientExceptionsKernel): points outside of the box one by one and in runs, upper
entries in slices far away, both in one list, lists of one part and of many, against sums in double precision; and the time of a batch
with a run of points outside, whose lists a whole chip has to share."""
import ctypes
import json

import numpy as np
import pytest
import torch

import qmlp
from helpers import require_gpu
from qmlp._lib import check, lib
from qmlp.classes import current_stream, desc
from test_overwritten_tables import grid

pytestmark = pytest.mark.gpu


def adjoint_call(enc, x, table, g, mode=2, overwrite=True, adj_x=None):
    """A function that runs one adjoint pass by slices, and the table gradients that it writes, or adds to."""
    size = ctypes.c_size_t()
    check(lib.qmlp_encoding_adjoint_memory(enc._handle, x.shape[0], mode, ctypes.byref(size)))
    assert size.value > 0
    memory = torch.empty(size.value, dtype=torch.uint8, device="cuda")
    out = torch.full((enc.num_parameters(),), float("nan"), device="cuda")
    adj_x = torch.zeros_like(x) if adj_x is None else adj_x
    descs = [desc(x), desc(g), desc(adj_x)]
    stream = current_stream(x.device)

    def run(keep=(x, g, table, adj_x, out, memory)):
        call = lib.qmlp_encoding_adjoint_overwriting if overwrite else lib.qmlp_encoding_adjoint_in
        check(call(enc._handle, descs[0], descs[1], descs[2], stream, desc(table), desc(out), mode, memory.data_ptr()))
    return run, out


def check_sums(enc, cfg, x, g, got):
    """The table gradients of adjoints g at points x against sums in double precision."""
    count, dims, features = x.shape[0], cfg["n_in"], cfg["n_features_per_level"]
    index, weight = enc.hashgrid_corners(x)   # (points, levels, corners)
    index, weight = index.cpu().numpy(), weight.cpu().numpy().astype(np.float64)
    adjoints = g.cpu().numpy().astype(np.float64).reshape(count, cfg["n_levels"], features)
    sums, magnitude, terms = (np.zeros(enc.num_parameters()) for _ in range(3))
    for f in range(features):   # (on the host: atomics of the whole batch on one entry take minutes)
        term = (weight * adjoints[:, :, f, None]).reshape(-1)
        at = (index + f).reshape(-1)
        sums += np.bincount(at, term, sums.size)
        magnitude += np.bincount(at, np.abs(term), sums.size)
        terms += np.bincount(at, minlength=sums.size)
    # Float additions in any order: each rounds by at most 2^-24 of a running sum that stays below the sum of magnitudes; a term is a
    # product of at most dims + 1 rounded factors, taken in another order here. Fixed-point sums are finer than 2^-35 of the largest
    # adjoint each.
    bound = (terms + 2 * dims + 4) * 2.0 ** -24 * magnitude + terms * 2.0 ** -35 * float(g.abs().max()) + 1e-12
    error = np.abs(got.cpu().numpy().astype(np.float64) - sums)
    assert (error <= bound).all(), float((error / bound).max())


def outside(x, beyond):
    """The points moved to just behind the upper border of the first coordinate."""
    y = x.clone()
    y[:, 0] = 1.0 + beyond * x[:, 0]
    return y


GRIDS = [grid(8, 2, 13, "float"), grid(9, 3, 14, "half", 2), grid(8, 2, 16, "float", 2, (100, 20000)), grid(8, 1, 12, "float", 4, (3, 20))]


@pytest.mark.parametrize("cfg", GRIDS)
@pytest.mark.parametrize("count", [(1 << 14) + 77, 3 * (1 << 15) - 1])
@pytest.mark.parametrize("kind", ["one", "spread", "run", "all"])
def test_against_sums_in_double_precision(cfg, count, kind):
    require_gpu(cfg, (2,))
    enc = qmlp.Encoding(json.dumps(cfg))
    dims = cfg["n_in"]
    print("exceptions", cfg["max_resolution"], count, kind, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(count)
    x = torch.rand(count, dims, device="cuda", generator=gen)
    where = {"one": slice(count // 2, count // 2 + 1), "spread": slice(3, None, 5), "run": slice(1000, 1000 + count // 3), "all": slice(None)}[kind]
    x[where] = outside(x[where], 1.0 / cfg["max_resolution"])   # at most a cell of the finest level: weights of at most two
    table = torch.zeros(enc.num_parameters(), device="cuda", dtype=enc.parameter_dtype())
    g = torch.randn(count, enc.num_output_channels(), device="cuda", generator=gen)
    run, got = adjoint_call(enc, x, table, g)
    run()
    check_sums(enc, cfg, x, g, got)


def time_of(run):
    for _ in range(3):
        run()
    times = []
    for _ in range(5):
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        begin.record()
        for _ in range(10):
            run()
        end.record()
        end.synchronize()
        times.append(begin.elapsed_time(end))
    return sorted(times)[2]


def test_a_run_of_points_outside_is_shared_out():
    """16 levels, 2^17 points: 2 048 points outside that lie next to each other add 2^17 pairs of entries with atomics, 25 us of them;
    walked through by a wavefront per region they took 14 times the whole pass of points inside, shared out 0.8 times as long."""
    cfg = grid(16, 2, 19, "float", 3, (16, 4096))
    require_gpu(cfg, (2,))
    enc = qmlp.Encoding(json.dumps(cfg))
    gen = torch.Generator(device="cuda").manual_seed(1)
    x = torch.rand(1 << 17, 3, device="cuda", generator=gen)
    table = torch.zeros(enc.num_parameters(), device="cuda", dtype=enc.parameter_dtype())
    g = torch.randn(x.shape[0], enc.num_output_channels(), device="cuda", generator=gen)
    inside = time_of(adjoint_call(enc, x, table, g)[0])
    x[:2048] = outside(x[:2048], 0.02)
    some = time_of(adjoint_call(enc, x, table, g)[0])
    print("inside", inside, "with a run outside", some, flush=True)
    assert some < 4 * inside
