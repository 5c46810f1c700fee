"""Table gradients of batches whose neighbours are neighbours in space (samples along rays, sorted points, one cell): the records of a
slice then lie in a few long segments, which the slice kernel cuts into parts; and of points spread evenly, in segments of a few
records to some dozens. Batches of up to a thousand regions and of more, parts
that take several rounds, floats too small for the sums, against sums in double precision; and the time of rays."""
import json

import pytest
import torch

import qmlp
from helpers import require_gpu
from test_gradient_exceptions import adjoint_call, check_sums, time_of
from test_overwritten_tables import grid

pytestmark = pytest.mark.gpu

GRIDS = {"many": grid(1, 8, -1, "half", 4, (32, 32)),   # 512 slices: four records to a segment
         "dense": grid(1, 4, -1, "float", 3, (64, 64)),
         "levels": grid(8, 2, 14, "half", 3, (5, 200)), "wide": grid(1, 8, -1, "float", 4, (20, 20))}


def points(kind, count, dims, gen):
    x = torch.rand(count, dims, device="cuda", generator=gen)
    if kind == "even":
        return x
    if kind == "sorted":
        return x[torch.argsort(x[:, 0])].contiguous()
    if kind == "cell":
        return 0.31 + 1e-3 * x
    if kind == "some":    # even, but for a run of neighbours
        x[5000:12000] = 0.31 + 1e-3 * x[5000:12000]
        return x
    rays = (count + 255) // 256
    begin, end = (torch.rand(rays, 1, dims, device="cuda", generator=gen) for _ in range(2))
    t = torch.linspace(0, 1, 256, device="cuda")[None, :, None]
    return (begin + t * (end - begin)).reshape(-1, dims)[:count].contiguous()


@pytest.mark.parametrize("name,count", [("dense", 1 << 16), ("dense", (1 << 20) + 12345), ("levels", 70001), ("levels", 1 << 14),
                                        ("wide", 150001), ("many", 1 << 16), ("many", 600001)])
@pytest.mark.parametrize("kind", ["even", "rays", "sorted", "cell", "some"])
@pytest.mark.parametrize("span", [0, 60])
def test_against_sums_in_double_precision(name, count, kind, span):
    cfg = GRIDS[name]
    require_gpu(cfg, (2,))
    enc = qmlp.Encoding(json.dumps(cfg))
    print("segments", name, count, kind, span, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(count + span)
    x = points(kind, count, cfg["n_in"], gen)
    table = torch.zeros(enc.num_parameters(), device="cuda", dtype=enc.parameter_dtype())
    g = torch.randn(count, enc.num_output_channels(), device="cuda", generator=gen)
    g = g * torch.exp2(-torch.randint(0, span + 1, g.shape, device="cuda", generator=gen).float())
    run, got = adjoint_call(enc, x, table, g)
    run()
    check_sums(enc, cfg, x, g, got)
    # added to gradients that are there: as much again (the last rounding is one of those that the bound counts)
    run, twice = adjoint_call(enc, x, table, g, overwrite=False)
    twice.copy_(got)
    run()
    check_sums(enc, cfg, x, g, twice - got)


def test_samples_along_rays_take_as_long_as_points_at_random():
    """One level of 64^3 nodes, 2^17 samples: each slice is met by a few rays, in segments of up to hundreds of records. Left to the eight or
    sixteen lanes that take a segment they took three times as long as points at random, shared out 1.1 times."""
    cfg = GRIDS["dense"]
    require_gpu(cfg, (2,))
    enc = qmlp.Encoding(json.dumps(cfg))
    gen = torch.Generator(device="cuda").manual_seed(1)
    table = torch.zeros(enc.num_parameters(), device="cuda")
    g = torch.randn(1 << 17, enc.num_output_channels(), device="cuda", generator=gen)
    times = []
    for x in (torch.rand(1 << 17, 3, device="cuda", generator=gen), points("rays", 1 << 17, 3, gen)):
        times.append(time_of(adjoint_call(enc, x, table, g)[0]))
    print("random, rays:", times, flush=True)
    assert times[1] < 2 * times[0]


def test_time_grows_with_the_batch():
    """Floats that are too small for the fixed-point sums of a slice grow with the square of its records: 2^20 points behind a dense 4-D
    grid of 8 features have more of them than the list of a workgroup holds. Reading all records a second time for these made the pass
    2.7 times as long as that of half as many points (twice where they are added right away)."""
    cfg = GRIDS["many"]
    require_gpu(cfg, (2,))
    enc = qmlp.Encoding(json.dumps(cfg))
    gen = torch.Generator(device="cuda").manual_seed(1)
    table = torch.zeros(enc.num_parameters(), device="cuda", dtype=enc.parameter_dtype())
    times = []
    for count in (1 << 19, 1 << 20):
        x, g = torch.rand(count, 4, device="cuda", generator=gen), torch.randn(count, 8, device="cuda", generator=gen)
        times.append(time_of(adjoint_call(enc, x, table, g)[0]))
    print("2^19, 2^20 points:", times, flush=True)
    assert times[1] < 2.45 * times[0]
