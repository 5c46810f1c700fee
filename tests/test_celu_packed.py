"""CELU's packed form (an IEEE minimum in the place of a comparison and a choice) gives the bits of its snippet, which another spelling keeps
from being recognised: pre-activations that are zero, minus zero, denormal, large, infinite or NaN, in every form of the backward kernel."""
import json

import pytest
import torch

import qmlp
from helpers import identity_cfg, warm_cache

pytestmark = pytest.mark.gpu

PLAIN = {"id": "celu_plain", "forward": "z = (__hgt(x, hZERO()) ? x : __hsub(hexp(x), __float2half(1.0f)))",
         "adjoint": "adjx = (__hgt(x, hZERO()) ? adjz : __hmul(adjz, hexp(x)))"}
SPECIAL = [0.0, -0.0, 2.0 ** -24, -2.0 ** -24, 2.0 ** -14, -2.0 ** -14, 1e-3, -1e-3, 0.7, -0.7, 9.0, -9.0, -20.0, 65504.0, -65504.0, -1.0]
OPTIONS = [{"cooperative_backward": 1}, {"cooperative_backward": 0}, {"cooperative_backward": 0, "recompute_intermediates": 0},
           {"cooperative_backward": 0, "fused_weight_update": 0}]


@pytest.mark.parametrize("options", OPTIONS)
@pytest.mark.parametrize("not_finite", [False, True])
def test_packed_celu_gives_the_bits_of_the_snippet(options, not_finite):
    """Weights of the first layer: the identity, so that its pre-activations are the inputs."""
    widths = [16, 32, 4]
    cfgs = [dict(identity_cfg(16, widths, [a, a, "identity"], [False, True, False], extra_acts=[PLAIN]), options=options) for a in ("celu", "celu_plain")]
    warm_cache(*cfgs)
    nets = [qmlp.FusedNetwork(json.dumps(c), weight_dtype=torch.float32) for c in cfgs]
    with torch.no_grad():
        a, b = (max(net.parameters(), key=torch.Tensor.numel) for net in nets)
        a.copy_(torch.rand(a.shape, generator=torch.Generator().manual_seed(1)).cuda() - 0.5)
        a.view(-1)[:256] = torch.eye(16, device="cuda").view(-1)
        b.copy_(a)
    for n in (1, 33, 1000):
        gen = torch.Generator(device="cuda").manual_seed(n)
        x = torch.randn(n, 16, device="cuda", generator=gen) * 3
        x[n // 2] = torch.tensor(SPECIAL, device="cuda")
        if not_finite:   # (every unit of the next layer then is NaN for such a point)
            x[n // 3, 3], x[n // 4, 5], x[n - 1, 7] = float("nan"), float("inf"), -float("inf")
        g = torch.randn(n, 4, device="cuda", generator=gen)
        results = []
        for net in nets:
            xs = x.clone().requires_grad_(True)
            out = net(xs)
            weights = max(net.parameters(), key=torch.Tensor.numel)
            results.append([out, *torch.autograd.grad(out, [xs, weights], g)])
        for got, expected in zip(*results):
            assert torch.equal(torch.isnan(got), torch.isnan(expected)) and torch.equal(torch.nan_to_num(got, nan=7.0), torch.nan_to_num(expected, nan=7.0))
        assert not_finite or torch.isfinite(results[0][1]).all()
