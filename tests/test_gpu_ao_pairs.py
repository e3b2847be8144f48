"""Ambient occlusion by (hit, tap) pairs: each claim size (8, 16, 32 rays), claims
with no hit and with a few, plane hits, points far apart and in one cell.  The
FP32 form against the formula on batch queries bit for bit; the mixed form
against the FP32 form within 40 taps * 3.5 * 1e-6 (each value is FP32-level, the
cumulative grid sums levels beforehand), doubled by the square."""
import math

import pytest
import torch

from nglod_amd import workloads
from nglod_amd.renderer import ambient_occlusion

pytestmark = pytest.mark.gpu


def _want(net, x, normal, hit, plane, lod):
    acc = torch.zeros(len(x), device=x.device)
    for k in range(40):
        dk = torch.tensor(0.1 * 0.25 * math.pow((k + 1) / 41.0, 1.6), dtype=torch.float64).float().item()
        r = net.sdf_hip((x + normal * dk).contiguous(), lod, ordered=False)[:, 0]
        r = torch.where(hit, r, r.clamp(max=dk))
        u = (torch.tensor(dk, device=x.device) - r) - torch.tensor(0.0015, device=x.device)
        acc = acc + torch.tensor(3.5, device=x.device) * u.clamp(min=0.0)
    v = (1.0 - acc).clamp(0.1, 1.0)
    return torch.where(hit | plane, v * v, torch.ones_like(v))


@pytest.mark.parametrize("pos_invariant", [True, False])
@pytest.mark.parametrize("n, spread, share", [(1, 1.0, 1.0), (7, 1.0, 0.5), (8, 1.0, 0.0), (65, 0.001, 1.0),
                                              (4099, 0.9, 0.6), (200003, 0.9, 0.3), (400009, 0.9, 0.05)])
def test_pairs(dev, n, spread, share, pos_invariant):
    net = workloads.make_sphere_model(radius=0.6, num_lods=4, pos_invariant=pos_invariant, device="cpu").to(dev)
    g = torch.Generator().manual_seed(n)
    lod = 3
    net.lod = lod
    normal = torch.nn.functional.normalize(torch.randn(n, 3, generator=g), dim=1)
    x = (normal * 0.6 + (torch.rand(n, 3, generator=g) - 0.5) * spread * 0.1 if spread > 0.1
         else torch.tensor([0.6, 0.0, 0.0]) + torch.rand(n, 3, generator=g) * spread)
    hit = torch.rand(n, generator=g) < share
    plane = ~hit & (torch.rand(n, generator=g) < share / 3)
    x, normal, hit, plane = (t.to(dev) for t in (x, normal, hit, plane))
    got = ambient_occlusion(net, x, normal, hit, plane).reshape(-1)
    want = _want(net, x, normal, hit, plane, lod)
    assert torch.equal(got, want)
    mixed = ambient_occlusion(net, x, normal, hit, plane, form="mixed").reshape(-1)
    assert (mixed - want).abs().max() <= 5e-4
    if n > 4000:
        assert (want < 0.99).sum() > n * share * 0.1
