"""The FP32 dense trace (32 rays per block of four waves) against the same
recurrence stepped over the whole batch with nglod_sdf_fwd, bit for bit: part-filled
groups, more rays than the GPU holds at once, coarsest grids that fit the block's
LDS table and that do not, rays that start inside the box and that miss it."""
import numpy as np
import pytest
import torch

from nglod_amd import workloads
from nglod_amd.sol_nglod import aabb
from nglod_amd.tracer import SphereTracer

from helpers import rand_rays

pytestmark = pytest.mark.gpu

MIN_DIS, FAR, H = 3e-4, 10.0, np.float32(1.0 / 192.0)


def _step_all(net, o, d, lod, steps):
    """SphereTracer.forward over the batch (SphereTracer.py:59-119)."""
    f = lambda p: net.sdf_hip(p, lod, ordered=False)[:, 0]
    x, t, hit = aabb(o, d)
    t, inside = t.reshape(-1), hit.reshape(-1).bool()
    cond = inside.clone()
    D = torch.where(inside, f(x), torch.zeros_like(t))
    Dp, hitflag, count = D.clone(), torch.zeros_like(cond), torch.zeros(len(t), dtype=torch.int32, device=t.device)
    alive = torch.ones_like(cond)
    for _ in range(steps):
        far = t.abs() < FAR
        go = alive & inside & (D.abs() > np.float32(MIN_DIS)) & (((D + Dp) * 0.5).abs() > np.float32(MIN_DIS * 3.0)) & far
        hitflag = torch.where(alive, far, hitflag)
        alive = go
        x = torch.where(go[:, None], o + d * t[:, None], x)
        v = f(x)
        Dp = torch.where(go, D, Dp)
        D = torch.where(go, v, D)
        t = torch.where(go, t + D, t)
        count += go.int()
    hit = hitflag & ~(x.abs() > 1.0).any(1)
    return x, t, hit, count


def _normals(net, x, lod):
    f = lambda p: net.sdf_hip(p, lod, ordered=False)[:, 0]
    g = []
    for a in range(3):
        e = torch.zeros(3, device=x.device)
        e[a] = float(H)
        g.append((f(x + e) - f(x - e)) / np.float32(2.0 / 192.0))
    return torch.nn.functional.normalize(torch.stack(g, 1), eps=1e-5)


@pytest.mark.parametrize("n, base_lod, num_lods, pos_invariant",
                         [(1, 2, 5, True), (31, 2, 5, False), (32, 0, 3, True), (33, 1, 8, False), (257, 2, 1, True),
                          (4099, 3, 4, True), (4099, 2, 2, False), (150001, 2, 5, True)])
def test_same_bits_as_whole_batch_steps(dev, n, base_lod, num_lods, pos_invariant):
    net = workloads.make_sphere_model(radius=0.6, num_lods=num_lods, base_lod=base_lod, pos_invariant=pos_invariant,
                                      device="cpu").to(dev)
    o, d = rand_rays(n, 5 + n)
    o[::7] *= 0.2
    o, d = torch.from_numpy(o).to(dev), torch.from_numpy(d).to(dev)
    lod = num_lods - 1
    net.lod = lod
    steps = torch.full((n,), -1, dtype=torch.int32, device=dev)
    rb = SphereTracer(num_steps=40, min_dis=MIN_DIS)(net, o, d, ray_steps=steps)
    x, t, hit, count = _step_all(net, o, d, lod, 40)
    assert torch.equal(rb.hit.reshape(-1), hit)
    assert torch.equal(rb.x, x)
    assert torch.equal(rb.depth.reshape(-1), t)
    assert torch.equal(steps, count)
    assert torch.all(rb.normal[~hit] == 0)
    if hit.any():
        # the same taps; torch's norm and division may round the last bits differently
        assert (rb.normal[hit] - _normals(net, x[hit], lod)).abs().max() <= 4e-7
    if n > 1000:
        assert n // 10 < hit.sum() < n


@pytest.mark.parametrize("n, num_lods, pos_invariant",
                         [(15, 5, False), (16, 1, False), (17, 5, True), (47, 3, False), (100, 8, True),
                          ((1 << 18) + 33, 2, False), ((1 << 19) + 1, 4, True)])
def test_few_rays_and_long_frames(dev, n, num_lods, pos_invariant):
    """Around the 16 and 8 rays from which a block's last trips go other ways, and
    frames long enough to go without them: the same bits."""
    base_lod = 1 if num_lods == 8 else 2
    net = workloads.make_sphere_model(radius=0.6, num_lods=num_lods, base_lod=base_lod, pos_invariant=pos_invariant,
                                      device="cpu").to(dev)
    o, d = rand_rays(n, 7 + n)
    o[::5] *= 0.2
    o, d = torch.from_numpy(o).to(dev), torch.from_numpy(d).to(dev)
    net.lod = num_lods - 1
    steps = torch.full((n,), -1, dtype=torch.int32, device=dev)
    rb = SphereTracer(num_steps=24, min_dis=MIN_DIS)(net, o, d, ray_steps=steps)
    x, t, hit, count = _step_all(net, o, d, num_lods - 1, 24)
    assert torch.equal(rb.hit.reshape(-1), hit)
    assert torch.equal(rb.x, x)
    assert torch.equal(rb.depth.reshape(-1), t)
    assert torch.equal(steps, count)
    if hit.any():
        assert (rb.normal[hit] - _normals(net, x[hit], num_lods - 1)).abs().max() <= 4e-7
