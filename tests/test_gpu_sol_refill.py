"""The sparse march by groups hands a finished ray's lane to the next claimed ray: a group
of 32 takes 64 rays a claim, so half of its refills come without a claim.  Rays end
at an evaluation, or in the walk without one (their voxels all lie behind them), whole
groups of them at a time; each form of refill gives the bits of a ray per lane."""
import pytest
import torch

from nglod_amd import mesh, workloads
from nglod_amd.sol import SolNGLOD
from nglod_amd.spc import SPC
from tests.helpers import rand_rays
from tests.test_gpu_sol_group import _march

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("behind", ["all", "every other", "runs of 32", "runs of 48"])
@pytest.mark.parametrize("n", [33, 64, 97, 20003])
def test_refill_without_a_claim(dev, n, behind):
    net = workloads.make_sphere_model(radius=0.6, num_lods=3, pos_invariant=False, device="cpu").to(dev)
    V, F = mesh.icosphere(3)
    spc = SPC.from_mesh(mesh.triangles(V * 0.6, F), 5, dev)
    sol = SolNGLOD.from_net(net, spc, fp16=False)
    o = torch.from_numpy(rand_rays(n, n, dist=(1.5, 2.5))[0]).to(dev)
    aim = 0.2 * torch.randn(n, 3, generator=torch.Generator().manual_seed(n)).to(dev)
    d = torch.nn.functional.normalize(aim - o, dim=-1)
    lists = spc.raytrace(o, d, 4)
    i = torch.arange(n, device=dev)
    turned = {"all": i >= 0, "every other": i % 2 == 0, "runs of 32": i // 32 % 2 == 0,
              "runs of 48": i // 48 % 2 == 0}[behind]
    d = torch.where(turned[:, None], -d, d).contiguous()
    desc = sol.descriptor(2)
    got = _march(sol, desc, o, d, lists)
    shifted = torch.empty(spc.points.numel() + 1, dtype=torch.int16, device=dev)
    shifted[1:] = spc.points.reshape(-1)
    desc.points = shifted.data_ptr() + 2
    want = _march(sol, desc, o, d, lists)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    has = lists[1][1:] > lists[1][:-1]
    assert (has & turned).any() and not (got[2].bool() & turned).any()
    assert bool(turned.all()) or got[2].any()
