"""Ambient occlusion claims rays in chunks, and more at once where a chunk holds no hit:
each hit's value is the one it has alone, whatever lies around it: no hits, single ones far
apart, runs longer than a wave's 32 after empty stretches, every ray, planes among them."""
import pytest
import torch

from nglod_amd import _lib, workloads
from nglod_amd.renderer import ambient_occlusion

pytestmark = pytest.mark.gpu


def _pattern(name, n, g):
    i = torch.arange(n)
    return {"none": i < 0, "all": i >= 0, "first": i == 0, "last": i == n - 1, "sparse": i % 997 == 5,
            "runs": (i // 700) % 3 == 1, "random": torch.rand(n, generator=g) < 0.02,
            "half": i >= n // 2}[name]


@pytest.mark.parametrize("pattern", ["none", "all", "first", "last", "sparse", "runs", "random", "half"])
@pytest.mark.parametrize("n", [1, 65, 5000, 250007, 700001])
@pytest.mark.parametrize("form, posinv", [("fp32", True), ("mixed", False)])
def test_patterns(dev, n, pattern, form, posinv):
    net = workloads.make_sphere_model(radius=0.6, num_lods=3, pos_invariant=posinv, device="cpu").to(dev)
    g = torch.Generator().manual_seed(n)
    u = torch.nn.functional.normalize(torch.randn(n, 3, generator=g), dim=1)
    x = (u * (0.58 + 0.02 * torch.rand(n, 1, generator=g))).to(dev)  # inside: occluded taps
    u = u.to(dev)
    hit = _pattern(pattern, n, g).to(dev)
    plane = (torch.arange(n, device=dev) % 13 == 3) & ~hit if pattern in ("random", "first") else None
    marked = hit if plane is None else hit | plane
    kw = dict(lod=2, form=form)
    if plane is not None:
        kw["plane_hit"] = plane
    ao = ambient_occlusion(net, x, u, hit, **kw)[:, 0]
    assert (ao[~marked] == 1.0).all()
    ids = marked.nonzero()[:, 0]
    if ids.numel() == 0:
        return
    # the marked rays by themselves, in reverse order
    ids = ids.flip(0)
    if plane is not None:
        kw["plane_hit"] = plane[ids].contiguous()
    alone = ambient_occlusion(net, x[ids].contiguous(), u[ids].contiguous(), hit[ids].contiguous(), **kw)[:, 0]
    assert torch.equal(ao[ids], alone)
    assert (alone < 1.0).any() and (ids.numel() < 100 or alone.unique().numel() > 20)


def test_workspace_of_256_bytes(dev):
    """What a workspace of one counter holds is enough."""
    n = 100003
    net = workloads.make_sphere_model(radius=0.6, num_lods=3, pos_invariant=True, device="cpu").to(dev)
    u = torch.nn.functional.normalize(torch.randn(n, 3, generator=torch.Generator().manual_seed(1)), dim=1)
    x, u = (0.59 * u).to(dev), u.to(dev)
    hit = (torch.arange(n, device=dev) % 5 != 0)
    want = ambient_occlusion(net, x, u, hit, lod=2)
    lib = _lib.load()
    assert lib.nglod_ao_workspace_size() > 256
    guard = torch.full((4096,), 7, dtype=torch.uint8, device=dev)
    ao = torch.empty(n, 1, device=dev)
    call = lambda size: lib.nglod_ao(net.descriptor(_lib.FP32), _lib.ptr(x), _lib.ptr(u), _lib.ptr(hit.view(torch.uint8)),
                                     None, n, 2, _lib.FP32, _lib.ptr(ao), _lib.ptr(guard), size, _lib.stream_of(x))
    assert call(255) == _lib.ERR_WORKSPACE
    assert call(256) == 0
    assert torch.equal(ao, want) and (guard[256:] == 7).all()
