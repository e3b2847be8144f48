"""The backward at the edges of its chunks (256 queries), tiles (32 and 64),
pieces (64 contributions per corner) and launch split (few queries: a level
per block), against FP64 autograd of the reference's operators; and two calls
that take the same sums another way.

Tolerance: FP32 sums of up to n terms against FP64: 1e-4 of the largest entry,
the bar of the package's other gradient tests."""
import pytest
import torch

from nglod_amd import workloads
from oracle.torch_ref import TorchOctreeSDF

pytestmark = pytest.mark.gpu


def _grads(net, x, gt):
    net.zero_grad()
    preds = net.sdf(x, return_lst=True)
    (sum(((p - gt) ** 2).sum() for p in preds) / x.shape[0]).backward()
    return {k: v.grad.detach().clone() for k, v in net.named_parameters()}


def _grads64(net, x, gt):
    ref = TorchOctreeSDF.from_module(net, dtype=torch.float64)
    params = ref.fms + ref.w0 + ref.b0 + ref.w1 + ref.b1
    for p in params:
        p.requires_grad_(True)
    preds = ref.sdf(x.cpu().double(), return_lst=True)
    (sum(((p - gt.cpu().double()) ** 2).sum() for p in preds) / x.shape[0]).backward()
    out = {}
    for i, f in enumerate(ref.fms):
        out[f"features.{i}.fm"] = f.grad
    for i in range(len(ref.w0)):
        out[f"louts.{i}.0.weight"], out[f"louts.{i}.0.bias"] = ref.w0[i].grad, ref.b0[i].grad
        out[f"louts.{i}.2.weight"], out[f"louts.{i}.2.bias"] = ref.w1[i].grad, ref.b1[i].grad
    return out


@pytest.mark.parametrize("n", [1, 2, 31, 33, 64, 65, 255, 257, 1000, 4097])
@pytest.mark.parametrize("pos_invariant", [True, False])
def test_edges_vs_fp64(dev, n, pos_invariant):
    net = workloads.make_model(num_lods=3, pos_invariant=pos_invariant, seed=n, device=dev)
    g = torch.Generator().manual_seed(n)
    x = (torch.rand(n, 3, generator=g) * 2.2 - 1.1).to(dev)  # some outside the box: clamped cells
    gt = torch.rand(n, 1, generator=g).to(dev)
    got, want = _grads(net, x, gt), _grads64(net, x, gt)
    for k, w in want.items():
        err = (got[k].cpu().double().reshape(w.shape) - w).abs().max().item()
        assert err <= 1e-4 * max(w.abs().max().item(), 1e-6), (k, err)


@pytest.mark.parametrize("n", [300, 20000])
def test_all_queries_in_one_cell(dev, n):
    """Runs of n contributions per corner, and empty corners."""
    net = workloads.make_model(num_lods=4, seed=1, device=dev)
    g = torch.Generator().manual_seed(2)
    x = (torch.rand(n, 3, generator=g) * 0.02 + 0.26).to(dev)
    gt = torch.rand(n, 1, generator=g).to(dev)
    got, want = _grads(net, x, gt), _grads64(net, x, gt)
    for k, w in want.items():
        err = (got[k].cpu().double().reshape(w.shape) - w).abs().max().item()
        assert err <= 1e-4 * max(w.abs().max().item(), 1e-6), (k, err)
    assert (got["features.3.fm"] != 0).any(1).sum().item() <= 8 * 4


def test_last_level_alone_is_the_call_at_its_lod(dev):
    """The last level's share of a call of every level, against the call at
    that LOD: the same sums, of other levels' zeros in the first."""
    net = workloads.make_model(num_lods=3, seed=4, device=dev)
    g = torch.Generator().manual_seed(5)
    x = (torch.rand(30000, 3, generator=g) * 2 - 1).to(dev)
    net.zero_grad()
    net.sdf(x, lod=2).sum().backward()
    a = {k: v.grad.clone() for k, v in net.named_parameters() if v.grad is not None}
    net.zero_grad()
    net.sdf(x, return_lst=True)[2].sum().backward()
    b = {k: v.grad.clone() for k, v in net.named_parameters() if v.grad is not None}
    for i in range(3):
        assert torch.equal(a[f"features.{i}.fm"], b[f"features.{i}.fm"])
    for k in ("louts.2.0.weight", "louts.2.0.bias", "louts.2.2.weight", "louts.2.2.bias"):
        assert torch.equal(a[k], b[k])


@pytest.mark.parametrize("n", [300, 40000])
@pytest.mark.parametrize("pos_invariant", [True, False])
def test_saved_features_give_the_same_bits(dev, n, pos_invariant, monkeypatch):
    """The backward on the forward's saved features against one that computes
    them again (a batch above the limit, or weights changed in between), and
    the predictions against the plain call's."""
    from nglod_amd import autograd

    net = workloads.make_model(num_lods=4, pos_invariant=pos_invariant, seed=7, device=dev)
    g = torch.Generator().manual_seed(8)
    x, gt = (torch.rand(n, 3, generator=g) * 2 - 1).to(dev), torch.rand(n, 1, generator=g).to(dev)
    a = _grads(net, x, gt)
    preds = net.sdf(x, return_lst=True)
    with torch.no_grad():
        for p, q in zip(preds, net.sdf(x, return_lst=True)):
            assert torch.equal(p, q)
    monkeypatch.setattr(autograd, "SAVE_LIMIT", 0)
    b = _grads(net, x, gt)
    for k in a:
        assert torch.equal(a[k], b[k]), k
    monkeypatch.undo()
    loss = sum(((p - gt) ** 2).sum() for p in net.sdf(x, return_lst=True))
    net.zero_grad()
    with torch.no_grad():
        net.louts[0][0].weight.mul_(2.0)
    loss.backward()  # on the new weights' features
    c = {k: v.grad.clone() for k, v in net.named_parameters()}
    monkeypatch.setattr(autograd, "SAVE_LIMIT", 0)
    with torch.no_grad():
        net.louts[0][0].weight.div_(2.0)
    loss = sum(((p - gt) ** 2).sum() for p in net.sdf(x, return_lst=True))
    net.zero_grad()
    with torch.no_grad():
        net.louts[0][0].weight.mul_(2.0)
    loss.backward()
    for k, v in net.named_parameters():
        assert torch.equal(c[k], v.grad), k
