"""The features that a forward keeps for its backward are used only where nothing can have
changed the weights in between: a loop of its own takes one set of weights, those the
backward finds, also when they were written through .data; Trainer.step_geometry, which
keeps them, gives such a loop's gradients bit for bit."""
import pytest
import torch

from nglod_amd import autograd, workloads
from nglod_amd.trainer import Trainer

pytestmark = pytest.mark.gpu


def _inputs(dev, n):
    g = torch.Generator().manual_seed(n)
    return (torch.rand(n, 3, generator=g) * 2 - 1).to(dev), torch.rand(n, 1, generator=g).to(dev)


def _grads(net):
    return {k: v.grad.detach().clone() for k, v in net.named_parameters()}


@pytest.mark.parametrize("what", ["features.1.fm", "louts.0.0.weight", "louts.2.0.bias", "louts.1.2.weight"])
@pytest.mark.parametrize("n", [300, 30000])
def test_weights_written_through_data_before_the_backward(dev, n, what):
    x, gt = _inputs(dev, n)
    g = torch.Generator(device=dev).manual_seed(1)
    nets = [workloads.make_model(num_lods=3, seed=3, device=dev) for _ in range(2)]
    new = dict(nets[0].named_parameters())[what].detach()
    new = new + 0.1 * torch.randn(new.shape, generator=g, device=dev)
    preds = nets[0].sdf(x, return_lst=True)
    with torch.no_grad():
        out_grads = [2.0 / n * (p - gt) for p in preds]
    dict(nets[0].named_parameters())[what].data.copy_(new)
    torch.autograd.backward(preds, out_grads)
    # the same incoming gradients on a model that had the new weights from the start
    with torch.no_grad():
        dict(nets[1].named_parameters())[what].copy_(new)
    torch.autograd.backward(nets[1].sdf(x, return_lst=True), out_grads)
    a, b = _grads(nets[0]), _grads(nets[1])
    for k in a:
        assert torch.equal(a[k], b[k]), k


@pytest.mark.parametrize("n", [1, 300, 40000])
@pytest.mark.parametrize("pos_invariant", [True, False])
def test_a_step_keeps_features_and_gives_the_loops_bits(dev, n, pos_invariant, monkeypatch):
    x, gt = _inputs(dev, n)
    grads = []
    for limit in (autograd.SAVE_LIMIT, 0):
        monkeypatch.setattr(autograd, "SAVE_LIMIT", limit)
        net = workloads.make_model(num_lods=4, pos_invariant=pos_invariant, seed=7, device=dev)
        Trainer(net).step_geometry(x, gt)
        grads.append(_grads(net))
    net = workloads.make_model(num_lods=4, pos_invariant=pos_invariant, seed=7, device=dev)
    (sum(((p - gt) ** 2).sum() for p in net.sdf(x, return_lst=True)) / n).backward()
    grads.append(_grads(net))
    for k in grads[0]:
        assert torch.equal(grads[0][k], grads[1][k]) and torch.equal(grads[0][k], grads[2][k]), k
