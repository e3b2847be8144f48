"""nglod_adam_step against torch.optim.Adam bit for bit over the whole range of beta1
(torch's lerp changes its formula at a weight of 1/2), with moments far larger than
the gradients that replace them."""
import pytest
import torch

from nglod_amd.optim import Adam
from tests.test_gpu_optim import _params, _set_grads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("beta1", [0.0, 1e-9, 0.3, 0.49999999, 0.5, 0.50000001, 0.5000001, 0.6, 0.9999999])
def test_beta1(dev, beta1):
    a, b = _params(dev), _params(dev)
    oa, ob = (o(p, lr=1e-3, betas=(beta1, 0.99)) for o, p in ((Adam, a), (torch.optim.Adam, b)))
    for step in range(5):
        _set_grads(a, step)
        _set_grads(b, step)
        for p, q in zip(a, b):
            if step == 1:
                p.grad.mul_(1e8)
                q.grad.mul_(1e8)
        oa.step()
        ob.step()
        for i, (p, q) in enumerate(zip(a, b)):
            assert torch.equal(p, q), (step, i)
            for k in ("step", "exp_avg", "exp_avg_sq"):
                assert torch.equal(oa.state[p][k], ob.state[q][k]), (step, i, k)
            if beta1 == 0.0:
                assert torch.equal(oa.state[p]["exp_avg"], p.grad)
