"""nglod_amd's Adam where torch's own step runs: on the CPU, with gradients and without."""
import pytest
import torch

from nglod_amd.optim import Adam


@pytest.mark.parametrize("grads", ["none", "some", "all"])
def test_steps_on_the_cpu(grads):
    torch.manual_seed(0)
    a = [torch.nn.Parameter(torch.randn(4, 3)), torch.nn.Parameter(torch.randn(5))]
    b = [torch.nn.Parameter(p.detach().clone()) for p in a]
    oa, ob = Adam(a, lr=0.1), torch.optim.Adam(b, lr=0.1)
    calls = []
    oa.register_step_post_hook(lambda *_: calls.append(1))
    for _ in range(3):
        for p, q in list(zip(a, b))[: {"none": 0, "some": 1, "all": 2}[grads]]:
            p.grad = torch.randn_like(p)
            q.grad = p.grad.clone()
        assert oa.step() is None and ob.step() is None
    assert all(torch.equal(p, q) for p, q in zip(a, b)) and len(calls) == 3
    assert len(oa.state) == len(ob.state)
