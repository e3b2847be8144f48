"""Gradients by products over shared cells: the same bits in input and in cell
order and under a mask, the finite differences the bits of nglod_normals_fd
(whose decoder runs on the vector ALU), the autodiff gradient against float64
autograd, and decoders with a weight that is not finite."""
import pytest
import torch

from nglod_amd import _lib, workloads

pytestmark = pytest.mark.gpu


def _points(n, spread, dev):
    g = torch.Generator().manual_seed(n)
    x = torch.rand(n, 3, generator=g) * spread - spread / 2
    if n > 8:
        x[2, 0], x[3, 1], x[4, 2], x[5] = 1.0, -1.0, 1.5, 0.0
    return x.to(dev)


@pytest.mark.parametrize("method", ["autodiff", "finitediff", "tetrahedron"])
@pytest.mark.parametrize("pos_invariant", [True, False])
@pytest.mark.parametrize("n, spread", [(1, 2.0), (32, 2.0), (33, 0.01), (65, 0.1), (257, 0.5), (30000, 2.2)])
def test_order_and_mask_keep_the_bits(dev, n, spread, pos_invariant, method):
    net = workloads.make_model(num_lods=5, pos_invariant=pos_invariant, seed=1, device=dev)
    x = _points(n, spread, dev)
    mask = torch.arange(n, device=dev) % 3 == 0
    for lod in (0, 2, 4):
        a = net.gradient_hip(x, lod, method, ordered=False)
        assert torch.equal(a, net.gradient_hip(x, lod, method, ordered=True))
        m = net.gradient_hip(x, lod, method, mask=mask, ordered=True)
        assert torch.equal(m, torch.where(mask[:, None], a, torch.zeros_like(a)))


@pytest.mark.parametrize("pos_invariant", [True, False])
@pytest.mark.parametrize("n, spread", [(1, 2.0), (63, 0.02), (500, 0.3), (20000, 2.2)])
def test_finite_differences_of_the_other_kernel(dev, n, spread, pos_invariant):
    net = workloads.make_model(num_lods=5, pos_invariant=pos_invariant, seed=2, device=dev)
    x = _points(n, spread, dev)
    for lod in (0, 3, 4):
        got = net.gradient_hip(x, lod, "finitediff", normalize=True)
        want = torch.empty_like(got)
        _lib.check(_lib.load().nglod_normals_fd(net.descriptor(), _lib.ptr(x), n, lod, 0, _lib.ptr(want),
                                                _lib.stream_of(x)), "nglod_normals_fd")
        assert torch.equal(got, want)


def _sdf64(net, x, lod):
    """The SDF in float64 from the module's parameters."""
    p = x.double().cpu().requires_grad_(True)
    f = 0.0
    for l in range(lod + 1):
        vol = net.features[l].fm.detach().double().cpu()
        f = f + torch.nn.functional.grid_sample(vol, p.reshape(1, -1, 1, 1, 3), align_corners=True,
                                                padding_mode="border")[0, :, :, 0, 0].T
    e = f if net.pos_invariant else torch.cat([p, f], 1)
    w0, b0, w1, b1 = (t.detach().double().cpu() for t in (net.louts[lod][0].weight, net.louts[lod][0].bias,
                                                         net.louts[lod][2].weight, net.louts[lod][2].bias))
    pre = e @ w0.T + b0
    y = torch.relu(pre) @ w1.T + b1
    return y.detach(), torch.autograd.grad(y.sum(), p)[0], pre.detach()


@pytest.mark.parametrize("pos_invariant", [True, False])
@pytest.mark.parametrize("spread", [0.05, 0.4, 1.98])
def test_autodiff_against_float64(dev, pos_invariant, spread):
    """Sums of at most 8 * 32 * 5 + 128 FP32 products of O(1) operands: 1e-5 of the
    largest, where no unit's pre-activation is within rounding of 0."""
    net = workloads.make_model(num_lods=5, pos_invariant=pos_invariant, seed=3, device=dev)
    g = torch.Generator().manual_seed(7)
    x = (torch.rand(3000, 3, generator=g) * spread - spread / 2).to(dev)
    for lod in (0, 4):
        y64, g64, pre = _sdf64(net, x, lod)
        sure = (pre.abs() > 1e-5 * pre.abs().max()).all(1)
        assert sure.sum() > 2000
        got = net.gradient_hip(x, lod, "autodiff").cpu().double()
        assert (got - g64)[sure].abs().max() <= 1e-5 * g64.abs().max()
        y, g2 = net.sdf_grad_hip(x, lod)
        assert torch.equal(g2.cpu().double(), got)
        assert (y.cpu().double() - y64).abs().max() <= 1e-5 * y64.abs().max().clamp_min(1.0)


def test_weight_that_is_not_finite(dev):
    """A unit with a weight of -inf is off where the feature is positive and passes
    no gradient there: the gradient without that unit."""
    net = workloads.make_model(num_lods=2, pos_invariant=True, seed=4, device=dev)
    x = _points(4000, 1.9, dev)
    with torch.no_grad():
        keep = net.louts[1][2].weight[0, 17].clone()
        net.louts[1][2].weight[0, 17] = 0.0
        want = net.gradient_hip(x, 1, "autodiff")
        net.louts[1][2].weight[0, 17] = keep
        net.louts[1][0].weight[17, 5] = -float("inf")
    f5 = sum(net.features[l](x)[:, 5] for l in (0, 1))
    off = f5 > 0
    assert 100 < off.sum() < 3900
    got = net.gradient_hip(x, 1, "autodiff")
    assert (got - want)[off].abs().max() <= 1e-5 * want.abs().max()
