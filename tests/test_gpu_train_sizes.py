"""Training at the largest sizes a model may have: a grid of 512^3 cells (more (corner,
channel) pairs than a launch holds threads), eight levels (all their decoders in
one block's LDS), and levels in any order of resolution, against FP64 autograd.

Tolerance: FP32 sums of up to n terms against FP64: 1e-4 of the largest entry,
the bar of the package's other gradient tests.  The units' biases are 1 or -1, far from
every ReLU's kink: among millions of units some lie within FP32 rounding of it otherwise,
and one on the other side moves an entry by about that bar."""
import ctypes

import pytest
import torch
import torch.nn.functional as F

from nglod_amd import _lib, workloads
from nglod_amd.trainer import Trainer
from tests.test_gpu_train_bits import _grads64

pytestmark = pytest.mark.gpu


def _close(got, want, what):
    err = (got.double().reshape(want.shape) - want).abs().max().item()
    assert err <= 1e-4 * max(want.abs().max().item(), 1e-6), (what, err)


def _corners(x, r):
    """Rows [n, 8] and weights of each point's cell in an r^3 grid: the coordinate rounded to
    FP32 as the kernels form it, the products FP64."""
    u = ((x + 1) * 0.5 * r).clamp(0, r).double()
    i = u.floor().clamp(max=r - 1)
    w = torch.stack([i + 1 - u, u - i])  # [2, n, xyz]
    i = i.long()
    rows, ws = [], []
    for k in range(8):
        b = [k & 1, (k >> 1) & 1, k >> 2]
        rows.append(((i[:, 2] + b[2]) * (r + 1) + i[:, 1] + b[1]) * (r + 1) + i[:, 0] + b[0])
        ws.append(w[b[0], :, 0] * w[b[1], :, 1] * w[b[2], :, 2])
    return torch.stack(rows, 1), torch.stack(ws, 1)


def _backward(res, x, seed):
    """nglod_sdf_bwd on random decoders, random features in the rows that x touches and random
    grad_out; and the same gradients in FP64: per level (rows, got, want, grid gradient), per decoder."""
    dev, n, L = x.device, x.shape[0], len(res)
    g = torch.Generator(device=dev).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev) * 0.1
    m, G = _lib.NglodModel(L, 32, 128, 1, L), _lib.NglodModelGrads()
    decs = [(rnd(128, 32), rnd(128).sign(), rnd(128), rnd(1)) for _ in res]
    go, keep, cells = rnd(L, n), [], []
    for l, r in enumerate(res):
        rows, w = _corners(x, r)
        used, at = torch.unique(rows, return_inverse=True)
        grid = torch.zeros((r + 1) ** 3, 32, device=dev)
        grid[used] = rnd(used.numel(), 32)
        grad = torch.empty_like(grid)
        dg = [torch.empty_like(t) for t in decs[l]]
        m.res[l], m.grid[l], G.grid[l] = r, grid.data_ptr(), grad.data_ptr()
        for name, t, d in zip(("w0", "b0", "w1", "b1"), decs[l], dg):
            getattr(m, name)[l], getattr(G, name)[l] = t.data_ptr(), d.data_ptr()
        keep.append((grid, grad, dg))
        cells.append((used, at, w, grid[used].double().requires_grad_(True)))
    lib = _lib.load()
    ws = torch.empty(lib.nglod_sdf_bwd_workspace_size(m, n, L - 1), dtype=torch.uint8, device=dev)
    _lib.check(lib.nglod_sdf_bwd(m, _lib.ptr(x), n, L - 1, _lib.ptr(go), (1 << L) - 1, ctypes.byref(G), _lib.ptr(ws),
                                 ws.numel(), _lib.stream_of(x)), "nglod_sdf_bwd")
    params = [[t.double().requires_grad_(True) for t in d] for d in decs]
    e = 0.0
    total = 0.0
    for l in range(L):
        _, at, w, feats = cells[l]
        e = e + (feats[at] * w[..., None]).sum(1)
        w0, b0, w1, b1 = params[l]
        total = total + ((F.relu(F.linear(e, w0, b0)) @ w1 + b1) * go[l].double()).sum()
    total.backward()
    levels = [(c[0], k[1][c[0]], c[3].grad, k[1]) for c, k in zip(cells, keep)]
    return levels, [list(zip(k[2], [t.grad for t in p])) for k, p in zip(keep, params)]


@pytest.mark.parametrize("res", [[512], [4, 512]])
def test_grid_of_512(dev, res):
    free = torch.cuda.mem_get_info()[0]
    if free < 80 << 30:
        pytest.skip(f"needs 80 GiB of free memory, has {free >> 30}")
    g = torch.Generator().manual_seed(1)
    x = torch.cat([torch.rand(2000, 3, generator=g) * 2 - 1,
                   1 - torch.rand(300, 3, generator=g) * 2e-3,  # 300 in the last cell of every grid
                   torch.rand(200, 3, generator=g) * 2e-3 - 1]).to(dev)
    levels, decs = _backward(res, x, 2)
    for r, (used, got, want, grad) in zip(res, levels):
        _close(got, want, r)
        touched = torch.cat([(p != 0).any(1).nonzero()[:, 0] + i * (1 << 24)
                             for i, p in enumerate(grad.split(1 << 24))])
        assert torch.isin(touched, used).all()
    for d in decs:
        for got, want in d:
            _close(got, want, "decoder")


@pytest.mark.parametrize("res", [[4, 64], [64, 4], [3, 33, 2, 5], [40]])
@pytest.mark.parametrize("n", [700, 20000])
def test_levels_in_any_order(dev, res, n):
    """Levels with many pieces per corner (a block per corner) before and after others."""
    g = torch.Generator().manual_seed(n)
    x = (torch.rand(n, 3, generator=g) * 2 - 1).to(dev)
    x[: n // 3] = 0.01 * x[: n // 3] + 0.3  # and many pieces in some corners of the others
    levels, decs = _backward(res, x, 3)
    for r, (_, got, want, _) in zip(res, levels):
        _close(got, want, r)
    for d in decs:
        for got, want in d:
            _close(got, want, "decoder")


@pytest.mark.parametrize("n", [390000, 393216, 400001])
def test_one_sort_or_a_sort_per_level(dev, n):
    """Eight levels: below 393216 queries one sort of all contributions, from there on a sort per
    level, on the same buffers one after the other."""
    res = [4, 2, 8, 16, 64, 32, 1, 24]
    g = torch.Generator().manual_seed(n)
    x = (torch.rand(n, 3, generator=g) * 2 - 1).to(dev)
    levels, decs = _backward(res, x, 4)
    for r, (used, got, want, grad) in zip(res, levels):
        _close(got, want, r)
        assert torch.isin((grad != 0).any(1).nonzero()[:, 0], used).all()
    for d in decs:
        for got, want in d:
            _close(got, want, "decoder")


@pytest.mark.parametrize("num_lods", [6, 7, 8])
@pytest.mark.parametrize("pos_invariant", [True, False])
@pytest.mark.parametrize("n", [500, 20000])
def test_step_of_many_levels(dev, num_lods, pos_invariant, n):
    """n = 20000: a block holds every level's decoder (19 KB each) in LDS; 500: a level per block."""
    net = workloads.make_model(num_lods=num_lods, base_lod=0, pos_invariant=pos_invariant, seed=num_lods, device=dev)
    g = torch.Generator().manual_seed(n)
    with torch.no_grad():
        for l in net.louts:
            l[0].bias.copy_(torch.randn(128, generator=g).sign())
    x, gt = (torch.rand(n, 3, generator=g) * 2 - 1).to(dev), torch.rand(n, 1, generator=g).to(dev)
    want = _grads64(net, x, gt)
    Trainer(net).step_geometry(x, gt)
    for k, p in net.named_parameters():
        _close(p.grad.cpu(), want[k], k)
