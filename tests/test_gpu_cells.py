"""The cell-by-cell gather of spatially ordered FP32 queries (and the radix sort
that orders them) gives the bits of the input-order kernel: part-filled waves
and tiles, one cell for all points, points of many cells, cells on the box's
faces, grids of one cell, tiles of the sort, and grids with NaN and infinities."""
import pytest
import torch

from nglod_amd import workloads

pytestmark = pytest.mark.gpu


def _same(net, x, lod):
    a = net.sdf_hip(x, lod, ordered=False)
    b = net.sdf_hip(x, lod, ordered=True)
    assert torch.equal(a.view(torch.int32), b.view(torch.int32))
    return a


@pytest.mark.parametrize("n", [1, 31, 32, 33, 63, 64, 65, 100, 4096, 4097, 12289, 200001])
@pytest.mark.parametrize("pos_invariant", [True, False])
def test_sizes(dev, n, pos_invariant):
    net = workloads.make_model(num_lods=5, pos_invariant=pos_invariant, seed=1, device=dev)
    g = torch.Generator().manual_seed(n)
    x = (torch.rand(n, 3, generator=g) * 2.4 - 1.2).to(dev)  # some outside the box
    for lod in (0, 2, 4):
        _same(net, x, lod)


@pytest.mark.parametrize("base_lod", [0, 1])
@pytest.mark.parametrize("spread", [0.0, 1e-4, 0.02, 0.3])
def test_clusters(dev, spread, base_lod):
    """From one point repeated to a cluster of many finest cells."""
    net = workloads.make_model(num_lods=5, base_lod=base_lod, seed=2, device=dev)
    g = torch.Generator().manual_seed(3)
    for centre in (-1.0, 0.25, 0.3, 1.0):
        x = (torch.rand(3001, 3, generator=g) * spread + centre).to(dev)
        for lod in (0, 4):
            _same(net, x, lod)


def test_positions_that_are_not_finite(dev):
    net = workloads.make_model(num_lods=4, seed=4, device=dev)
    x = torch.rand(1000, 3, device=dev) * 2 - 1
    x[::7, 0] = float("nan")
    x[3::11, 1] = float("inf")
    x[5::13, 2] = -float("inf")
    _same(net, x, 3)


def test_non_finite_cells_stay_with_their_queries(dev):
    """A NaN, an infinity and the largest finite values in a few corners: only
    the points of the cells around them see these."""
    net = workloads.make_model(num_lods=4, seed=5, device=dev)
    with torch.no_grad():
        fm = net.features[3].fm
        fm[0, :, 3, 4, 5] = float("nan")
        fm[0, 7, 20, 20, 20] = float("inf")
        net.features[1].fm[0, 0, 0, 0, 0] = 3.4e38
    x = torch.rand(60000, 3, device=dev) * 2 - 1
    y = _same(net, x, 3)
    assert 0 < (~torch.isfinite(y)).sum().item() < 600
