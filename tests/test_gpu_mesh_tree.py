"""nglod_mesh2sdf_f64 walks a tree over the triangles instead of all of them:
the same distances and signs as the oracle's loop, at the tree's and the
sort's edges (1, 8, 8 + 1, 64 + 1 triangles; part-filled waves, a tile of the
sort and one more), on meshes with no structure, and with degenerate
triangles, NaN vertices and points that are not finite.

Tolerance: both sides compute in FP64 and differ by the fused multiply-adds
of the device code, a few 2^-53 of the coordinates' size."""
import numpy as np
import pytest
import torch

from nglod_amd import _lib, mesh
from oracle import oracle

pytestmark = pytest.mark.gpu


def _run(pts, tris, dev, ordered=True):
    lib = _lib.load()
    p = torch.from_numpy(np.ascontiguousarray(pts, dtype=np.float32)).to(dev)
    m = torch.from_numpy(np.ascontiguousarray(tris, dtype=np.float32)).to(dev)
    n, nf = p.shape[0], m.shape[0]
    size = lib.nglod_mesh2sdf_ordered_workspace_size(n, nf) if ordered else lib.nglod_mesh2sdf_workspace_size(nf)
    ws = torch.empty(size, dtype=torch.uint8, device=dev)
    d32 = torch.full((n,), 7.0, device=dev)
    d64 = torch.full((n,), 7.0, dtype=torch.float64, device=dev)
    _lib.check(lib.nglod_mesh2sdf_f64(_lib.ptr(p), n, _lib.ptr(m), nf, _lib.ptr(d32), _lib.ptr(d64), _lib.ptr(ws),
                                      ws.numel(), _lib.stream_of(p)), "nglod_mesh2sdf_f64")
    return d32.cpu().numpy(), d64.cpu().numpy()


def _same(pts, tris, dev, scale=1.0, ordered=True):
    d32, d64 = _run(pts, tris, dev, ordered)
    want = oracle.mesh2sdf(pts.astype(np.float32), tris.astype(np.float32))
    np.testing.assert_array_equal(np.signbit(d64), np.signbit(want))
    np.testing.assert_allclose(d64, want, rtol=1e-12, atol=4e-15 * scale)
    np.testing.assert_array_equal(d32, d64.astype(np.float32))


def _soup(rng, nf, size):
    return rng.uniform(-1, 1, (nf, 1, 3)) + rng.normal(0, size, (nf, 3, 3))


@pytest.mark.parametrize("nf", [1, 7, 8, 9, 64, 65, 513, 4097])
@pytest.mark.parametrize("ordered", [True, False])
def test_triangle_soup(dev, nf, ordered):
    rng = np.random.default_rng(nf)
    for size in (0.02, 0.8):
        _same(rng.uniform(-1.3, 1.3, (700, 3)), _soup(rng, nf, size), dev, scale=4.0, ordered=ordered)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 257, 4096, 4097, 20001])
def test_point_counts(dev, n):
    V, F = mesh.displaced_icosphere(3, level=2)
    rng = np.random.default_rng(n)
    _same(rng.uniform(-1.1, 1.1, (n, 3)), mesh.triangles(V, F), dev)


@pytest.mark.parametrize("scale", [1e-2, 1.0, 300.0])
@pytest.mark.parametrize("shift", [0.0, 5.0])
def test_closed_concave_mesh(dev, scale, shift):
    """Two nested spheres and a far one: points between the shells, in the
    hollow and in the gap outside, some of them on the surface's vertices."""
    V, F = mesh.icosphere(2)
    T = mesh.triangles(V, F)
    tris = np.concatenate([T, 0.4 * T[:, ::-1], 0.3 * T + [1.6, 0.2, 0.0]]) * scale + shift * scale
    rng = np.random.default_rng(1)
    pts = np.concatenate([rng.uniform(-1.2, 2.0, (3000, 3)) * scale + shift * scale, tris[::50, 0]])
    # vertices sit on ties of the line test: compare their distance only
    d32, d64 = _run(pts, tris, dev)
    want = oracle.mesh2sdf(pts.astype(np.float32), tris.astype(np.float32))
    np.testing.assert_array_equal(np.signbit(d64[:3000]), np.signbit(want[:3000]))
    np.testing.assert_allclose(np.abs(d64), np.abs(want), rtol=1e-12, atol=4e-15 * 8 * scale)


def test_degenerate_and_not_finite(dev):
    rng = np.random.default_rng(2)
    tris = _soup(rng, 100, 0.3)
    tris[10] = tris[10, :1]                       # a point
    tris[20, 2] = 0.5 * (tris[20, 0] + tris[20, 1])  # about a line
    tris[30] = np.float32(1e-6) * tris[30]        # no stab determinant above the threshold
    pts = rng.uniform(-1.5, 1.5, (500, 3))
    _same(pts, tris, dev, scale=4.0)
    # points that are not finite: no distance, never inside
    pts[7, 1] = np.nan
    pts[8] = np.inf
    pts[9, 0] = -np.inf
    _same(pts, tris, dev, scale=4.0)
    # A triangle with a NaN vertex is looked at for every point.  Whether it
    # adds to the distance hangs on the signs of NaNs, but the other triangles'
    # distance bounds it; its lines' t is NaN, a hit behind the point.
    tris[40, 1, 2] = np.nan
    d32, d64 = _run(pts, tris, dev)
    f32 = tris.astype(np.float32)
    rest = oracle.mesh2sdf(pts.astype(np.float32), np.delete(f32, 40, 0))
    assert np.all(np.abs(d64) <= np.abs(rest) * (1 + 1e-12) + 1.6e-14)
    np.testing.assert_array_equal(np.signbit(d64), np.signbit(oracle.mesh2sdf(pts.astype(np.float32), f32)))


def test_all_triangles_equal(dev):
    rng = np.random.default_rng(4)
    tris = np.repeat(_soup(rng, 1, 0.5), 300, 0)
    _same(rng.uniform(-1, 1, (300, 3)), tris, dev, scale=4.0)
