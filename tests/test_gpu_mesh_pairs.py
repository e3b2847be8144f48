"""Signed mesh distances on both sides of the lines between every point against every
triangle and the tree over them, and between the numbers of lanes that share a point:
the oracle's distances and signs, and the same bits for a point in whatever batch.

Tolerance: both sides compute in FP64 and differ by the fused multiply-adds of the
device code, a few 2^-53 of the coordinates' size."""
import numpy as np
import pytest

from nglod_amd import mesh
from oracle import oracle
from tests.test_gpu_mesh_tree import _run, _same, _soup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, nf", [(1, 1), (1, 1280), (3, 1281), (4095, 63), (4096, 64), (4097, 65), (4097, 24),
                                   (4097, 25), (4097, 320), (4097, 321), (4099, 1281), (65536, 20), (65537, 20),
                                   (131072, 12), (131073, 12), (52428, 320), (52429, 320), (262143, 64), (262145, 64)])
def test_both_sides_of_the_lines(dev, n, nf):
    rng = np.random.default_rng(n + nf)
    _same(rng.uniform(-1.3, 1.3, (n, 3)), _soup(rng, nf, 0.3), dev, scale=4.0)


@pytest.mark.parametrize("nf", [320, 400])
def test_degenerate_and_not_finite_in_large_batches(dev, nf):
    """5000 points: 320 triangles one by one, 400 by the tree."""
    rng = np.random.default_rng(2)
    tris = _soup(rng, nf, 0.3)
    tris[10] = tris[10, :1]
    tris[20, 2] = 0.5 * (tris[20, 0] + tris[20, 1])
    tris[30] = np.float32(1e-6) * tris[30]
    pts = rng.uniform(-1.5, 1.5, (5000, 3))
    pts[7, 1], pts[8], pts[9, 0] = np.nan, np.inf, -np.inf
    _same(pts, tris, dev, scale=4.0)
    tris[40, 1, 2] = np.nan
    d32, d64 = _run(pts, tris, dev)
    f32 = tris.astype(np.float32)
    rest = oracle.mesh2sdf(pts.astype(np.float32), np.delete(f32, 40, 0))
    assert np.all(np.abs(d64) <= np.abs(rest) * (1 + 1e-12) + 1.6e-14)
    np.testing.assert_array_equal(np.signbit(d64), np.signbit(oracle.mesh2sdf(pts.astype(np.float32), f32)))


def test_a_point_in_any_batch(dev):
    """A mesh's distances by 64, 4, 2 lanes a point and by the tree: the same bits."""
    V, F = mesh.displaced_icosphere(3, level=2)
    tris = mesh.triangles(V, F)
    pts = np.random.default_rng(0).uniform(-1.1, 1.1, (52429, 3))
    whole = _run(pts, tris, dev)  # 320 triangles x 52429 points: the tree
    for n in (1, 777, 4096, 4097, 52428):
        part = _run(pts[:n], tris, dev)
        for a, b in zip(part, whole):
            np.testing.assert_array_equal(a, b[:n])
    more = np.concatenate([pts, pts, pts])[:131072]
    few = tris[:20]
    whole = _run(np.concatenate([more, more]), few, dev)
    for n in (4096, 65536, 65537, 131072):
        for a, b in zip(_run(more[:n], few, dev), whole):
            np.testing.assert_array_equal(a, b[:n])
