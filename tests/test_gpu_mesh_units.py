"""Signed mesh distances in any units: the boxes of the tree over the triangles keep to
the triangles' size, so a mesh in large units is walked as one in small units is, with
the same distances and signs as the oracle's loop over all triangles.

Tolerance: both sides compute in FP64 and differ by the fused multiply-adds of the
device code, a few 2^-53 of the coordinates' size."""
import numpy as np
import pytest
import torch

from nglod_amd import mesh
from nglod_amd.meshdata import MeshData
from tests.test_gpu_mesh_tree import _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [1e-3, 2e3, 9e3, 1e5, 1e7])
@pytest.mark.parametrize("turned", [False, True])
def test_values(dev, scale, turned):
    """turned: a box with faces at 45 degrees, whose determinants are 0 or rounding."""
    if turned:
        c, s = np.cos(np.pi / 4), np.sin(np.pi / 4)
        V = np.array([[x, y, z] for x in (-.5, .5) for y in (-.4, .4) for z in (-.3, .3)])
        F = np.array([[0, 1, 3], [0, 3, 2], [4, 6, 7], [4, 7, 5], [0, 4, 5], [0, 5, 1], [2, 3, 7], [2, 7, 6],
                      [0, 2, 6], [0, 6, 4], [1, 5, 7], [1, 7, 3]])
        V = V @ np.array([[1, 0, 0], [0, c, -s], [0, s, c]]).T
    else:
        V, F = mesh.displaced_icosphere(3, level=2)
    tris = mesh.triangles(V, F)
    rng = np.random.default_rng(5)
    _same(rng.uniform(-1.1, 1.1, (1500, 3)) * scale, tris * scale, dev, scale=4.0 * scale)


def _ms(f, reps=4):
    f()
    best = []
    for _ in range(reps):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        f()
        b.record()
        torch.cuda.synchronize()
        best.append(a.elapsed_time(b))
    return min(best)


def test_large_units_are_culled(dev):
    """32 times the time in units of 1 / 9000 when nothing is."""
    V, F = mesh.displaced_icosphere(0, level=4)
    ms = []
    for scale in (1.0, 9e3):
        md = MeshData(V * scale, F, dev)
        x = (torch.rand(100000, 3, device=dev, generator=torch.Generator(device=dev).manual_seed(0)) * 2 - 1) * scale
        ms.append(_ms(lambda: md.sdf(x)))
    assert ms[1] < 4 * ms[0], ms
