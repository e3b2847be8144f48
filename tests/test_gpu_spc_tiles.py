"""The single-pass traversal where a wave takes many tiles: its lists kept back until
their place is known, tiles on the depth-first fallback and empty tiles between
them, and a point table off its 8-byte alignment, against the same rays a few
tiles at a time (which the oracle tests cover)."""
import ctypes

import pytest
import torch

from nglod_amd import _lib, workloads
from nglod_amd.spc import SPC
from tests.helpers import full_octree

pytestmark = pytest.mark.gpu

N = 200003  # more tiles of 64 than the GPU has waves for


def _rays(dev):
    o, d = workloads.camera_rays(640, 400, eye=(0.4, 2.2, 2.5), fov=60.0, device="cpu")
    g = torch.Generator().manual_seed(1)
    o, d = o[:N].clone(), d[:N].clone()
    away = torch.rand(N // 64 + 1, generator=g).repeat_interleave(64)[:N] < 0.5
    d[away] = -d[away]  # whole tiles that miss
    return o.to(dev), d.to(dev)


def test_many_tiles_a_wave(dev):
    spc = SPC(torch.from_numpy(full_octree(6)), dev)
    o, d = _rays(dev)
    nug, offs = spc.raytrace(o, d, 6)
    per_tile = torch.bincount((nug[:, 0] // 64).long(), minlength=N // 64 + 1)
    assert (per_tile > 2048).sum() > 100 and (per_tile == 0).sum() > 1000
    base = 0
    for i in range(0, N, 4096):
        a, b = spc.raytrace(o[i:i + 4096].contiguous(), d[i:i + 4096].contiguous(), 6)
        a = a + torch.tensor([i, 0], dtype=torch.int32, device=dev)
        assert torch.equal(nug[base:base + len(a)], a)
        assert torch.equal(offs[i:i + len(b)], b + base)
        base += len(a)
    assert base == len(nug)


def test_points_off_their_alignment(dev):
    spc = SPC(torch.from_numpy(full_octree(4)), dev)
    o, d = _rays(dev)
    o, d = o[:5000].contiguous(), d[:5000].contiguous()
    want, woffs = spc.raytrace(o, d, 4)
    shifted = torch.empty(spc.points.numel() + 1, dtype=torch.int16, device=dev)
    shifted[1:] = spc.points.reshape(-1)
    nug = torch.empty(len(want), 2, dtype=torch.int32, device=dev)
    offs = torch.empty(5001, dtype=torch.int32, device=dev)
    status = torch.empty(2, dtype=torch.int32, device=dev)
    lib = _lib.load()
    ws = torch.empty(int(lib.nglod_spc_raytrace_async_workspace_size(5000)), dtype=torch.uint8, device=dev)
    _lib.check(lib.nglod_spc_raytrace_async(_lib.ptr(spc.octree), _lib.ptr(spc.prefix), shifted.data_ptr() + 2,
                                            ctypes.cast(spc._pyr_c, ctypes.c_void_p), spc.level, _lib.ptr(o),
                                            _lib.ptr(d), 5000, 4, _lib.ptr(nug), len(want), _lib.ptr(offs),
                                            _lib.ptr(status), _lib.ptr(ws), ws.numel(), _lib.stream_of(o)), "raytrace")
    assert torch.equal(nug, want) and torch.equal(offs, woffs)
    assert status.tolist() == [len(want), 0]
