"""Binned untiled scatters: event counts around the size rule, frames around
the tile edges, both flush orders, strided outputs, sets that do not fit the
listing array, against the direct kernels (a named schedule) and the oracle."""
import numpy as np
import pytest
import torch

from oracle import lib as O
from srf_amd import _lib, ops, physics, preprocess

pytestmark = pytest.mark.gpu
DEV = "cuda"
MODEL = (6.0, 1139.77)


def _events(n, size, seed, steep=False):
    """Lines through the frame with slopes up to 45 degrees in both in-slice
    axes (steep: mostly along op x, which lists far more tiles)."""
    r = np.random.default_rng(seed)
    half = np.asarray(size) / 2
    mid = r.uniform(-0.9, 0.9, (n, 3)) * half
    d = np.column_stack([r.uniform(-1, 1, n), r.uniform(-1, 1, n), np.ones(n)])
    if steep:
        d[:, 0] = 40.0 * np.sign(d[:, 0])
    t = r.uniform(0.5, 1.0, n)[:, None] * size[2]
    p1, p2 = mid - d * t, mid + d * t
    pc = p1 + r.uniform(0.3, 0.7, n)[:, None] * (p2 - p1)
    lors = np.ascontiguousarray(
        np.vstack([p1.T, p2.T, pc.T, r.uniform(0.7, 1.2, n)[None]]), np.float32)
    return torch.from_numpy(lors).to(DEV), torch.from_numpy(
        r.uniform(0.5, 2.0, n).astype(np.float32)).to(DEV)


def _rel(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm())


@pytest.mark.parametrize("grid,pitch,kw,n", [
    ((33, 11, 13), 2.0, 4.0, 50_000),     # one voxel past every tile edge, 3 x 3 box
    ((32, 10, 12), 2.0, 4.0, 50_000),     # exactly one tile
    ((64, 40, 25), 1.6, 4.0, 30_000),     # 4 x 4 box
    ((70, 50, 31), 2.0, 8.0, 9_000),      # chord walks
    ((200, 3, 5), 2.0, 4.0, 70_000),      # thin frame
    ((64, 64, 48), 2.0, 4.0, 600_001),    # two pieces, odd split
])
def test_binned_scatters_match_direct(grid, pitch, kw, n):
    """Same weights, FP64 sums per tile then FP32 atomics against FP32 atomics
    alone: the difference is the direct sums' rounding, below 1e-5 (the bar of
    every projector op)."""
    size = tuple(g * pitch for g in grid)
    lors, v = _events(n, size, 7)
    like = torch.empty(grid[::-1], device=DEV)
    args = (grid, (0.0, 0.0, 0.0), size)
    for geo in (False, True):
        b = ops.backprojection(like, lors, v, *args, *MODEL, kw, geo)
        d = ops.backprojection(like, lors, v, *args, *MODEL, kw, geo, schedule=(1, 256))
        assert _rel(b, d) <= 1e-5
    g = v - 1.2  # signed
    b = ops.backprojection_adjoint(like, lors, g, *args, *MODEL, kw)
    d = ops.backprojection_adjoint(like, lors, g, *args, *MODEL, kw, schedule=(1, 256))
    assert _rel(b, d) <= 1e-5
    rows = torch.cat([lors[0:6], lors[9:10]]).contiguous()
    b = ops.maplors(like, *args, rows, v, kw)
    d = ops.maplors(like, *args, rows, v, kw, schedule=(1, 256))
    assert _rel(b, d) <= 1e-5
    x = torch.rand(grid[::-1], device=DEV) + 0.5
    b = ops.osem_subset(lors, x, *args, kw, False, *MODEL)
    d = ops.osem_subset(lors, x, *args, kw, False, *MODEL, schedule=(1, 256))
    assert _rel(b, d) <= 1e-5


def test_binned_against_oracle():
    grid, size, kw = (40, 30, 26), (80.0, 60.0, 57.2), 4.0
    lors, v = _events(60_000, size, 3)
    like = torch.empty(grid[::-1], device=DEV)
    b = ops.backprojection(like, lors, v, grid, (0, 0, 0), size, *MODEL, kw, False)
    ref = O.tor_backproject(lors.cpu().numpy(), v.cpu().numpy(), grid, (0, 0, 0), size, kw, False,
                            *MODEL, prec="f64")
    assert _rel(b.cpu().reshape(-1), torch.from_numpy(ref).reshape(-1)) <= 1e-5


@pytest.mark.parametrize("axis", ["x", "y", "z"])
def test_binned_strided_accumulate(axis):
    """World-layout output of every axis group, added onto what is there."""
    shape = (45, 37, 29)
    pitch = (2.0, 2.1, 2.2)
    size = [s * p for s, p in zip(shape, pitch)]
    out = torch.rand(shape, device=DEV)
    g, c, sz, st = physics.group_frame(shape, (0, 0, 0), size, out.stride(), axis)
    lors, v = _events(80_000, sz, 11)
    cg, m = _lib.make_grid(g, c, sz, st), _lib.make_tor_model(4.0, False, *MODEL)
    outs = []
    for flags in (0, 1 << 4):  # default, one lane per event (direct)
        o = out.clone()
        _lib.call("srfx_tor_backproject", lors.data_ptr(), lors.shape[1], lors.shape[1],
                  v.data_ptr(), cg, m, o.data_ptr(), _lib.SRFX_ACCUMULATE | flags,
                  torch.cuda.current_stream().cuda_stream)
        outs.append(o)
    assert _rel(outs[0], outs[1]) <= 1e-5


def test_binned_set_that_does_not_fit():
    """Lines far from the slice axis list more tiles than the array holds: the
    direct scatter runs instead."""
    grid, size = (200, 60, 24), (400.0, 120.0, 48.0)
    lors, v = _events(60_000, size, 5, steep=True)
    like = torch.empty(grid[::-1], device=DEV)
    args = (grid, (0.0, 0.0, 0.0), size, 6.0, 1e6, 4.0, False)
    b = ops.backprojection(like, lors, v, *args)
    d = ops.backprojection(like, lors, v, *args, schedule=(1, 256))
    assert _rel(b, d) <= 1e-5


def test_special_values_and_capture():
    """Values that add nothing (NaN, 0, below the threshold) and a captured
    call, which keeps the direct kernels."""
    grid, size = (40, 40, 36), (80.0, 80.0, 72.0)
    lors, v = _events(40_000, size, 9)
    v[::7] = 0.0
    v[1::7] = float("nan")
    v[2::7] = 1e-8
    like = torch.empty(grid[::-1], device=DEV)
    args = (grid, (0.0, 0.0, 0.0), size, *MODEL, 4.0, False)
    b = ops.backprojection(like, lors, v, *args)
    d = ops.backprojection(like, lors, v, *args, schedule=(1, 256))
    assert bool(torch.isfinite(b).all()) and _rel(b, d) <= 1e-5
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        c = ops.backprojection(like, lors, v, *args)
    for _ in range(3):
        c.fill_(-1.0)
        graph.replay()
        torch.cuda.synchronize()
        assert _rel(c, d) <= 1e-5


def test_adjoint_of_values_far_from_one():
    """A power-of-two factor of one event's value scales every weight exactly
    (the tile sums one event in FP64, each voxel is flushed once)."""
    grid, size = (40, 40, 36), (80.0, 80.0, 72.0)
    lors, _ = _events(40_000, size, 13)
    like = torch.empty(grid[::-1], device=DEV)
    args = (grid, (0.0, 0.0, 0.0), size, *MODEL, 4.0, False)
    g = torch.zeros(40_000, device=DEV)
    g[1234] = -1.25
    a = ops.backprojection_adjoint(like, lors, g, *args)
    b = ops.backprojection_adjoint(like, lors, g * 2.0 ** -90, *args)
    assert bool((a < 0).any()) and torch.equal(a, b * 2.0 ** 90)


def test_negative_tof_bin():
    """The weights' sign follows the TOF bin's, as in the direct scatter."""
    grid, size = (40, 40, 36), (80.0, 80.0, 72.0)
    lors, v = _events(40_000, size, 17)
    like = torch.empty(grid[::-1], device=DEV)
    args = (grid, (0.0, 0.0, 0.0), size, -6.0, MODEL[1], 4.0, False)
    b = ops.backprojection(like, lors, v, *args)
    d = ops.backprojection(like, lors, v, *args, schedule=(1, 256))
    assert bool((d < 0).any()) and _rel(b, d) <= 1e-5
