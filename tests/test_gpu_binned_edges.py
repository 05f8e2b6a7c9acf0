"""Binned untiled scatters where tiles have remainders, just past the size rule and
far past it, every set checked to run binned, against the direct kernels; Siddon
sets of more than one piece against sums of calls below the rule."""
import numpy as np
import pytest
import torch

from srf_amd import _lib, ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
TOF, NO_TOF = (6.0, 1139.77), (6.0, 1.0e6)


def _rel(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm())


def _events(n, size, seed):
    r = np.random.default_rng(seed)
    half = np.asarray(size) / 2
    mid = r.uniform(-0.9, 0.9, (n, 3)) * half
    d = np.column_stack([r.uniform(-1, 1, n), r.uniform(-1, 1, n), np.ones(n)])
    t = r.uniform(0.5, 1.0, n)[:, None] * size[2]
    p1, p2 = mid - d * t, mid + d * t
    pc = p1 + r.uniform(0.3, 0.7, n)[:, None] * (p2 - p1)
    lors = np.vstack([p1.T, p2.T, pc.T, r.uniform(0.7, 1.2, n)[None]]).astype(np.float32)
    return torch.from_numpy(np.ascontiguousarray(lors)).to(DEV), torch.from_numpy(
        r.uniform(0.5, 2.0, n).astype(np.float32)).to(DEV)


def _first_binned(grid, size, model):
    """The smallest number of events that runs binned."""
    lo, hi = 0, 1 << 24
    while hi - lo > 1:
        mid = (lo + hi) // 2
        lo, hi = (lo, mid) if _lib.tor_scatter_binned(mid, grid, size, model) else (mid, hi)
    return hi


# one voxel past every tile edge, exactly one tile, several, one voxel less and
# thinner than a tile, for each walk (3 x 3 and 4 x 4 boxes, rows)
GRIDS = [(33, 11, 13), (32, 10, 12), (64, 20, 24), (31, 9, 11), (200, 3, 14), (5, 64, 25)]


@pytest.mark.parametrize("grid", GRIDS)
@pytest.mark.parametrize("pitch,kw,model", [(2.0, 4.0, TOF), (1.6, 4.0, NO_TOF), (2.0, 8.0, TOF)])
@pytest.mark.parametrize("factor", [1.0, 2.3])
def test_tile_edges(grid, pitch, kw, model, factor):
    """FP64 sums per tile, then one FP32 atomic a voxel and chunk, against FP32 atomics
    alone: below 1e-5, the bar of every projector op."""
    size = tuple(g * pitch for g in grid)
    m = _lib.make_tor_model(kw, False, *model)
    n = int(_first_binned(grid, size, m) * factor)
    assert _lib.tor_scatter_binned(n, grid, size, m) and n < 1_200_000
    lors, v = _events(n, size, 7)
    like = torch.empty(grid[::-1], device=DEV)
    args = (grid, (0.0, 0.0, 0.0), size)
    direct = dict(schedule=(1, 256))
    b = ops.backprojection(like, lors, v, *args, *model, kw, False)
    d = ops.backprojection(like, lors, v, *args, *model, kw, False, **direct)
    assert bool((d > 0).any()) and _rel(b, d) <= 1e-5
    g = v - 1.2
    b = ops.backprojection_adjoint(like, lors, g, *args, *model, kw)
    d = ops.backprojection_adjoint(like, lors, g, *args, *model, kw, **direct)
    assert _rel(b, d) <= 1e-5
    x = torch.rand(grid[::-1], device=DEV) + 0.5
    b = ops.osem_subset(lors, x, *args, kw, False, *model)
    d = ops.osem_subset(lors, x, *args, kw, False, *model, **direct)
    assert _rel(b, d) <= 1e-5
    n = int(_first_binned(grid, size, _lib.make_tor_model(kw, False, *NO_TOF)) * factor)
    n = min(n, lors.shape[1])
    if _lib.tor_scatter_binned(n, grid, size, _lib.make_tor_model(kw, False, *NO_TOF)):
        rows = torch.cat([lors[0:6, :n], lors[9:10, :n]]).contiguous()
        b = ops.maplors(like, *args, rows, v[:n], kw)
        d = ops.maplors(like, *args, rows, v[:n], kw, **direct)
        assert _rel(b, d) <= 1e-5


def _rays(n, size, seed):
    r = np.random.default_rng(seed)
    half = np.asarray(size) / 2
    p = r.uniform(-1.1, 1.1, (n, 3)) * half
    d = r.normal(0, 1, (n, 3))
    d[::11, 0:2] = 0.0
    d[1::11, 1:3] = 0.0
    d /= np.linalg.norm(d, axis=1)[:, None]
    L = 2.0 * np.linalg.norm(size)
    a, b = p - L * d, p + 0.8 * L * d
    return torch.from_numpy(np.ascontiguousarray(
        np.vstack([a.T, b.T, r.normal(0, 20, n)[None]]), np.float32)).to(DEV)


@pytest.mark.parametrize("n", [(1 << 19) + 1, 1_300_001])
@pytest.mark.parametrize("ts2", [400.0, 1.0e6])
def test_siddon_pieces(n, ts2):
    """Two and three pieces of at most 2^19 rays (their own offsets into rows and
    values, state and projections used again) against direct calls over parts below
    the rule, summed in FP64: the direct sums' FP32 rounding, 1e-5."""
    grid, size = (33, 17, 9), (66.0, 35.7, 22.5)
    geo = (grid, (0.0, 0.0, 0.0), size)
    part = 60_000
    assert _lib.siddon_scatter_binned(n, grid, size, 6.0, ts2)
    assert not _lib.siddon_scatter_binned(part, grid, size, 6.0, ts2)
    L = _rays(n, size, 3)
    X = torch.rand(grid[::-1], device=DEV) + 0.5
    V = torch.rand(n, device=DEV) + 0.5
    V[::13] = 0.0
    G = V - 0.9

    def parts(f):
        out = torch.zeros(grid[::-1], dtype=torch.float64, device=DEV)
        for a in range(0, n, part):
            out += f(L[:, a:a + part].contiguous(), slice(a, a + part)).double()
        return out

    assert _rel(ops.siddon_backprojection(X, L, V, *geo, 6.0, ts2),
                parts(lambda l, s: ops.siddon_backprojection(X, l, V[s], *geo, 6.0, ts2))) <= 1e-5
    assert _rel(ops.siddon_backprojection_adjoint(X, L, G, *geo, 6.0, ts2),
                parts(lambda l, s: ops.siddon_backprojection_adjoint(X, l, G[s], *geo, 6.0,
                                                                     ts2))) <= 1e-5
    assert _rel(ops.siddon_maplors(X, *geo, L, V),
                parts(lambda l, s: ops.siddon_maplors(X, *geo, l, V[s]))) <= 1e-5
    assert _rel(ops.siddon_osem_subset(L, X, *geo, 6.0, ts2),
                parts(lambda l, s: ops.siddon_osem_subset(l, X, *geo, 6.0, ts2))) <= 1e-5


@pytest.mark.parametrize("kw", [4.0, 5.0, 8.0])
def test_sets_that_do_not_fit(kw):
    """Lines far from the slice axis list more tiles than the array holds: every pass
    after the count returns and the direct scatter runs, also in the OSEM pass."""
    grid, size, n = (200, 60, 24), (400.0, 120.0, 48.0), 60_000
    r = np.random.default_rng(5)
    mid = r.uniform(-0.9, 0.9, (n, 3)) * np.asarray(size) / 2
    d = np.column_stack([40.0 * r.choice([-1, 1], n), r.uniform(-1, 1, n), np.ones(n)])
    t = r.uniform(0.5, 1.0, n)[:, None] * size[2]
    p1, p2 = mid - d * t, mid + d * t
    pc = p1 + r.uniform(0.3, 0.7, n)[:, None] * (p2 - p1)
    lors = torch.from_numpy(np.ascontiguousarray(
        np.vstack([p1.T, p2.T, pc.T, np.ones((1, n))]), np.float32)).to(DEV)
    v = torch.rand(n, device=DEV) + 0.5
    x = torch.rand(grid[::-1], device=DEV) + 0.5
    args = (grid, (0.0, 0.0, 0.0), size)
    assert _lib.tor_scatter_binned(n, grid, size, _lib.make_tor_model(kw, False, *NO_TOF))
    direct = dict(schedule=(1, 256))
    b = ops.backprojection(x, lors, v, *args, *NO_TOF, kw, False)
    assert _rel(b, ops.backprojection(x, lors, v, *args, *NO_TOF, kw, False, **direct)) <= 1e-5
    b = ops.osem_subset(lors, x, *args, kw, False, *NO_TOF)
    assert _rel(b, ops.osem_subset(lors, x, *args, kw, False, *NO_TOF, **direct)) <= 1e-5
