"""Span walks and binned scatters of the untiled Siddon ops: set sizes on both
sides of the size rules, image sizes around the tile edges, strided outputs,
rays along axes, faces and diagonals, against the FP64 oracle (rel L2 <= 1e-5,
the bar of every projector op) and captured replays against eager calls."""
import numpy as np
import pytest
import torch

from oracle import lib as O
from srf_amd import _lib, ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rays(n, size, seed):
    """Rays through the box, among them some along an axis, along a voxel face
    and along diagonals, and some that miss."""
    r = np.random.default_rng(seed)
    half = np.asarray(size) / 2
    p = r.uniform(-1.2, 1.2, (n, 3)) * half
    d = r.normal(0, 1, (n, 3))
    d[0::11, 0:2] = 0.0                     # along z
    d[1::11, 1:3] = 0.0                     # along x
    d[2::11] = np.sign(d[2::11])            # diagonals
    p[3::11, 1] = 0.0                       # in the plane y = 0 ...
    d[3::11, 1] = 0.0                       # ... (a voxel face of an even grid)
    d[4::11, 2] *= 1e-7                     # almost in a slice
    d /= np.linalg.norm(d, axis=1)[:, None]
    L = 2.0 * np.linalg.norm(size)
    a, b = p - L * d, p + 0.8 * L * d
    return np.ascontiguousarray(np.vstack([a.T, b.T, r.normal(0, 20, n)[None]]), np.float32)


def _rel(a, b):
    a, b = np.asarray(a, np.float64).ravel(), np.asarray(b, np.float64).ravel()
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("grid", [(17, 16, 9), (16, 33, 8), (40, 24, 20), (5, 64, 3)])
@pytest.mark.parametrize("n", [600, 30_000, 140_000])
@pytest.mark.parametrize("ts2", [400.0, 1.0e6])
def test_ops_against_oracle(grid, n, ts2):
    size = (grid[0] * 2.0, grid[1] * 2.1, grid[2] * 2.5)
    geo = (grid, (0.0, 0.0, 0.0), size)
    lors = _rays(n, size, 3)
    rng = np.random.default_rng(4)
    img = rng.uniform(0.2, 2.0, grid[::-1]).astype(np.float32)
    v = rng.uniform(0.5, 2.0, n).astype(np.float32)
    v[::13] = 0.0
    L, X, V = (torch.from_numpy(a).to(DEV) for a in (lors, img, v))
    p = ops.siddon_projection(L, X, *geo, 6.0, ts2).cpu().numpy()
    assert _rel(p, O.siddon_project(lors, img, *geo, 6.0, ts2, prec="f64")) <= 1e-5
    b = ops.siddon_backprojection(X, L, V, *geo, 6.0, ts2).cpu().numpy()
    assert _rel(b, O.siddon_backproject(lors, v, *geo, 6.0, ts2, prec="f64")) <= 1e-5
    g = v - 1.2
    a = ops.siddon_backprojection_adjoint(X, L, torch.from_numpy(g).to(DEV), *geo, 6.0,
                                          ts2).cpu().numpy()
    assert _rel(a, O.siddon_backproject_adjoint(lors, g, *geo, 6.0, ts2, prec="f64")) <= 1e-5
    m = ops.siddon_maplors(X, *geo, L, V).cpu().numpy()
    assert _rel(m, O.siddon_map(lors, v, *geo, prec="f64")) <= 1e-5
    o = ops.siddon_osem_subset(L, X, *geo, 6.0, ts2)
    q = ops.siddon_backprojection(X, L, torch.from_numpy(p).to(DEV), *geo, 6.0, ts2)
    assert _rel(o.cpu().numpy(), q.cpu().numpy()) <= 1e-6


@pytest.mark.parametrize("strides", [(1, 40, 40 * 24), (24 * 20, 20, 1), (20, 40 * 20, 1)])
def test_strided_output_accumulates(strides):
    grid, size = (40, 24, 20), (80.0, 50.4, 50.0)
    n = 60_000
    lors = _rays(n, size, 7)
    v = np.random.default_rng(8).uniform(0.5, 2.0, n).astype(np.float32)
    L, V = torch.from_numpy(lors).to(DEV), torch.from_numpy(v).to(DEV)
    out = torch.empty_strided(grid, strides, device=DEV).fill_(0.25)
    cg = _lib.make_grid(grid, (0, 0, 0), size, strides)
    _lib.call("srfx_siddon_backproject", L.data_ptr(), n, n, V.data_ptr(), cg, 6.0, 1.0e6,
              out.data_ptr(), _lib.SRFX_ACCUMULATE, torch.cuda.current_stream().cuda_stream)
    ref = O.siddon_backproject(lors, v, grid, (0, 0, 0), size, 6.0, 1.0e6, prec="f64")
    ref = ref.reshape(grid[::-1]).transpose(2, 1, 0) + 0.25
    assert _rel(out.cpu().numpy(), ref) <= 1e-5


def test_captured_call():
    grid, size, n = (40, 24, 20), (80.0, 50.4, 50.0), 60_000
    geo = (grid, (0.0, 0.0, 0.0), size)
    L = torch.from_numpy(_rays(n, size, 9)).to(DEV)
    V = torch.rand(n, device=DEV) + 0.5
    X = torch.empty(grid[::-1], device=DEV)
    eager = ops.siddon_backprojection(X, L, V, *geo, 6.0, 400.0)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.siddon_backprojection(X, L, V, *geo, 6.0, 400.0)
    for _ in range(3):
        out.fill_(-1.0)
        graph.replay()
        torch.cuda.synchronize()
        assert _rel(out.cpu().numpy(), eager.cpu().numpy()) <= 1e-5
