"""The row walk of wide tubes (boxes of more than four voxels): one and several
blocks of columns, images narrower than a block, patches over every image edge,
against the FP64 oracle, the untiled scatter and the whole patch."""
import numpy as np
import pytest
import torch

from oracle import lib as O
from srf_amd import ops
from srf_amd.plan import TorPlan

pytestmark = pytest.mark.gpu
DEV = "cuda"
MODEL = (6.0, 1139.77)


def _events(n, size, seed, slope=1.0):
    r = np.random.default_rng(seed)
    half = np.asarray(size) / 2
    mid = r.uniform(-1.1, 1.1, (n, 3)) * half
    d = np.column_stack([r.uniform(-slope, slope, n), r.uniform(-slope, slope, n), np.ones(n)])
    t = r.uniform(0.5, 1.0, n)[:, None] * size[2]
    p1, p2 = mid - d * t, mid + d * t
    pc = p1 + r.uniform(0.3, 0.7, n)[:, None] * (p2 - p1)
    return np.ascontiguousarray(
        np.vstack([p1.T, p2.T, pc.T, r.uniform(0.7, 1.2, n)[None]]), np.float32)


def _rel(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm())


@pytest.mark.parametrize("grid,pitch,kw,slope", [
    ((33, 11, 25), 2.0, 6.0, 1.0),    # five columns
    ((40, 30, 26), 2.0, 8.0, 1.0),    # six
    ((40, 30, 26), 2.0, 8.0, 2.5),    # steep: some events wider than one block
    ((37, 29, 14), 1.6, 8.0, 1.0),    # eight
    ((41, 40, 13), 1.0, 8.0, 1.0),    # twelve and more
    ((3, 4, 30), 2.0, 8.0, 1.0),      # image narrower than a block
])
@pytest.mark.parametrize("model", [MODEL, (6.0, 1.0e6), (6.0, 0.05)])
def test_row_walk(grid, pitch, kw, slope, model):
    """FP32 weights and sums: 1e-5, the bar of every projector op.  The last model's
    TOF sigma is below the tube's, which turns the weights' exponent positive."""
    size = tuple(g * pitch for g in grid)
    lors = _events(3000, size, 3, slope)
    x = np.random.default_rng(4).uniform(0.5, 1.5, grid[::-1]).astype(np.float32)
    args = (grid, (0.0, 0.0, 0.0), size)
    L, X = torch.from_numpy(lors).to(DEV), torch.from_numpy(x).to(DEV)
    plan = TorPlan(L, *args, kw, False, *model)
    assert plan.walks()[0] == 0
    p = plan.projection(X, op_frame=True)
    untiled = ops.projection(L, X, *args, kw, False, *model, full_patch=True)
    assert _rel(p, untiled) <= 1e-5
    for schedule in (None, (1, 256), (4, 64)):
        assert _rel(ops.projection(L, X, *args, kw, False, *model, schedule=schedule),
                    untiled) <= 1e-5
    ref = torch.from_numpy(O.tor_project(lors, x, *args, kw, False, *model, prec="f64"))
    if model[1] > 1.0:
        assert _rel(p.cpu(), ref.reshape(-1)) <= 1e-5
    b = plan.osem_subset(X)
    d = ops.backprojection(X, L, untiled, *args, *model, kw, False, schedule=(1, 256))
    # an event whose projection lies at the ratio's threshold may fall on either side
    assert _rel(b, d) <= 1e-5
    v = torch.rand(3000, device=DEV) - 0.5
    a = plan.backprojection_adjoint(v)
    d = ops.backprojection_adjoint(X, L, v, *args, *model, kw, False, schedule=(1, 256))
    assert _rel(a, d) <= 1e-5


def test_row_walk_leaves_other_voxels_alone():
    """Voxels outside every tube may hold anything."""
    grid, kw = (30, 30, 20), 8.0
    size = (60.0, 60.0, 40.0)
    lors = _events(40, (20.0, 20.0, 40.0), 9, 0.1)
    L = torch.from_numpy(lors).to(DEV)
    args = (grid, (0.0, 0.0, 0.0), size)
    plan = TorPlan(L, *args, kw, False, *MODEL)
    hit = plan.backprojection_adjoint(torch.ones(40, device=DEV)) > 0
    X = torch.rand(grid[::-1], device=DEV) + 0.5
    want = plan.projection(X, op_frame=True)
    bad = torch.where(hit, X, torch.full_like(X, float("nan")))
    bad[-1, -1, -1] = float("inf") if not bool(hit[-1, -1, -1]) else bad[-1, -1, -1]
    assert torch.equal(plan.projection(bad, op_frame=True), want)
