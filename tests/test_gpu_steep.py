"""Events nearly parallel to the slices, against the FP64 oracle."""
import numpy as np
import pytest
import torch

from oracle import lib as O
from srf_amd import ops
from srf_amd.plan import TorPlan

pytestmark = pytest.mark.gpu
DEV = "cuda"
TOF, NO_TOF = (6.0, 1139.77), (6.0, 1.0e6)

# |weight error| of a nearly parallel event: its direction cosines are rounded to
# FP32 (2^-25 of one), which moves d2 = dx^2 + dy^2 - (u . d)^2 by up to
# 4 |d|^2 2^-25; with |d| below the patch's 14 mm and an exponent factor of at most
# 0.5 / sigma^2 = 18 / kw^2 that is 5e-6 (kw 8) to 3e-5 (kw 4), beside the FP32
# weights and sums (1e-5).  A dropped event is an error of its whole share.
TOL = 5e-5


def _flat(n, size, grid, axis, cosine, seed, spread=2.0):
    """n events across the frame along op x (axis 0) or y (1), each crossing one
    slice at the direction cosine `cosine`."""
    r = np.random.default_rng(seed)
    pitch = np.asarray(size) / np.asarray(grid)
    p1 = r.uniform(-0.45, 0.45, (n, 3)) * size
    half = 0.55 * size[axis]
    s = r.integers(0, grid[2], n)
    zs = -size[2] / 2 + (s + 0.5) * pitch[2]
    p1[:, axis] = -half
    p2 = p1.copy()
    p2[:, axis] = half
    p2[:, 1 - axis] += r.uniform(-spread, spread, n)
    # end points either side of the slice's plane, whose coordinate is an exact
    # float: the difference is exact too
    zs = np.round(zs * 64) / 64
    h = np.maximum(np.round(half * cosine * 2 ** 18) / 2 ** 18, 2.0 ** -18)
    p1[:, 2] = zs - h
    p2[:, 2] = zs + h
    pc = p1 + r.uniform(0.3, 0.7, n)[:, None] * (p2 - p1)
    return np.vstack([p1.T, p2.T, pc.T, np.ones((1, n))]).astype(np.float32)


def _fill(n, size, seed):
    """Ordinary events."""
    r = np.random.default_rng(seed)
    half = np.asarray(size) / 2
    mid = r.uniform(-0.9, 0.9, (n, 3)) * half
    d = np.column_stack([r.uniform(-1, 1, n), r.uniform(-1, 1, n), np.ones(n)])
    t = r.uniform(0.5, 1.0, n)[:, None] * size[2]
    p1, p2 = mid - d * t, mid + d * t
    pc = p1 + r.uniform(0.3, 0.7, n)[:, None] * (p2 - p1)
    return np.vstack([p1.T, p2.T, pc.T, np.ones((1, n))]).astype(np.float32)


def _rel(a, b):
    a, b = torch.as_tensor(a).double().reshape(-1).cpu(), torch.as_tensor(b).double().reshape(-1)
    return float((a - b).norm() / b.norm())


@pytest.mark.parametrize("kw", [4.0, 8.0])
@pytest.mark.parametrize("axis", [0, 1])
def test_crossing_on_a_voxel_face(kw, axis):
    """At a direction cosine of 1e-6 the track starts 1e8 voxels away and a crossing
    carries 1e-8 voxel of rounding: the face it lies on (the middle of the frame)
    is the reference's."""
    grid, size = (170, 160, 96), (340.0, 320.0, 192.0)
    args = (grid, (0.0, 0.0, 0.0), size, kw, False, 6.0, 1.0e6)
    lors = _flat(200, size, grid, axis, 1e-6, 3)
    x = np.random.default_rng(4).uniform(0.5, 1.5, grid[::-1]).astype(np.float32)
    L, X = torch.from_numpy(lors).to(DEV), torch.from_numpy(x).to(DEV)
    want = O.tor_project(lors, x, *args, prec="f64").reshape(-1)
    assert _rel(ops.projection(L, X, *args, full_patch=True), want) <= TOL


@pytest.mark.parametrize("axis", [0, 1])
@pytest.mark.parametrize("kw", [4.0, 8.0])
def test_columns_and_rows_beyond_2_to_19(axis, kw):
    """An image of 2^19 + 2^17 columns (rows): the fixed-point crossing holds 2^19 and
    the reference's arithmetic takes the rest."""
    m = (1 << 19) + (1 << 17)
    pitch = 2.0
    grid = (m, 4, 3) if axis == 0 else (4, m, 3)
    size = tuple(g * pitch for g in grid)
    r = np.random.default_rng(6)
    n = 300
    mid = r.uniform(-0.4, 0.4, (n, 3)) * size
    # columns around 0, around 2^19 and to the end
    at = np.concatenate([r.uniform(0, 40, 100), (1 << 19) + r.uniform(-40, 40, 100),
                         m - r.uniform(0, 90000, 100)])
    mid[:, axis] = np.round(((at - m / 2) * pitch) * 16) / 16
    d = r.uniform(-0.7, 0.7, (n, 3))
    d[:, 2] = 1.0
    t = 8.0
    p1, p2 = mid - d * t, mid + d * t
    lors = np.vstack([p1.T, p2.T, mid.T, np.ones((1, n))]).astype(np.float32)
    x = r.uniform(0.5, 1.5, grid[::-1]).astype(np.float32)
    args = (grid, (0.0, 0.0, 0.0), size)
    L, X = torch.from_numpy(lors).to(DEV), torch.from_numpy(x).to(DEV)
    want = O.tor_project(lors, x, *args, kw, False, 6.0, 1.0e6, prec="f64").reshape(-1)
    got = ops.projection(L, X, *args, kw, False, 6.0, 1.0e6).cpu().double().numpy().reshape(-1)
    assert (want > 0).sum() > 250
    # offsets from the crossing are differences of coordinates near 6e5 mm, FP64 to
    # 1e-10 mm: the FP32 weights and sums alone, 1e-5
    assert _rel(got, want) <= 1e-5
    v = np.ones(n, np.float32)
    back = O.tor_backproject(lors, v, *args, kw, False, 6.0, 1.0e6, prec="f64").reshape(-1)
    b = ops.backprojection(X, L, torch.from_numpy(v).to(DEV), *args, 6.0, 1.0e6, kw, False)
    assert _rel(b, back) <= 1e-5


# More voxels than a walk record's 15 bits hold: cosine 6e-5, a span of ~33000 at a
# 4 mm tube, 1e-5: ~200000, 1e-6: ~4e6 (8 mm).  Without TOF there: the TOF exponent
# is a quadratic in the slice with FP64 coefficients, which cancel from
# (pitch slice / cosine)^2, 4e16 mm^2 at 96 slices of 2 mm, of which FP64 keeps 4.
WIDE = [
    (4.0, 0, 6e-5, TOF), (4.0, 1, 6e-5, TOF), (4.0, 0, 1e-5, NO_TOF), (4.0, 1, 1e-5, TOF),
    (5.0, 1, 4e-5, TOF), (8.0, 0, 6e-5, TOF), (8.0, 1, 6e-5, NO_TOF), (8.0, 0, 1e-6, NO_TOF),
    (8.0, 1, 1e-6, NO_TOF),
    # parallel to op y as well: three columns and ~33000 rows
    (4.0, 1, 6e-5, TOF, 0.0), (5.0, 1, 6e-5, NO_TOF, 0.0),
]


@pytest.mark.parametrize("kw,axis,cosine,model,spread", [(w + (2.0,))[:5] for w in WIDE])
def test_flat_events_of_plans(kw, axis, cosine, model, spread):
    grid, size = (40, 36, 24), (80.0, 72.0, 48.0)
    args = (grid, (0.0, 0.0, 0.0), size)
    lors = _flat(200, size, grid, axis, cosine, 3, spread)
    x = np.random.default_rng(4).uniform(0.5, 1.5, grid[::-1]).astype(np.float32)
    L, X = torch.from_numpy(lors).to(DEV), torch.from_numpy(x).to(DEV)
    want = O.tor_project(lors, x, *args, kw, False, *model, prec="f64").reshape(-1)
    assert (want > 0).mean() > 0.9
    plan = TorPlan(L, *args, kw, False, *model)
    assert _rel(plan.projection(X, op_frame=True), want) <= TOL
    assert _rel(ops.projection(L, X, *args, kw, False, *model), want) <= TOL
    v = np.random.default_rng(5).uniform(0.5, 2.0, 200).astype(np.float32)
    V = torch.from_numpy(v).to(DEV)
    back = O.tor_backproject(lors, v, *args, kw, False, *model, prec="f64").reshape(-1)
    assert _rel(plan.backprojection(V), back) <= TOL
    assert _rel(ops.backprojection(X, L, V, *args, *model, kw, False), back) <= TOL


@pytest.mark.parametrize("kw,axis,cosine,model,spread", [(w + (2.0,))[:5] for w in WIDE])
def test_flat_events_in_large_sets(kw, axis, cosine, model, spread):
    """A few among enough ordinary events for the ordered projection and the binned
    scatters."""
    grid, size = (170, 160, 96), (340.0, 320.0, 192.0)
    args = (grid, (0.0, 0.0, 0.0), size)
    n, m = 140_000, 60
    lors = _fill(n, size, 1)
    at = np.sort(np.random.default_rng(2).choice(n, m, replace=False))
    lors[:, at] = _flat(m, size, grid, axis, cosine, 3, spread)
    few = np.ascontiguousarray(lors[:, at])
    x = np.random.default_rng(4).uniform(0.5, 1.5, grid[::-1]).astype(np.float32)
    L, X = torch.from_numpy(lors).to(DEV), torch.from_numpy(x).to(DEV)
    want = O.tor_project(few, x, *args, kw, False, *model, prec="f64").reshape(-1)
    p = ops.projection(L, X, *args, kw, False, *model).reshape(-1)
    assert _rel(p[torch.from_numpy(at).to(DEV)], want) <= TOL
    v = np.random.default_rng(5).uniform(0.5, 2.0, m).astype(np.float32)
    V = torch.zeros(n, device=DEV)
    V[torch.from_numpy(at).to(DEV)] = torch.from_numpy(v).to(DEV)
    back = O.tor_backproject(few, v, *args, kw, False, *model, prec="f64").reshape(-1)
    assert _rel(ops.backprojection(X, L, V, *args, *model, kw, False), back) <= TOL
