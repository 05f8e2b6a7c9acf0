"""Events nearly parallel to the slices, against the FP64 oracle."""
import numpy as np
import pytest
import torch

from oracle import lib as O
from srf_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"

# |weight error| of a nearly parallel event: its direction cosines are rounded to
# FP32 (2^-25 of one), which moves d2 = dx^2 + dy^2 - (u . d)^2 by up to
# 4 |d|^2 2^-25; with |d| below the patch's 14 mm and an exponent factor of at most
# 0.5 / sigma^2 = 18 / kw^2 that is 5e-6 (kw 8) to 3e-5 (kw 4), beside the FP32
# weights and sums (1e-5).  A dropped event is an error of its whole share.
TOL = 5e-5


def _flat(n, size, grid, axis, cosine, seed):
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
    p2[:, 1 - axis] += r.uniform(-2, 2, n)
    # end points either side of the slice's plane, whose coordinate is an exact
    # float: the difference is exact too
    zs = np.round(zs * 64) / 64
    h = np.maximum(np.round(half * cosine * 2 ** 18) / 2 ** 18, 2.0 ** -18)
    p1[:, 2] = zs - h
    p2[:, 2] = zs + h
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
