"""Crossing points where the fixed-point split of a slice's crossing can go
wrong: on and beside voxel boundaries, left of and below the grid (the
reference's cast truncates towards zero), and many grids away."""
import numpy as np
import pytest
import torch

from oracle import lib as O
from srf_amd import ops

pytestmark = pytest.mark.gpu
GRID, CENTER, SIZE, KW = (24, 20, 16), (0.0, 0.0, 0.0), (48.0, 40.0, 32.0), 4.0


def _lors(xs, ys, slopes, far=40.0, z=0.0):
    """Lines through (x, y, z) with the given slopes."""
    x, y, a, b = [v.ravel() for v in np.meshgrid(xs, ys, slopes, slopes, indexing="ij")]
    rows = np.stack([x - a * far, y - b * far, np.full_like(x, z - far), x + a * far, y + b * far,
                     np.full_like(x, z + far), x, y, np.full_like(x, z), np.ones_like(x)])
    return np.ascontiguousarray(rows, np.float32)


CASES = {
    # voxel boundaries lie at even coordinates; FP32 rows resolve 2^-22 near 10
    "boundary": _lors(np.array([-24.0, -2.0, 0.0, 10.0, 24.0])[:, None] +
                      np.array([0.0, 1e-6, -1e-6, 1e-4, -1e-4]), [0.0, 2.0 + 1e-6, -20.0],
                      [0.0, 1e-7, 0.5]),
    # within two voxels outside every edge
    "outside": _lors([-28.0, -26.5, -25.0, -24.2, 24.2, 25.9, 27.0], [-23.9, -20.1, 21.0],
                     [0.0, 0.05, -0.3]),
    # inside the grid on the slice at z = 1, far beyond it on its neighbours, and
    # beyond it on all
    "far": np.ascontiguousarray(np.vstack([
        _lors([0.0, 3.3], [1.7], [3.0e3, 2.0e6, -7.0e6], far=2.5, z=1.0).T,
        _lors([1.0e6, -1.0e6, 3.0e8], [5.0e5, -4.0e7], [0.0, 0.4]).T]).T, np.float32),
}


@pytest.mark.parametrize("name", CASES)
@pytest.mark.parametrize("model", [(6.0, 1139.77), (6.0, 1.0e6)])
def test_crossings_match_oracle(cuda, name, model):
    """Counts are exact; sums agree to the 1e-5 of every projector op."""
    lors = CASES[name]
    t = torch.from_numpy(lors).to(cuda)
    rng = np.random.default_rng(1)
    image = rng.uniform(0.5, 1.5, GRID[::-1]).astype(np.float32)
    geo = (GRID, CENTER, SIZE)
    per, tot = ops.count_nnz(t, *geo, KW)
    ref_per = np.asarray(O.tor_count(lors, *geo, KW, False))
    assert np.array_equal(per.cpu().numpy(), ref_per.astype(per.cpu().numpy().dtype))
    if name == "far" and model[1] < 1e5:
        return  # the TOF exponent's expansion over slices is no good at slopes of 1e6
    ref = np.asarray(O.tor_project(lors, image, *geo, KW, False, *model, prec="f64")).ravel()
    for schedule in (None, (1, 256), (4, 64)):
        p = ops.projection(t, torch.from_numpy(image).to(cuda), *geo, KW, False, *model,
                           schedule=schedule).cpu().numpy()
        assert np.all(np.abs(p - ref) <= 1e-5 * np.abs(ref) + 1e-9)
    v = rng.uniform(0.5, 2.0, lors.shape[1]).astype(np.float32)
    like = torch.empty(GRID[::-1], device=cuda)
    b = ops.backprojection(like, t, torch.from_numpy(v).to(cuda), *geo, *model, KW, False)
    rb = np.asarray(O.tor_backproject(lors, v, *geo, KW, False, *model, prec="f64")).ravel()
    d = b.cpu().numpy().ravel() - rb
    assert np.linalg.norm(d) <= 1e-5 * max(np.linalg.norm(rb), 1e-9)
