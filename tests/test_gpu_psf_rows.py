"""PSF blur at the edges of its row kernel: column counts around its vectors,
chunks and limits, bands inside and beyond LDS, rows without entries and with
more than one batch of them, non-finite voxels, against the FP64 restatement
(rel L2 <= 1e-6, the bar of the PSF tests)."""
import numpy as np
import pytest
import torch

from tests import helpers as H
from tests.test_gpu_psf import _mats

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz", [3, 4, 5, 63, 64, 65, 127, 128, 129, 255, 257, 300, 512, 513])
@pytest.mark.parametrize("band", [(0, 0), (3, 6), None])
def test_columns_and_bands(cuda, nz, band):
    from oracle import psf as OPSF
    from srf_amd.data import Image
    from srf_amd.psf import PSF
    grid = (5, 7, nz)
    xy, z = _mats(grid, 1, nnz_row=33 if nz < 10 else 9, empty_rows=2, band=band)
    x = np.random.default_rng(2).uniform(0.5, 2.0, grid).astype(np.float32)
    p = PSF(xy, z, grid, cuda)
    img = Image(torch.from_numpy(x).to(cuda), (0, 0, 0), (1, 1, 1))
    assert H.rel_l2(p.forward(img).data.cpu().numpy(), OPSF.psf_forward(x, xy, z)) <= 1e-6
    assert H.rel_l2(p.backward(img).data.cpu().numpy(), OPSF.psf_backward(x, xy, z)) <= 1e-6


def test_non_finite_voxels_stay_local(cuda):
    """An infinite voxel reaches the voxels its entries and its band reach, no
    others."""
    from scipy import sparse
    from srf_amd.data import Image
    from srf_amd.psf import PSF
    grid = (6, 6, 37)
    z = np.eye(37) + np.eye(37, k=1) + np.eye(37, k=-1)
    x = np.ones(grid, np.float32)
    x[2, 3, 20] = np.inf
    p = PSF(sparse.eye(36), z, grid, cuda)
    f = p.forward(Image(torch.from_numpy(x).to(cuda), (0, 0, 0), (1, 1, 1))).data.cpu().numpy()
    bad = np.zeros(grid, bool)
    bad[2, 3, 19:22] = True
    assert np.array_equal(~np.isfinite(f), bad)
