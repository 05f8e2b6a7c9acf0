"""The scatters' weights one by one: the binned box and row walks of untiled calls
and the row walk of plans are no less precise than the direct scatter."""
import numpy as np
import pytest
import torch

from oracle import lib as O
from srf_amd import ops
from srf_amd.plan import TorPlan

pytestmark = pytest.mark.gpu
DEV = "cuda"
TOF = (6.0, 1139.77)


def _apart(size, pitch, gap, seed):
    """Events nearly along op z whose tubes share no voxel, the TOF centre at the
    far end: TOF exponents up to -10."""
    r = np.random.default_rng(seed)
    x, y = [np.arange(-size[k] / 2 + gap, size[k] / 2 - gap, 2 * gap) for k in (0, 1)]
    x, y = [v.ravel() for v in np.meshgrid(x, y)]
    n = x.size
    x, y = x + r.uniform(-pitch, pitch, n), y + r.uniform(-pitch, pitch, n)
    dx, dy = r.uniform(-1, 1, (2, n)) * pitch
    z = np.full(n, size[2] / 2)
    p1, p2 = np.stack([x, y, -z - 5]), np.stack([x + dx, y + dy, z + 5])
    pc = np.stack([x, y, -z + r.uniform(0, 20, n)])
    return np.vstack([p1, p2, pc, np.ones((1, n))]).astype(np.float32)


def _rms(a, ref):
    """Relative error of the weights, root mean square."""
    a = a.double().cpu().reshape(-1)
    ref = torch.from_numpy(ref).reshape(-1)
    k = ref != 0
    assert bool((a[~k] == 0).all())
    return float((a[k] / ref[k] - 1).square().mean().sqrt())


@pytest.mark.parametrize("pitch,kw", [(2.0, 4.0), (1.6, 4.0), (2.0, 8.0)])
def test_weights_as_precise_as_the_direct_scatter(pitch, kw):
    """The same roundings as the direct scatter's, whose sums hold one term here: the
    error's root mean square over more than 20000 weights is its own to 5 % (half
    a percent of sampling; a TOF exponent summed into the tube's adds 9 to 20 %)."""
    grid = (120, 120, 60)
    size = tuple(g * pitch for g in grid)
    lors = _apart(size, pitch, kw + 2 * pitch, 3)
    m = lors.shape[1]
    args = (grid, (0.0, 0.0, 0.0), size)
    g = np.random.default_rng(4).uniform(0.5, 2.0, m).astype(np.float32)
    ref = O.tor_backproject_adjoint(lors, g, *args, kw, False, *TOF, prec="f64")
    assert (ref != 0).sum() > 20000
    # the size rule of the binned scatters: more events, of value 0
    n = 100_000
    L = torch.from_numpy(np.ascontiguousarray(np.tile(lors, -(-n // m))[:, :n])).to(DEV)
    G = torch.zeros(n, device=DEV)
    G[:m] = torch.from_numpy(g).to(DEV)
    like = torch.empty(grid[::-1], device=DEV)
    direct = _rms(ops.backprojection_adjoint(like, L, G, *args, *TOF, kw, schedule=(1, 256)), ref)
    assert _rms(ops.backprojection_adjoint(like, L, G, *args, *TOF, kw), ref) <= 1.05 * direct
    plan = TorPlan(L[:, :m].contiguous(), *args, kw, False, *TOF)
    assert _rms(plan.backprojection_adjoint(G[:m]), ref) <= 1.05 * direct
    if plan.walks()[0] == 0:
        V = torch.from_numpy(1.0 / g.astype(np.float64)).to(torch.float32).to(DEV)
        back = O.tor_backproject(lors, V.cpu().numpy(), *args, kw, False, *TOF, prec="f64")
        d = _rms(ops.backprojection(like, L[:, :m].contiguous(), V, *args, *TOF, kw, False,
                                    schedule=(1, 256)), back)
        assert _rms(plan.backprojection(V), back) <= 1.05 * d


@pytest.mark.parametrize("n", [361, 200_000])
def test_siddon_tof_weights(n):
    """Values of TOF segments one by one, direct and binned: distance, variance and
    quotient in FP64, then FP32.  Roundings of 2^-24 / sqrt(12) of a value, root mean
    square 1.7e-8 at the bottom of a binade to 3.4e-8 at its top: segment length,
    Gaussian, reciprocal root, their products, weight, bin and scale, eight in all,
    9e-8 at most, and the exponent's two (the quotient and its product with log2 e, up
    to 6.5 of a base-2 exponent: 2^-22 ln 2 / sqrt(3) at most, in the outer third of the
    values), 5e-8 over all: 1.1e-7, with a tenth to spare for the hardware functions'
    ulp.  The quotient in FP32 makes it 1.5e-7."""
    grid, size, ts2 = (120, 120, 100), (240.0, 240.0, 220.0), 400.0
    geo = (grid, (0.0, 0.0, 0.0), size)
    r = np.random.default_rng(3)
    x, y = [np.arange(-size[k] / 2 + 6.0, size[k] / 2 - 6.0, 12.0) for k in (0, 1)]
    x, y = [v.ravel() for v in np.meshgrid(x, y)]  # rays apart: a voxel holds one value
    m = x.size
    x, y = x + r.uniform(-2, 2, m), y + r.uniform(-2, 2, m)
    dx, dy = r.uniform(-2.5, 2.5, (2, m))
    z = np.full(m, size[2] / 2 + 5)
    lors = np.vstack([x - dx, y - dy, -z, x + dx, y + dy, z,
                      r.uniform(-40, 40, m)]).astype(np.float32)
    g = r.uniform(0.5, 2.0, m).astype(np.float32)
    ref = O.siddon_backproject_adjoint(lors, g, *geo, 6.0, ts2, prec="f64")
    assert m == 361 and (ref != 0).sum() > 20000
    L = torch.from_numpy(np.ascontiguousarray(np.tile(lors, -(-n // m))[:, :n])).to(DEV)
    G = torch.zeros(n, device=DEV)
    G[:m] = torch.from_numpy(g).to(DEV)
    like = torch.empty(grid[::-1], device=DEV)
    assert _rms(ops.siddon_backprojection_adjoint(like, L, G, *geo, 6.0, ts2), ref) <= 1.25e-7
