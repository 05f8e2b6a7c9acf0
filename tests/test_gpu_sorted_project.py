"""Projections of large event sets through the locality order: against the
kernels that walk the events as they come (a named schedule), at the rule's
lower edges, over two pieces, for every walk, strided images and events that
cross nothing."""
import numpy as np
import pytest
import torch

from srf_amd import _lib, ops, physics

pytestmark = pytest.mark.gpu
DEV = "cuda"
TOF = (6.0, 1139.77)
NO_TOF = (6.0, 1.0e6)


def _events(n, size, seed):
    r = np.random.default_rng(seed)
    half = np.asarray(size) / 2
    mid = r.uniform(-1.2, 1.2, (n, 3)) * half
    d = np.column_stack([r.uniform(-1, 1, n), r.uniform(-1, 1, n), np.ones(n)])
    t = r.uniform(0.3, 1.0, n)[:, None] * size[2]
    p1, p2 = mid - d * t, mid + d * t
    pc = p1 + r.uniform(0.2, 0.8, n)[:, None] * (p2 - p1)
    lors = np.ascontiguousarray(
        np.vstack([p1.T, p2.T, pc.T, r.uniform(0.7, 1.2, n)[None]]), np.float32)
    lors[5, ::97] = lors[2, ::97]  # no slice crossed
    lors[0, ::101] = 1.0e6         # far outside
    lors[3, 5] = np.inf
    return torch.from_numpy(lors).to(DEV)


def _check(a, b):
    """Sums of at most ~2000 terms in FP32, all of one sign: each within
    2000 2^-24 = 1.2e-4 of its value."""
    ok = torch.isclose(a, b, rtol=1.2e-4, atol=1e-6, equal_nan=True)
    assert bool(ok.all()), (a[~ok][:5], b[~ok][:5])


@pytest.mark.parametrize("grid,pitch,kw,n,model", [
    ((190, 120, 112), 2.0, 4.0, 131_073, TOF),      # 3 x 3 box, first sorted size
    ((190, 120, 112), 2.0, 4.0, 140_001, NO_TOF),
    ((190, 120, 112), 1.5, 4.0, 131_137, TOF),      # 4 x 4 box
    ((160, 140, 120), 2.0, 12.0, 131_073, TOF),     # row walks
    ((190, 120, 112), 4.0, 4.0, (1 << 20) + 77, TOF),  # two pieces
])
def test_sorted_projection_matches(grid, pitch, kw, n, model):
    size = tuple(g * pitch for g in grid)
    lors = _events(n, size, 3)
    image = torch.rand(grid[::-1], device=DEV) + 0.1
    args = (grid, (0.0, 0.0, 0.0), size, kw)
    for geo in (False, True):
        a = ops.projection(lors, image, *args, geo, *model)
        b = ops.projection(lors, image, *args, geo, *model, schedule=(1, 256))
        assert float((b > 0).float().mean()) > 0.5
        _check(a, b)
        # whichever events share a wave, an event's sum is the same
        assert torch.equal(a, ops.projection(lors, image, *args, geo, *model))


@pytest.mark.parametrize("axis", ["x", "y", "z"])
def test_sorted_projection_strided_image(axis):
    """The world image read with an axis group's strides; rows of the event
    array further apart than the events."""
    shape = (140, 130, 150)
    size = [2.0 * s for s in shape]
    image = torch.rand(shape, device=DEV)
    g, c, sz, st = physics.group_frame(shape, (0, 0, 0), size, image.stride(), axis)
    n, ld = 131_100, 131_207
    lors = torch.zeros(10, ld, device=DEV)
    lors[:, :n] = _events(n, sz, 5)
    cg, m = _lib.make_grid(g, c, sz, st), _lib.make_tor_model(4.0, False, *TOF)
    outs = []
    for flags in (0, 1 << 4):  # default, one lane per event
        o = torch.full((n + 1,), -1.0, device=DEV)
        _lib.call("srfx_tor_project", lors.data_ptr(), n, ld, image.data_ptr(), cg, m,
                  o.data_ptr(), flags, torch.cuda.current_stream().cuda_stream)
        assert float(o[n]) == -1.0
        outs.append(o[:n])
    _check(*outs)


def test_sorted_projection_captured():
    """A captured call keeps the kernels without workspace."""
    grid, size = (190, 120, 112), (380.0, 240.0, 224.0)
    lors = _events(131_073, size, 9)
    image = torch.rand(grid[::-1], device=DEV)
    args = (grid, (0.0, 0.0, 0.0), size, 4.0, False, *TOF)
    ref = ops.projection(lors, image, *args)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        c = ops.projection(lors, image, *args)
    for _ in range(3):
        c.fill_(-1.0)
        graph.replay()
        torch.cuda.synchronize()
        _check(c, ref)
