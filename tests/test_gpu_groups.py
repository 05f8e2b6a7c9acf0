"""A subset's groups in shared launches against the same plans one by one: one
to three groups, event counts around the lane rule, every box class, groups of
different walks (refused), a captured call."""
import numpy as np
import pytest
import torch

from srf_amd import physics, preprocess
from srf_amd.data import Image, split_from_groups
from srf_amd.plan import TorPlan

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _data(n, axes, size, seed):
    """n events of every axis in axes: lines through the image, mostly along
    the axis."""
    r = np.random.default_rng(seed)
    rows = []
    for a in axes:
        k = "xyz".index(a)
        d = r.uniform(-0.5, 0.5, (n, 3))
        d[:, k] = 1.0
        mid = r.uniform(-0.35, 0.35, (n, 3)) * np.asarray(size)
        rows.append(np.column_stack([mid - 150 * d, mid + 150 * d, r.normal(0, 20, n)]))
    rows = torch.from_numpy(np.concatenate(rows).astype(np.float32)).to(DEV)
    return split_from_groups(preprocess.recon_process(rows, 530.0))


@pytest.mark.parametrize("n,axes,pitch,kw", [
    (1, "xy", 2.0, 4.0), (700, "xyz", 2.0, 4.0), (24576, "xy", 2.0, 4.0),
    (24577, "xy", 2.0, 4.0), (3000, "z", 2.0, 4.0), (3000, "xy", 1.6, 4.0),
    (3000, "xyz", 2.0, 8.0),
])
def test_groups_together(n, axes, pitch, kw):
    """The same walks; the tile flushes meet in another order: 1e-6."""
    shape = (45, 37, 33)
    size = [s * pitch for s in shape]
    image = Image(torch.rand(shape, device=DEV) + 0.5, [0.0, 0.0, 0.0], size)
    data = _data(n, axes, size, n)
    model = physics.SplitLoRsModel(kw, tof_sigma2=1139.77, tof_bin=6.0)
    plans = model.make_plans(image, data)
    groups = [p for p in plans.values() if p is not None]
    x = image.data
    out, ref = torch.rand(shape, device=DEV), None
    ref = out.clone()
    assert TorPlan.osem_groups(groups, x, out)
    scales = [p.scales() for p in groups]
    for a, p in plans.items():
        if p is not None:
            model.plan_osem_group(p, x, ref, a)
    for p, s in zip(groups, scales):
        t = p.scales()
        assert float((s - t).norm()) <= 1e-6 * float(t.norm())
    assert float((out - ref).norm()) <= 1e-6 * float(ref.norm())
    full = model.osem_subset(image, data, out=torch.zeros_like(x), plans=plans).data
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    bp = torch.zeros_like(x)
    with torch.cuda.graph(graph):
        model.osem_subset(image, data, out=bp, plans=plans)
    for _ in range(3):
        bp.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert float((bp - full).norm()) <= 1e-6 * float(full.norm())


def test_groups_of_different_walks():
    """A 4 mm tube on voxels that are 2 mm along x and y, 1 mm along z: the
    groups need different boxes and run one by one."""
    shape = (40, 40, 60)
    size = [80.0, 80.0, 60.0]
    image = Image(torch.rand(shape, device=DEV) + 0.5, [0.0, 0.0, 0.0], size)
    data = _data(2000, "xz", size, 5)
    model = physics.SplitLoRsModel(4.0, tof_sigma2=1139.77, tof_bin=6.0)
    plans = model.make_plans(image, data)
    groups = [p for p in plans.values() if p is not None]
    assert len({p.walks()[0] for p in groups}) == 2
    out = torch.zeros_like(image.data)
    assert not TorPlan.osem_groups(groups, image.data, out) and not bool(out.any())
    got = model.osem_subset(image, data, plans=plans).data
    for a in "xz":
        model.plan_osem_group(plans[a], image.data, out, a)
    assert float((got - out).norm()) <= 1e-6 * float(out.norm())
    with pytest.raises(ValueError):
        TorPlan.osem_groups(groups, image.data[:, :, :30], out)
