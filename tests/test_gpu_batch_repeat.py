"""A batch places its events in buckets in whatever order they arrive: their
projections do not depend on which events share a wave."""
import numpy as np
import pytest
import torch

from srf_amd import physics
from srf_amd.batch import BatchedOSEM
from srf_amd.data import Image, split_from_groups

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("schedule", [(4, 64), (16, 64), (1, 64)])
@pytest.mark.parametrize("kw", [4.0, 5.0, 8.0])
def test_order_of_events_does_not_matter(cuda, kw, schedule):
    """The bits of one iteration, events in two orders.  Its other sums are exact: no
    TOF, so that weights lie within 2^7 of one another and ratios within 2^6, and a
    few hundred events, one chunk a tile: FP64 holds 24 + 13 + 9 bits and more, and
    every voxel is flushed once, onto zero."""
    shape, size, n = (40, 36, 32), (80.0, 72.0, 64.0), 500
    r = np.random.default_rng(7)
    p1 = np.column_stack([r.uniform(-6, 6, (n, 2)), r.uniform(-31, 0, n)])
    d = np.column_stack([r.uniform(-0.1, 0.1, (n, 2)), np.ones(n)])
    p2 = p1 + d * r.uniform(16, 31, n)[:, None]
    rows = np.vstack([p1.T, p2.T, (0.5 * (p1 + p2)).T, np.ones((1, n))]).astype(np.float32)
    x0 = r.uniform(0.5, 1.5, shape).astype(np.float32)
    images = []
    for order in (np.arange(n), r.permutation(n), np.arange(n)[::-1]):
        soa = torch.from_numpy(np.ascontiguousarray(rows[:, order])).to(cuda)
        rec = {"image": Image(torch.from_numpy(x0).to(cuda), (0, 0, 0), size),
               "emap": Image(torch.ones(shape, device=cuda), (0, 0, 0), size),
               "data": split_from_groups({"x": soa[:, :0], "y": soa[:, :0], "z": soa})}
        model = physics.SplitLoRsModel(kw, tof_sigma2=1.0e6, tof_bin=6.0)
        batch = BatchedOSEM([rec], model, 1)
        batch.set_schedule(*schedule)
        batch.iterate(1)
        torch.cuda.synchronize()
        images.append(rec["image"].data.clone())
    assert bool((images[0] > 0).any())
    assert torch.equal(images[0], images[1]) and torch.equal(images[0], images[2])
