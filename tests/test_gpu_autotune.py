"""The autotuner measures the library's own rules beside the named schedules, which
switch off the binned scatters and the ordered projection of large sets."""
import json

import numpy as np
import pytest
import torch

from srf_amd import autotune, physics
from srf_amd.data import Image, split_from_groups

pytestmark = pytest.mark.gpu
GRID, PITCH, MODEL = (200, 200, 100), 2.0, (6.0, 1139.77)


def _rows(n, seed):
    r = np.random.default_rng(seed)
    size = np.array([g * PITCH for g in GRID])
    mid = r.uniform(-0.4, 0.4, (n, 3)) * size
    d = np.column_stack([r.uniform(-1, 1, n), r.uniform(-1, 1, n), np.ones(n)])
    p1, p2 = mid - 100.0 * d, mid + 100.0 * d
    return torch.from_numpy(np.ascontiguousarray(
        np.vstack([p1.T, p2.T, mid.T, np.ones((1, n))]), np.float32)).to("cuda")


def test_large_scatters_keep_the_default(tmp_path):
    """200k events of one group: the binned scatter takes 0.4 ms, the direct ones 3 and
    more, so any timing keeps the default."""
    rows = _rows(200_000, 1)
    data = split_from_groups({"x": rows[:, :0], "y": rows[:, :0], "z": rows})
    size = [g * PITCH for g in GRID]
    image = Image(torch.rand(GRID, device="cuda") + 0.5, (0.0, 0.0, 0.0), size)
    model = physics.SplitLoRsModel(4.0, tof_sigma2=MODEL[1], tof_bin=MODEL[0])
    report = model.autotune(image, data, reps=1, ops_=("backprojection", "osem_subset"))
    for op in ("backprojection", "osem_subset"):
        assert set(report[op]) == {None, *autotune.SCHEDULES}
        assert model.schedule[op] is None
    frame = torch.rand(GRID[::-1], device="cuda") + 0.5
    args = (GRID, (0.0, 0.0, 0.0), size, 4.0, False, *MODEL)
    best, times = autotune.tune("backprojection", rows, frame, *args, reps=1)
    assert best is None and None in times
    assert autotune.lookup("backprojection", GRID, size, 4.0, True) is None
    assert autotune.tune("backprojection", rows, frame, *args) == (None, None)
    autotune.save(tmp_path / "tuned.json")
    autotune.load(tmp_path / "tuned.json")
    assert [v for k, v in json.load(open(tmp_path / "tuned.json"))
            if k[0] == "backprojection"] == [None]


def test_fastest():
    assert autotune.fastest({None: 1.0, (4, 256): 0.99}) is None
    assert autotune.fastest({None: 1.0, (4, 256): 0.9}) == (4, 256)
    assert autotune.fastest({(1, 64): 2.0, (4, 256): 1.0}) == (4, 256)
