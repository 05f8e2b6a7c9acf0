"""LOR preprocessing kernels against the torch operations they stand for: the
same bits (FP64 in the same order, rounded once) and the same row orders, at
row counts around a workgroup's, both row types and several layouts."""
import numpy as np
import pytest
import torch
from torch.autograd import forward_ad

from srf_amd import preprocess as P
from tests.test_preprocess import _events

pytestmark = pytest.mark.gpu


def _rows(n, seed):
    rows = _events(max(n, 8), seed)
    if n >= 1000:
        rows[5::97, 0] = np.nan                 # no dominant axis: dropped
        rows[7::101, 3:6] = rows[7::101, 0:3]   # zero length
        rows[11::103, 5] = 900.0                # axial
        rows[13::89, 3:6] = rows[13::89, 0:3] + np.array([50.0, -50.0, 50.0])  # ties
    return rows[:n]


def _same(a, b):
    return a.shape == b.shape and torch.equal(torch.nan_to_num(a, nan=-7.0),
                                              torch.nan_to_num(b, nan=-7.0))


def _layouts(rows, dtype, dev):
    t = torch.from_numpy(rows).to(dtype)
    wide = torch.zeros(rows.shape[0], rows.shape[1] + 3, dtype=dtype, device=dev)
    wide[:, 2:2 + rows.shape[1]] = t.to(dev)
    return [t.to(dev), wide[:, 2:2 + rows.shape[1]], t.to(dev).t().contiguous().t()]


@pytest.mark.parametrize("n", [1, 255, 1023, 1024, 1025, 9000])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("tof_res", [530.0, 1.0e4, -1.0])
def test_recon_process(cuda, n, dtype, tof_res):
    rows = _rows(n, 3)
    want, wo = P.recon_process(torch.from_numpy(rows).to(dtype), tof_res, return_order=True)
    for x in _layouts(rows, dtype, cuda):
        got, go = P.recon_process(x, tof_res, return_order=True)
        for a in "xyz":
            assert torch.equal(go[a].cpu(), wo[a]), a
            assert _same(got[a].cpu(), want[a]), a
        plain = P.recon_process(x, tof_res)
        assert all(_same(plain[a], got[a]) for a in "xyz")


@pytest.mark.parametrize("n", [1, 1024, 9000])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_map_process(cuda, n, dtype):
    rows = _rows(n, 4)[:, :6].copy()
    want, wo = P.map_process(torch.from_numpy(rows).to(dtype), return_order=True)
    for x in _layouts(rows, dtype, cuda):
        got, go = P.map_process(x, return_order=True)
        for a in "xyz":
            assert torch.equal(go[a].cpu(), wo[a]) and _same(got[a].cpu(), want[a]), a


@pytest.mark.parametrize("n,K", [(1, 1), (1, 3), (700, 1), (5000, 7), (5000, 5000), (40, 100)])
def test_locality_order(cuda, n, K):
    soa = torch.cat(list(P.recon_process(torch.from_numpy(_events(max(2 * n, 8), 6)).to(cuda),
                                         530.0).values()), 1)[:, :n].contiguous()
    n = soa.shape[1]
    key = P.locality_key(soa, 1.5)
    want = torch.cat([(k * n) // K + torch.argsort(key[(k * n) // K:((k + 1) * n) // K],
                                                   stable=True) for k in range(K)])
    assert torch.equal(P.locality_order(soa, K, 1.5), want)
    out, orders = P.reorder_groups({"x": soa}, K, {"x": 1.5})
    assert torch.equal(orders["x"], want) and torch.equal(out["x"], soa[:, want])


def test_rows_with_a_tangent(cuda):
    """Forward-mode rows keep their tangent."""
    rows = torch.from_numpy(_rows(300, 8)).to(cuda)
    with forward_ad.dual_level():
        dual = forward_ad.make_dual(rows, torch.ones_like(rows))
        got = P.recon_process(dual, 530.0)
        want = P.recon_process(rows, 530.0)
        for a in "xyz":
            primal, tangent = forward_ad.unpack_dual(got[a])
            assert torch.equal(primal, want[a])
            assert tangent is not None and bool((tangent[0] == 1).any())
