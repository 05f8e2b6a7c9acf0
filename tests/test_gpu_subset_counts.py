"""Subset counts that are no whole numbers are refused on the device as on the host."""
import numpy as np
import pytest
import torch

from srf_amd import preprocess as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 500])
@pytest.mark.parametrize("device", ["cpu", "cuda"])
@pytest.mark.parametrize("bad", [2.0, 2.5, np.float64(3.0), "2"])
def test_refused(n, device, bad):
    soa = torch.rand(10, n, device=device)
    with pytest.raises(TypeError):
        P.locality_order(soa, bad)
    with pytest.raises(TypeError):
        P.reorder_groups({"x": soa}, bad)


@pytest.mark.parametrize("K", [3, np.int64(3), torch.tensor(3), True])
def test_accepted(K):
    soa = torch.rand(10, 500, device="cuda")
    assert torch.equal(P.locality_order(soa, K), P.locality_order(soa, int(K)))
    assert torch.equal(P.reorder_groups({"x": soa}, K)[1]["x"], P.locality_order(soa, int(K)))
