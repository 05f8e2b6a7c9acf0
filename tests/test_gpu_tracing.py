"""Preprocessing under tracers: the traced program computes its own rows' groups, as
the tensor operations it is made of do, not those of the rows it was traced with."""
import numpy as np
import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx

from srf_amd import preprocess as P
from tests.test_preprocess import _events

pytestmark = pytest.mark.gpu


def _rows(n, seed, cols=7):
    return torch.from_numpy(np.ascontiguousarray(_events(n, seed)[:, :cols])).to("cuda")


CASES = {
    "recon": (lambda r: P.recon_process(r, 530.0)["x"], 7),
    "map": (lambda r: P.map_process(r)["y"], 6),
}


@pytest.mark.parametrize("name", CASES)
def test_jit_trace(name):
    f, cols = CASES[name]
    traced = torch.jit.trace(f, (_rows(400, 1, cols),), check_trace=False)
    other = _rows(300, 2, cols)
    assert torch.equal(traced(other), f(other))


@pytest.mark.parametrize("name", CASES)
def test_make_fx(name):
    """The program records the row's operations (its sizes are those it was traced
    with, as of any data-dependent shape)."""
    f, cols = CASES[name]
    rows = _rows(400, 1, cols)
    program = make_fx(f)(rows)
    calls = [n for n in program.graph.nodes if n.op == "call_function"]
    assert len(calls) > 20
    assert torch.equal(program(rows), f(rows))


def test_order_under_a_tracer():
    soa = P.recon_process(_rows(600, 3), 530.0)["x"]
    other = soa.flip(1).contiguous()
    traced = torch.jit.trace(lambda s: P.locality_order(s, 1), (soa,), check_trace=False)
    assert torch.equal(traced(other), P.locality_order(other, 1))
