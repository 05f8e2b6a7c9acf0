"""The memory pool of the calls' workspaces: bounded after a synchronisation, given
back on request, and with several streams and threads on it."""
import threading

import numpy as np
import pytest
import torch

from srf_amd import _lib, ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
GRID, SIZE, MODEL = (128, 128, 96), (256.0, 256.0, 192.0), (6.0, 1.0e6)
N = 500_000


def _events(n, seed):
    r = np.random.default_rng(seed)
    mid = r.uniform(-0.8, 0.8, (n, 3)) * np.asarray(SIZE) / 2
    d = np.column_stack([r.uniform(-1, 1, n), r.uniform(-1, 1, n), np.ones(n)])
    p1, p2 = mid - 150.0 * d, mid + 150.0 * d
    return torch.from_numpy(np.ascontiguousarray(
        np.vstack([p1.T, p2.T, mid.T, np.ones((1, n))]), np.float32)).to(DEV)


def _held():
    """Device memory in use outside torch's allocator."""
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free - torch.cuda.memory_reserved()


def test_pool_is_bounded_and_given_back():
    assert _lib.tor_scatter_binned(N, GRID, SIZE, _lib.make_tor_model(4.0, False, *MODEL))
    lors, v = _events(N, 1), torch.ones(N, device=DEV)
    like = torch.empty(GRID[::-1], device=DEV)
    args = (GRID, (0.0, 0.0, 0.0), SIZE, *MODEL, 4.0, False)
    streams = [torch.cuda.Stream() for _ in range(8)]

    def run():  # eight workspaces of a quarter GiB at once
        outs = []
        torch.cuda.synchronize()
        for s in streams:
            with torch.cuda.stream(s):
                outs.append(ops.backprojection(like, lors, v, *args))
        for s in streams:
            s.synchronize()
        torch.cuda.synchronize()
        return outs

    run()  # the streams' queues and the kernels' own memory
    ops.release_workspace()
    base = _held()
    outs = run()
    kept = _held() - base
    assert 100 << 20 < kept <= (1 << 30) + (256 << 20)
    ops.release_workspace()
    assert _held() - base < 64 << 20
    ref = ops.backprojection(like, lors, v, *args, schedule=(1, 256))
    for o in outs:
        assert float((o - ref).norm() / ref.norm()) <= 1e-5


def test_threads():
    """Four threads, each on a stream of its own, allocate, free and trim."""
    lors, v = _events(60_000, 2), torch.ones(60_000, device=DEV)
    like = torch.empty(GRID[::-1], device=DEV)
    args = (GRID, (0.0, 0.0, 0.0), SIZE, *MODEL, 4.0, False)
    ref = ops.backprojection(like, lors, v, *args, schedule=(1, 256))
    torch.cuda.synchronize()
    outs, errors = [None] * 4, []

    def work(k):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(6):
                    outs[k] = ops.backprojection(like, lors, v, *args)
                    if k == 0:
                        ops.release_workspace()
                torch.cuda.current_stream().synchronize()
        except Exception as e:  # noqa: BLE001 - reported below
            errors.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    for o in outs:
        assert float((o - ref).norm() / ref.norm()) <= 1e-5
