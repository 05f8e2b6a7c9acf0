"""The size rules by which untiled scatters run binned (host only)."""
import pytest

from srf_amd import _lib

TOF, NO_TOF = (6.0, 1139.77), (6.0, 1.0e6)


def _tor(n, grid, pitch, kw, model=TOF, schedule=None):
    m = _lib.make_tor_model(kw, False, *model)
    return _lib.tor_scatter_binned(n, grid, [g * pitch for g in grid], m, schedule)


def test_weights_of_the_set():
    """200 x 200 x 100, 2 mm, 4 mm tube: 3.14 voxels by 100 slices an event."""
    assert _tor(8000, (200, 200, 100), 2.0, 4.0)
    assert not _tor(7000, (200, 200, 100), 2.0, 4.0)
    assert not _tor(0, (200, 200, 100), 2.0, 4.0)
    assert _tor(100_000_000, (200, 200, 100), 2.0, 4.0)
    assert not _tor(1_000_000, (200, 200, 100), 2.0, 4.0, schedule=(1, 256))


@pytest.mark.parametrize("grid,pitch,kw,model,binned", [
    # tubes thinner than the voxels: few weights an event, however many events
    ((40, 40, 20), 10.0, 4.0, TOF, False), ((40, 40, 40), 10.0, 4.0, NO_TOF, False),
    ((40, 40, 20), 10.0, 3.0, TOF, False), ((64, 64, 32), 6.3, 3.0, TOF, False),
    ((64, 64, 64), 6.3, 3.0, NO_TOF, True), ((64, 64, 32), 6.3, 4.0, TOF, True),
    ((80, 80, 40), 5.0, 3.0, TOF, True),
])
def test_weights_of_an_event(grid, pitch, kw, model, binned):
    assert _tor(1_600_000, grid, pitch, kw, model) is binned


def test_siddon():
    """128 x 128 x 64, 3 mm: 160 planes a ray, with TOF 91 of them."""
    args = ((128, 128, 64), (384.0, 384.0, 192.0), 6.0)
    assert _lib.siddon_scatter_binned(12_600, *args, 1.0e6)
    assert not _lib.siddon_scatter_binned(12_400, *args, 1.0e6)
    assert not _lib.siddon_scatter_binned(12_600, *args, 1139.77)
    assert _lib.siddon_scatter_binned(23_000, *args, 1139.77)


def test_bad_arguments():
    with pytest.raises(_lib.SrfxError):
        _tor(-1, (40, 40, 20), 2.0, 4.0)
    with pytest.raises(_lib.SrfxError):
        _lib.siddon_scatter_binned(-1, (4, 4, 4), (8.0, 8.0, 8.0), 6.0, 1e6)
