"""The library's own choice of launch form: what the batch reports, and the
calls that keep it."""
import numpy as np
import pytest

from oidt_amd import variants
from oidt_amd.solver import Batch, Monitor

from test_gpu_blocked2d import outcome, run, same, small
from test_gpu_blocked3d import strip

LOSSY = dict(sgl_wg_length=1.5e-6, port_length=0.3e-6, points_per_wl=16, ny_clad_wl=0.4, buffer_xhat=5, num_cpml=6)


def write_back(b):
    variant, xchunk, grid = b.launch()
    b.set_launch(xchunk, grid, variant)


@pytest.mark.gpu
@pytest.mark.parametrize('scheme', ['tm', 'te'])
def test_reported_form_is_the_running_one(scheme):
    """Before and between the chunks of a run, with the reported knobs written
    back each time."""
    a = small(scheme, 'float32', 97, 70, 90)
    print('case', scheme, flush=True)
    b = Batch(scheme, np.float32, max_slots=2)
    slot = b.add(*a)
    assert b.launch() == (4, 8, 0)
    for _ in range(3):
        b.advance(1)
        write_back(b)
        assert b.launch() == (4, 8, 0)
    b.sync()
    same(outcome(b, [slot], scheme), run(scheme, 'float32', [a], 'f', (4, 0, 2)), True)
    b.close()
    b = Batch(scheme, np.float32, max_slots=1)
    b.add(*a)
    b.set_launch(4, 0, 2)
    assert b.launch() == (2, 4, 0)
    b.close()


@pytest.mark.gpu
@pytest.mark.parametrize('npts', [1, 2])
def test_reported_form_with_monitors(npts):
    """A monitor the blocked step folds, and one that it does not."""
    a = small('te', 'float32', 97, 70, 64)
    mon = Monitor('hz', [(0, 0), (1, 0)][:npts], 1.0, [(0, 70), (0, 70)], 64, after_h=True, cs=np.ones((64, 2)))
    print('case', npts, flush=True)
    out = []
    for written in (False, True):
        b = Batch('te', np.float32, max_slots=1)
        slot = b.add(*a)
        idx = b.add_monitor(slot, mon)
        if written:
            write_back(b)
        assert b.launch() == ((4, 8, 0) if npts == 1 else (2, 4, 0))
        b.advance(2)
        out.append(b.read_monitor(slot, idx))
        b.close()
    for x, y in zip(*out):
        assert np.array_equal(x, y)


@pytest.mark.gpu
def test_reported_form_of_lossy_runs():
    c = variants.truncate(variants.config('tm', 'scattering_loss', **LOSSY), 64)
    b, runs = variants.prepare_batch([c])
    print('case', c.nx, c.ny, flush=True)
    assert b.launch() == (4, 8, 0)
    write_back(b)
    b.advance(1)
    write_back(b)
    assert b.launch() == (4, 8, 0)
    b.close()


@pytest.mark.gpu
# fields of 205 and 231 MiB
@pytest.mark.parametrize('copies,nx,ny,nz,form', [(120, 33, 37, 61, (1, 4, 0)), (12, 70, 48, 250, (4, 2, 0))])
def test_large_3d_batches_take_the_blocked_form_where_its_tiles_cover(copies, nx, ny, nz, form):
    """Runs just past the tile edges stay with the march."""
    a = strip(nx, ny, nz, 64)
    print('case', copies, nx, ny, nz, flush=True)
    b = Batch('3d', np.float32, max_slots=copies)
    for _ in range(copies):
        b.add(*a)
    assert b.launch() == form
    b.close()
