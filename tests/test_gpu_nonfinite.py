"""Infinite and NaN fields: the blocked steps hold them in the cells in which
the two-kernel forms hold them.  The source turns infinite, its front spreads
one cell per step into the slabs and to the cells outside the update ranges."""
import dataclasses

import numpy as np
import pytest

from oidt_amd import variants
from oidt_amd.solver import COMP_KEYS, Batch, Monitor, Solver

from test_gpu_blocked2d import FIELDS, run, small
from test_gpu_blocked3d import alone, strip


def infinite(s, step=2):
    J = np.array(s.J_SRC)
    J[step] = np.inf
    return dataclasses.replace(s, J_SRC=J)


def same_cells(x, y, exact=True):
    assert np.array_equal(np.isnan(x), np.isnan(y))
    if exact:
        assert np.array_equal(x, y, equal_nan=True)
    else:
        assert np.array_equal(np.isposinf(x), np.isposinf(y)) and np.array_equal(np.isneginf(x), np.isneginf(y))
        ok = np.isfinite(y)
        assert np.array_equal(ok, np.isfinite(x)) and np.allclose(x[ok], y[ok], rtol=0, atol=1e-12 * np.abs(y[ok]).max())


@pytest.mark.gpu
@pytest.mark.parametrize('scheme', ['tm', 'te'])
@pytest.mark.parametrize('precision', ['float32', 'float64'])
@pytest.mark.parametrize('direction', ['f', 'b'])
@pytest.mark.parametrize('nx,copies', [(97, 1), (129, 20)])   # narrow and wide tiles
def test_blocked_2d_keeps_border_cells(scheme, precision, direction, nx, copies):
    s, fg = small(scheme, precision, nx, 98, 70)
    print('case', scheme, precision, direction, nx, copies, flush=True)
    runs = [(infinite(s), fg)] * copies
    (got, dft), (ref, dft2) = (run(scheme, precision, runs, direction, launch)[-1] for launch in (None, (4, 0, 2)))
    for k in FIELDS[scheme]:
        assert not np.isfinite(ref[k][:, 3]).all()      # the front has reached the border
        same_cells(got[k], ref[k], precision == 'float32')
    if precision == 'float32':
        for k in dft:
            assert np.array_equal(dft[k], dft2[k], equal_nan=True)


@pytest.mark.gpu
@pytest.mark.parametrize('scheme', ['te', 'tm'])
@pytest.mark.parametrize('monitored', [True, False])
def test_blocked_studies_keep_border_cells(scheme, monitored):
    over = dict(port1_length=0.3e-6) if scheme == 'te' else dict(port_length=0.3e-6)
    c = variants.truncate(variants.config(scheme, 'scattering_loss', sgl_wg_length=1.5e-6, points_per_wl=16, ny_clad_wl=0.4,
                                          **over), 90)
    c.J_SRC = np.array(c.J_SRC)
    c.J_SRC[2] = np.inf
    print('case', scheme, monitored, c.nx, c.ny, flush=True)
    out = []
    for launch in ((2, 4, 0), (0, 0, 0)):
        if monitored:
            out.append(variants.run(c, launch))
            continue
        s, fg, cb = variants.build(c)
        sol = Solver.from_arrays(variants.LossyTmArrays(c, fg), c.nt) if scheme == 'tm' else Solver(s, fg, cb=cb)
        if launch[0]:
            sol.set_launch(launch[1], launch[2], launch[0])
        sol.run()
        out.append({k: sol.field(k) for k in FIELDS[scheme]})
        sol.close()
    assert any(not np.isfinite(v).all() for v in out[0].values())
    for k, ref in out[0].items():
        assert np.array_equal(np.asarray(out[1][k]), np.asarray(ref), equal_nan=True), k


@pytest.mark.gpu
def test_infinite_weights_take_the_monitor_kernel():
    """Zero fields fold to NaN under an infinite weight, at the border too."""
    s, fg = small('te', 'float32', 97, 70, 40)
    cs = np.ones((40, 2))
    cs[20] = np.inf
    mon = Monitor('hz', [(0, 0)], 1.0, [(0, 97), (0, 70)], 40, after_h=True, cs=cs)
    out = []
    for launch in (False, True):
        b = Batch('te', np.float32, max_slots=1)
        slot = b.add(s, fg)
        idx = b.add_monitor(slot, mon)
        if launch:
            b.set_launch(4, 0, 2)
        assert b.launch() == (2, 4, 0)
        b.advance(2)
        out.append(b.read_monitor(slot, idx))
        b.close()
    assert np.isnan(out[0][0][:, 0]).all()      # the first row stays zero
    for x, y in zip(*out):
        assert np.array_equal(x, y, equal_nan=True)


@pytest.mark.gpu
@pytest.mark.parametrize('nx,ny,nz,direction', [(33, 37, 61, 'f'), (64, 48, 120, 'b'), (65, 49, 121, 'f')])
def test_blocked_3d_keeps_the_marchs_cells(nx, ny, nz, direction):
    s, fg = strip(nx, ny, nz, 45)
    print('case', nx, ny, nz, direction, flush=True)
    got, ref = (alone((infinite(s), fg), launch, direction) for launch in ((2, 0, 4), (4, 0, 1)))
    assert any(not np.isfinite(x).all() for x in ref)
    for x, y in zip(got, ref):
        assert np.array_equal(x, y, equal_nan=True)


@pytest.mark.gpu
@pytest.mark.parametrize('scheme', ['tm', '3d'])
def test_dft_planes_hold_the_compact_phasors(scheme):
    """dft() and read_dft() form the same complex values (a zero frequency has
    a NaN imaginary part beside an infinite real one)."""
    s, fg = small('tm', 'float32', 97, 98, 70) if scheme == 'tm' else strip(64, 48, 120, 60)
    freqs = np.array(s.sparam_freqs, float)
    freqs[0] = 0.0
    s = dataclasses.replace(infinite(s), sparam_freqs=freqs)
    print('case', scheme, s.shape, flush=True)
    dev = Solver(s, fg).run()
    N, planes = s.num_cpml, dev.dft()
    w = (slice(None), slice(N, s.ny - N)) if scheme == 'tm' else (slice(None), slice(N, s.nx - N), slice(N, s.ny - N))
    assert any(not np.isfinite(z[w]).all() for z in planes.values())
    for (k, port), z in planes.items():
        ref = dev.read_dft(port - 1, COMP_KEYS[scheme].index(k)).reshape(z[w].shape)
        for x, y in ((z[w].real, ref.real), (z[w].imag, ref.imag)):
            assert np.array_equal(x, y, equal_nan=True)
            assert np.array_equal(np.signbit(x)[~np.isnan(x)], np.signbit(y)[~np.isnan(y)])
    dev.close()
