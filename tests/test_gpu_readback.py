"""Fields read back through the packed, piecewise copy equal the oracle's,
cell by cell: rows with and without padding, one piece and several, the last
one partial."""
import numpy as np
import pytest

from oidt_amd import configs, materials
from oidt_amd.solver import COMP_KEYS, Solver

from helpers import device_inputs, oracle_run, rel_l2


@pytest.mark.gpu
@pytest.mark.parametrize('p', [
    configs.slab2d(140, ny=64, nt=40, nf=2, core=12, port_len=25, source_type=1, gauss_pulse_deg=-1.0),
    configs.slab2d(141, ny=67, nt=40, nf=2, core=12, port_len=25, scheme='te', source_type=1, gauss_pulse_deg=-1.0),
    # 34 x 33 rows of 469 values: pieces of 1117 rows and 5 rows
    configs.strip3d(469, nx=34, ny=33, nt=33, nf=2, precision='float64', width=12, height=8, port_len=10, buffer_z=6,
                    source_type=1, gauss_pulse_deg=-1.0),
    configs.strip3d(64, nx=34, ny=36, nt=33, nf=2, precision='float64', width=12, height=8, port_len=10, buffer_z=6,
                    source_type=1, gauss_pulse_deg=-1.0),
], ids=['2d_padless', '2d_padded', '3d_two_pieces', '3d_padless'])
def test_fields_read_whole(p):
    s, up, lo, fg = device_inputs(p)
    o, _ = oracle_run(p, up, lo)
    print('case', s.shape, flush=True)
    dev = Solver(s, fg).run()
    for k, ref in o.fields().items():
        got = dev.field(k)
        assert got.shape == ref.shape
        assert rel_l2(got, ref) < 1e-10, k
    dev.close()


@pytest.mark.gpu
@pytest.mark.parametrize('scheme,nf', [('tm', 3), ('te', 700), ('3d', 40)])
def test_dft_planes_equal_compact_read(scheme, nf):
    """The full-plane phasors (3 x 52 and 40 x 16 x 14 cells fit one read-back
    piece, 700 x 412 take two) hold the compact ones in the window and zeros
    elsewhere, and a run given by CB maps equals the one given by material
    indexes."""
    if scheme == '3d':
        p = configs.strip3d(56, nx=36, ny=34, nt=70, nf=nf, width=12, height=8, port_len=10, buffer_z=6,
                            source_type=1, gauss_pulse_deg=-1.0)
    else:
        p = configs.slab2d(140, ny=72 if scheme == 'tm' else 432, nt=70, nf=nf, scheme=scheme, core=12, port_len=25,
                           source_type=1, gauss_pulse_deg=-1.0)
    p.update(rough_std=15e-9, rough_acl=40e-9, seed=4)
    s, up, lo, fg = device_inputs(p)
    dev, maps = Solver(s, fg).run(), Solver(s, fg, cb=materials.cb_maps(s, fg)).run()
    N = s.num_cpml
    compact = {k: dev.read_dft(port, comp) for port in (0, 1) for comp, k in
               enumerate([(c, port + 1) for c in COMP_KEYS[scheme]])}
    full, other = dev.dft(), maps.dft()
    assert set(full) == set(compact)
    for k, z in full.items():
        ref = np.zeros_like(z)
        w = (slice(None), slice(N, s.ny - N)) if scheme != '3d' else (slice(None), slice(N, s.nx - N), slice(N, s.ny - N))
        ref[w] = compact[k].reshape(ref[w].shape)
        assert k[1] == 2 or np.abs(ref).max() > 0   # the pulse has passed port 1 only
        assert np.array_equal(z, ref) and np.array_equal(z, other[k]), k
    dev.close()
    maps.close()
