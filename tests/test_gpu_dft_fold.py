"""The chunk fold of the port DFT at the edges of its matrix tiles: 1, 7, 8, 9
and 33 frequencies (tiles of 8, items of up to 32), windows of 16, 65 and 129
cells (groups of 16, items of 64 and 128), step counts that leave a partial
chunk.  FP64 against the oracle: relative L2 1e-10, the parity bar."""
import numpy as np
import pytest

from oidt_amd import configs
from oidt_amd.solver import Batch

from helpers import device_inputs, oracle_run, rel_l2, window


@pytest.mark.gpu
@pytest.mark.parametrize('scheme', ['tm', 'te'])
@pytest.mark.parametrize('ny,nf,nt,copies', [(36, 1, 33, 1), (85, 7, 45, 1), (85, 8, 64, 1), (149, 9, 71, 1),
                                             (149, 33, 45, 1), (149, 33, 45, 30)])
def test_fold_edges_fp64(scheme, ny, nf, nt, copies):
    p = configs.slab2d(60, ny=ny, nt=nt, nf=nf, scheme=scheme, core=12, port_len=8, buffer_x=4, source_type=1,
                       gauss_pulse_deg=-1.0)
    s, up, lo, fg = device_inputs(p)
    o, _ = oracle_run(p)
    print('case', scheme, ny, nf, nt, copies, flush=True)
    b = Batch(scheme, np.float64, max_slots=copies)
    slots = [b.add(s, fg) for _ in range(copies)]
    b.advance(-(-s.nt // 32))
    b.sync()
    w, od = window(scheme, o.c), o.dft()
    for slot in (slots[0], slots[-1]):
        for k, z in b.dft(slot).items():
            assert rel_l2(z[w], od[k][w]) < 1e-10, k
    b.close()


@pytest.mark.gpu
def test_fold_edges_3d_fp64():
    """Four-tap samples, windows of 16 x 14 cells, 10 frequencies."""
    p = configs.strip3d(56, nx=36, ny=34, nt=70, nf=10, precision='float64', width=12, height=8, port_len=10,
                        buffer_z=6, source_type=1, gauss_pulse_deg=-1.0)
    s, up, lo, fg = device_inputs(p)
    o, _ = oracle_run(p)
    b = Batch('3d', np.float64, max_slots=1)
    slot = b.add(s, fg)
    b.advance(3)
    b.sync()
    w, od = window('3d', o.c), o.dft()
    for k, z in b.dft(slot).items():
        assert rel_l2(z[w], od[k][w]) < 1e-10, k
    b.close()
