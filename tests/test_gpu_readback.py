"""Fields read back through the packed, piecewise copy equal the oracle's,
cell by cell: rows with and without padding, one piece and several, the last
one partial."""
import pytest

from oidt_amd import configs
from oidt_amd.solver import Solver

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
