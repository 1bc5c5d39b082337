"""Sources and captures outside the update ranges: the blocked 2D step drives
and captures the cells that the two-kernel form does, finite and infinite
fields alike (FP32: the same bits, FP64: to 1e-12)."""
import dataclasses

import numpy as np
import pytest

from oidt_amd.solver import Batch, RunArrays

from test_gpu_blocked2d import FIELDS, same, small


class Border(RunArrays):
    """A source over rows and planes of a corner and the ports on the first
    and the last planes a capture may take."""

    def __init__(self, s, fg, box, ports):
        super().__init__(s, fg)
        self.src_box = box
        self.ports = ports

    def desc(self):
        d = super().desc()
        d.port[0], d.port[1] = self.ports
        return d


def outcome(arrays, s, scheme, launch):
    b = Batch(scheme, s.precision, max_slots=len(arrays))
    if launch:
        b.set_launch(*launch)
    slots = [b.add_arrays(a, s) for a in arrays]
    b.advance(-(-s.nt // 32))
    b.sync()
    out = [({n: b.field(k, n) for n in FIELDS[scheme]}, b.dft(k)) for k in slots]
    b.close()
    return out


@pytest.mark.gpu
@pytest.mark.parametrize('scheme', ['tm', 'te'])
@pytest.mark.parametrize('precision', ['float32', 'float64'])
@pytest.mark.parametrize('copies', [1, 7])     # narrow and wide tiles
@pytest.mark.parametrize('high', [False, True])
def test_source_and_captures_outside_the_update_ranges(scheme, precision, copies, high):
    nx, ny = 97, 98
    s, fg = small(scheme, precision, nx, ny, 45)
    boxes = [[nx - 4, nx, ny - 30, ny, 0, 1], [nx - 1, nx, 0, ny, 0, 1]] if high else \
            [[0, 4, 0, 30, 0, 1], [1, 2, 0, ny, 0, 1]]
    ports = (nx - 2, nx - 3) if high else (0, 1)
    print('case', scheme, precision, copies, high, flush=True)
    arrays = [Border(s, fg, box, ports) for box in boxes] * copies
    same(outcome(arrays, s, scheme, None), outcome(arrays, s, scheme, (4, 0, 2)), precision == 'float32')
    J = np.array(s.J_SRC)
    J[2] = np.inf
    s = dataclasses.replace(s, J_SRC=J)
    arrays = [Border(s, fg, box, ports) for box in boxes] * copies
    for (f, d), (g, e) in zip(outcome(arrays, s, scheme, None), outcome(arrays, s, scheme, (4, 0, 2))):
        for k in f:
            assert np.array_equal(np.isnan(f[k]), np.isnan(g[k])) and np.array_equal(np.isinf(f[k]), np.isinf(g[k])), k
        if precision == 'float32':
            for got, ref in ((f, g), (d, e)):
                for k in got:
                    assert np.array_equal(got[k], ref[k], equal_nan=True), k
