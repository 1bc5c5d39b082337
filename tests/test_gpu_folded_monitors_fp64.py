"""Monitors folded by the blocked 2D step in FP64 (the studies run in FP32):
the two-kernel form's sums to 1e-12, in a batch whose narrow tiles have a CU
each and in one with more, boxes that take the whole plane, part of it and its
last row, before and after the H half-step, records that start late and end
early."""
from types import SimpleNamespace

import numpy as np
import pytest

from oidt_amd import _lib, variants
from oidt_amd.solver import Batch, Monitor

from helpers import rel_l2
from test_gpu_blocked2d import small


class LossyFp64(variants.LossyTmArrays):
    """The lossy TMz study's run in double precision."""

    def __init__(self, c, fg):
        super().__init__(c, fg)
        self.k = {n: np.ascontiguousarray(a, np.float64) if np.ndim(a) else a for n, a in self.k.items()}
        self.cb = [a.astype(np.float64) for a in self.cb]
        self.jsrc = self.jsrc.astype(np.float64)

    def desc(self):
        d = super().desc()
        d.precision = _lib.F64
        return d


def te_runs(copies):
    runs = [small('te', 'float64', 97, 98, 75 + k, seed=5 + k) for k in range(copies)]
    return Batch('te', np.float64, max_slots=copies), lambda b: [b.add(s, fg) for s, fg in runs], runs[0][0]


def lossy_runs(copies):
    cs = [variants.truncate(variants.config('tm', 'scattering_loss', sgl_wg_length=1.5e-6, port_length=0.3e-6, points_per_wl=16,
                                            ny_clad_wl=0.4, profile_number=k), 75 + k) for k in range(copies)]
    meta = [SimpleNamespace(nt=c.nt, precision=np.float64, shape=(c.nx, c.ny), sparam_freqs=np.zeros(0)) for c in cs]
    arrays = [LossyFp64(c, variants.tm_mask(c, None, None)) for c in cs]
    return (Batch('tm_lossy', np.float64, max_slots=copies),
            lambda b: [b.add_arrays(a, m) for a, m in zip(arrays, meta)], cs[0])


@pytest.mark.gpu
@pytest.mark.parametrize('runs,names', [(te_runs, ('ey', 'hz')), (lossy_runs, ('hy', 'ez', 'hx'))], ids=['te', 'tm_lossy'])
@pytest.mark.parametrize('copies', [1, 13])
def test_fp64_folded_monitors_match_monitor_kernel(runs, names, copies):
    out = []
    for launch in (None, (4, 0, 2)):
        b, add, c = runs(copies)
        print('case', names, copies, c.nx, c.ny, launch, flush=True)
        if launch:
            b.set_launch(*launch)
        boxes = [[(0, c.nx), (0, c.ny)], [(17, 60), (20, 67)], [(c.nx - 33, c.nx), (c.ny - 1, c.ny)]]
        rng = np.random.default_rng(3)
        sums = []
        slots = add(b)
        mons = [(slot, b.add_monitor(slot, Monitor(n, [(0, 0)], 0.7, boxes[(k + r) % 3], 50, after_h=bool(k & 1),
                                                   shift=-11 + 6 * k, cs=rng.standard_normal((50, 2)))))
                for r, slot in enumerate(slots) for k, n in enumerate(names)]
        assert b.launch() == ((2, 4, 0) if launch else (4, 8, 0))
        b.advance(-(-(75 + copies) // 32))
        for slot, idx in mons:
            sums += list(b.read_monitor(slot, idx))
        b.close()
        out.append(sums)
    assert max(np.abs(x).max() for x in out[1]) > 0
    for got, ref in zip(*out):
        assert rel_l2(got, ref) < 1e-12
