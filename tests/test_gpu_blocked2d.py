"""The blocked 2D step at the sizes where its tiles can go wrong: it gives the
two-kernel form's fields and port DFT (FP32: the same bits, FP64: to 1e-12),
and the library's own choice of form gives the same results under monitors
that come and go."""
import numpy as np
import pytest

from oidt_amd import configs, variants
from oidt_amd.solver import Batch, Monitor, Solver

from helpers import device_inputs, rel_l2

FIELDS = {'tm': ('ez', 'hx', 'hy'), 'te': ('ex', 'ey', 'hz')}


def small(scheme, precision, nx, ny, nt, seed=5, **over):
    p = configs.slab2d(nx, ny=ny, nt=nt, nf=4, precision=precision, scheme=scheme, core=12, port_len=8, buffer_x=4,
                       source_type=1, gauss_pulse_deg=-1.0)
    p.update(over)
    p.update(rough_std=15e-9, rough_acl=40e-9, seed=seed)
    s, up, lo, fg = device_inputs(p)
    return s, fg


def outcome(b, slots, scheme):
    return [({n: b.field(k, n) for n in FIELDS[scheme]}, b.dft(k)) for k in slots]


def same(got, ref, exact):
    for (f, d), (g, e) in zip(got, ref):
        for k, v in list(f.items()) + list(d.items()):
            w = g[k] if k in g else e[k]
            if exact:
                assert np.array_equal(v, w), k
            else:
                assert rel_l2(v, w) < 1e-12, k


def run(scheme, precision, runs, direction, launch):
    b = Batch(scheme, np.dtype(precision).type, max_slots=len(runs))
    if launch:
        b.set_launch(*launch)
    slots = [b.add(s, fg, direction) for s, fg in runs]
    b.advance(-(-max(s.nt for s, _ in runs) // 32))
    b.sync()
    out = outcome(b, slots, scheme)
    b.close()
    return out


# x extents around the narrow (16 own planes) and wide (32) tiles, y extents
# around the 48 own rows; enough runs in one batch for the wide tile.
@pytest.mark.gpu
@pytest.mark.parametrize('scheme', ['tm', 'te'])
@pytest.mark.parametrize('precision', ['float32', 'float64'])
@pytest.mark.parametrize('sizes,copies,direction', [
    (((48, 44, 40), (49, 48, 33), (63, 49, 70)), 1, 'f'),
    (((64, 96, 41), (65, 97, 64), (95, 53, 7)), 1, 'b'),
    (((96, 98, 45), (97, 143, 39), (129, 145, 32)), 12, 'f'),
])
def test_default_2d_form_matches_two_kernel(scheme, precision, sizes, copies, direction):
    runs = [small(scheme, precision, nx, ny, nt, seed=5 + k) for k, (nx, ny, nt) in enumerate(sizes * copies)]
    print('case', scheme, precision, sizes, copies, direction, flush=True)
    same(run(scheme, precision, runs, direction, None), run(scheme, precision, runs, direction, (4, 0, 2)),
         precision == 'float32')


@pytest.mark.gpu
@pytest.mark.parametrize('scheme', ['tm', 'te'])
def test_form_changes_between_chunks(scheme):
    """A monitored run joins a batch in progress and leaves again: the library
    changes between the blocked and the two-kernel form at chunk boundaries,
    and every run ends as it does alone."""
    a, c = small(scheme, 'float32', 97, 70, 150), small(scheme, 'float32', 70, 98, 70, seed=9)
    name = FIELDS[scheme][0]
    mon = Monitor(name, [(0, 0)], 1.0, [(0, 70), (0, 98)], 70, after_h=True, cs=np.ones((70, 2)))
    b = Batch(scheme, np.float32, max_slots=2)
    ka = b.add(*a)
    b.advance(1)
    kc = b.add(*c)
    idx = b.add_monitor(kc, mon)
    b.advance(2)
    b.sync()
    mid = b.field(ka, name)
    b.advance(1)
    b.sync()
    got_c, got_mon = outcome(b, [kc], scheme), b.read_monitor(kc, idx)
    b.remove(kc)
    b.advance(1)
    b.sync()
    got_a = outcome(b, [ka], scheme)
    b.close()
    same(got_a, run(scheme, 'float32', [a], 'f', (4, 0, 2)), True)
    same(got_c, run(scheme, 'float32', [c], 'f', (4, 0, 2)), True)
    b = Batch(scheme, np.float32, max_slots=1)
    k = b.add(*a)
    b.advance(3)
    assert np.array_equal(mid, b.field(k, name))
    b.close()
    b = Batch(scheme, np.float32, max_slots=1)
    k = b.add(*c)
    i = b.add_monitor(k, mon)
    b.advance(3)
    for x, y in zip(got_mon, b.read_monitor(k, i)):
        assert np.array_equal(x, y)
    b.close()


# whole-plane and partial boxes, before and after the H half-step, records that
# start late and end early, a batch small enough for the narrow tile and one
# that is not
@pytest.mark.gpu
@pytest.mark.parametrize('scheme', ['te', 'tm'])
@pytest.mark.parametrize('copies', [1, 9])
def test_folded_monitors_match_monitor_kernel(scheme, copies):
    names = ('ey', 'hz') if scheme == 'te' else ('hy', 'ez', 'hx')
    over = dict(port1_length=1e-6) if scheme == 'te' else dict(port_length=1e-6)
    cs = [variants.truncate(variants.config(scheme, 'scattering_loss', sgl_wg_length=6e-6, points_per_wl=20,
                                            gauss_pulse_deg=-1, profile_number=k, **over), 75 + k) for k in range(copies)]
    print('case', scheme, copies, cs[0].nx, cs[0].ny, flush=True)
    out = []
    for launch in ((2, 4, 0), (0, 0, 0)):
        out.append(variants.run_batch(cs, launch))
        c = cs[0]
        rng = np.random.default_rng(3)
        boxes = [[(0, c.nx), (0, c.ny)], [(17, 60), (40, 97)], [(c.nx - 33, c.nx), (c.ny - 1, c.ny)]]
        s, fg, cb = variants.build(c)
        sol = Solver.from_arrays(variants.LossyTmArrays(c, fg), c.nt) if scheme == 'tm' else Solver(s, fg, cb=cb)
        if launch[0]:
            sol.set_launch(launch[1], launch[2], launch[0])
        ids = [sol.add_monitor(Monitor(n, [(0, 0)], 0.7, boxes[(k + 1) % 3], 50, after_h=bool(k & 1), shift=-11 + 6 * k,
                                       cs=rng.standard_normal((50, 2)))) for k, n in enumerate(names)]
        sol.run()
        out[-1].append({(n, part): a for n, i in zip(names, ids) for part, a in enumerate(sol.read_monitor(i))})
        sol.close()
    for ref, got in zip(*out):
        for k in ref:
            assert np.array_equal(got[k], ref[k]), k
