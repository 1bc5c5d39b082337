"""The blocked 3D step gives the march's bits in FP32, at the sizes where its
tiles can go wrong (32 planes x 12 rows x 60 z-cells), and a batch that
changes between the two forms while runs join and leave gives every run the
bits it has alone."""
import numpy as np
import pytest

from oidt_amd import configs
from oidt_amd.solver import Batch

from helpers import device_inputs

NAMES = ('ex', 'ey', 'ez', 'hx', 'hy', 'hz')


def strip(nx, ny, nz, nt, source='TE', seed=5):
    p = configs.strip3d(nz, nx=nx, ny=ny, nt=nt, nf=5, precision='float32', width=12, height=8, port_len=8, buffer_z=6,
                        source_condition=source, source_type=1, gauss_pulse_deg=-1.0)
    p.update(rough_std=15e-9, rough_acl=40e-9, seed=seed)
    s, up, lo, fg = device_inputs(p)
    return s, fg


def outcome(b, slot):
    return [b.field(slot, n) for n in NAMES] + list(b.dft(slot).values())


def alone(run, launch, direction='f'):
    b = Batch('3d', np.float32, max_slots=1)
    b.set_launch(*launch)
    slot = b.add(*run, direction)
    b.advance(-(-run[0].nt // 32))
    b.sync()
    out = outcome(b, slot)
    b.close()
    return out


@pytest.mark.gpu
# (the TM source box does not fit the smallest cross-sections)
@pytest.mark.parametrize('nx,ny,nz,nt,source,direction', [
    (31, 35, 59, 33, 'TE', 'f'), (32, 36, 60, 64, 'TE', 'b'), (33, 37, 61, 45, 'TE', 'f'), (64, 48, 120, 50, 'TE', 'b'),
    (64, 48, 120, 50, 'TM', 'f'), (65, 49, 121, 70, 'TM', 'b'), (97, 61, 182, 47, 'TE', 'f'), (97, 61, 182, 47, 'TM', 'b'),
])
def test_blocked_3d_gives_the_marchs_bits(nx, ny, nz, nt, source, direction):
    run = strip(nx, ny, nz, nt, source)
    print('case', nx, ny, nz, nt, source, direction, flush=True)
    for x, y in zip(alone(run, (4, 0, 1), direction), alone(run, (2, 0, 4), direction)):
        assert np.array_equal(x, y)


@pytest.mark.gpu
def test_default_3d_form_changes_between_chunks():
    """206 MiB of fields join a small run in progress (the blocked step from
    then on) and leave again."""
    small, large = strip(36, 34, 56, 150), strip(150, 150, 400, 50, seed=9)
    print('case', small[0].shape, large[0].shape, flush=True)
    b = Batch('3d', np.float32, max_slots=2)
    ks = b.add(*small)
    b.advance(1)
    kl = b.add(*large)
    b.advance(2)
    b.sync()
    got_large = outcome(b, kl)
    b.remove(kl)
    b.advance(2)
    b.sync()
    got_small = outcome(b, ks)
    b.close()
    for got, run in ((got_small, small), (got_large, large)):
        for x, y in zip(got, alone(run, (4, 0, 1))):
            assert np.array_equal(x, y)
