"""The material given as one byte per cell holds the CB maps' values, for every
scheme and precision and for masks that reach the grid's edges; CB maps asked
for or assigned take its place."""
import numpy as np
import pytest

from oidt_amd import configs, materials
from oidt_amd.solver import RunArrays

COMPS = {'tm': (2,), 'te': (0, 1), '3d': (0, 1, 2)}


def setup(scheme, precision):
    if scheme == '3d':
        p = configs.strip3d(31, nx=37, ny=34, nt=8, nf=2, precision=precision, width=12, height=8, port_len=6, buffer_z=3)
    else:
        p = configs.slab2d(61, ny=47, nt=8, nf=2, precision=precision, scheme=scheme, core=12, port_len=8, buffer_x=4)
    s, _, _ = configs.realise(p)
    return s


@pytest.mark.parametrize('scheme', ['tm', 'te', '3d'])
@pytest.mark.parametrize('precision', ['float32', 'float64'])
@pytest.mark.parametrize('mask', ['random', 'none', 'all', 'bytes'])
def test_material_index_holds_cb_maps(scheme, precision, mask):
    s = setup(scheme, precision)
    fg = np.random.default_rng(3).random(s.shape) < 0.5
    fg = {'none': np.zeros_like(fg), 'all': np.ones_like(fg), 'bytes': fg.astype(np.uint8) * 7}.get(mask, fg)
    index, values = materials.material_index(s, fg)
    assert index.dtype == np.uint8 and index.shape == tuple(s.shape) and values.dtype == s.precision
    for c, ref in zip(COMPS[scheme], materials.cb_maps(s, fg)):
        assert np.array_equal(values[c][(index >> (2 * c)) & 3], ref)


@pytest.mark.parametrize('scheme', ['tm', 'te', '3d'])
def test_run_arrays_give_and_take_cb_maps(scheme):
    s = setup(scheme, 'float32')
    fg = np.random.default_rng(4).random(s.shape) < 0.5
    ra = RunArrays(s, fg)
    assert ra.material is not None
    for got, ref in zip(ra.cb, materials.cb_maps(s, fg)):
        assert np.array_equal(got, ref)
    assert ra.material is None
    ra = RunArrays(s, fg)
    maps = [2 * a for a in materials.cb_maps(s, fg)]
    ra.cb = maps
    assert ra.material is None and ra.cb is maps and ra.inputs().cb[0] == maps[0].ctypes.data
