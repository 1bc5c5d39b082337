"""A run is given to the library by what its object's ``inputs()`` returns: the
material index stands in only for a RunArrays' own ``inputs()``."""
import numpy as np
import pytest

from oidt_amd import configs, materials, solver
from oidt_amd.solver import Batch, RunArrays, Solver


class Recorder:
    """The library's calls, each succeeding without a device."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            self.calls.append((name, args))
            return 0
        return call


@pytest.fixture
def calls(monkeypatch):
    rec = Recorder()
    monkeypatch.setattr(solver, 'lib', lambda: rec)
    return rec.calls


def arrays_of(cls):
    s, up, lo = configs.realise(configs.small('tm', 'float32'))
    return s, cls(s, materials.fg_mask(s, up, lo))


class Overridden(RunArrays):
    def inputs(self):
        r = super().inputs()
        self.maps = [2 * a for a in self.cb]
        r.cb[0] = self.maps[0].ctypes.data
        return r


class OwnMaps(RunArrays):
    @property
    def cb(self):
        return self.__dict__.setdefault('maps', [np.ones(self.setup.shape, np.float32)])


class Other:
    """No RunArrays, with an attribute of that name."""
    material = 'silicon'

    def __init__(self, s, fg):
        self.run = RunArrays(s, fg)
        self.maps = self.run.cb

    def desc(self):
        return self.run.desc()

    def inputs(self):
        return self.run.inputs()


def create(arrays, s, batch):
    if not batch:
        return Solver.from_arrays(arrays, s.nt)
    b = Batch.__new__(Batch)
    b.h, b.runs = None, {}
    b.add_arrays(arrays, s)
    return b


@pytest.mark.parametrize('batch', [False, True])
@pytest.mark.parametrize('cls', [Overridden, OwnMaps, Other])
def test_own_inputs_are_what_the_library_reads(calls, cls, batch):
    s, arrays = arrays_of(cls)
    keep = create(arrays, s, batch)
    name, args = calls[0]
    assert name == ('oidt_batch_add' if batch else 'oidt_solver_create')
    inputs = args[2 if batch else 1]._obj
    assert inputs.cb[0] == arrays.maps[0].ctypes.data
    del keep


@pytest.mark.parametrize('batch', [False, True])
def test_run_arrays_go_by_material_index(calls, batch):
    s, arrays = arrays_of(RunArrays)
    keep = create(arrays, s, batch)
    name, args = calls[0]
    assert name == ('oidt_batch_add_indexed' if batch else 'oidt_solver_create_indexed')
    assert arrays.material is not None and not args[2 if batch else 1]._obj.cb[0]
    del keep


@pytest.mark.parametrize('batch', [False, True])
def test_an_instances_own_inputs(calls, batch):
    s, arrays = arrays_of(RunArrays)
    given = arrays.inputs()
    arrays.cb = None
    arrays.material = materials.material_index(s, np.zeros(s.shape, bool))
    arrays.inputs = lambda: given
    keep = create(arrays, s, batch)
    name, args = calls[0]
    assert name == ('oidt_batch_add' if batch else 'oidt_solver_create')
    assert args[2 if batch else 1]._obj is given
    del keep
