"""The autotuner's cached choice is taken only with the library build it was
measured with."""
import json

import pytest

from oidt_amd import autotune, configs


@pytest.fixture
def timed(monkeypatch):
    """Candidates' times without a device: smaller x-chunk, shorter step."""
    timed = []

    def step_time(runs, variant, xchunk, grid=0, chunks=2):
        timed.append((variant, xchunk, grid))
        return float(xchunk)
    monkeypatch.setattr(autotune, 'step_time', step_time)
    return timed


def tune(path):
    s, _, _ = configs.realise(configs.small('tm', 'float32'))
    return autotune.tune([(s, None)], candidates=[(2, 4, 0), (4, 8, 0)], cache_path=str(path))[0]


def test_choice_is_kept_for_the_same_build(tmp_path, timed):
    path = tmp_path / 'tune.json'
    assert tune(path) == (2, 4, 0) and timed
    timed.clear()
    assert tune(path) == (2, 4, 0) and not timed


@pytest.mark.parametrize('build', ['another', None])
def test_choice_of_another_build_is_measured_again(tmp_path, timed, build):
    path = tmp_path / 'tune.json'
    tune(path)
    cache = json.loads(path.read_text())
    for entry in cache.values():
        entry['choice'] = [4, 8, 0]
        entry.pop('build', None)
        if build:
            entry['build'] = build
    path.write_text(json.dumps(cache))
    timed.clear()
    assert tune(path) == (2, 4, 0) and timed


def test_build_follows_the_library(tmp_path, monkeypatch):
    a, b = tmp_path / 'a.so', tmp_path / 'b.so'
    a.write_bytes(b'one')
    b.write_bytes(b'two')
    ids = []
    for p in (a, b, a):
        monkeypatch.setattr(autotune._lib, 'LIB_PATH', str(p))
        ids.append(autotune.build_id())
    assert ids[0] == ids[2] != ids[1]
