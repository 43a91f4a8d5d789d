"""The tuner's candidates hold the library's own choice, which is left unset where it wins (CPU)."""
import types

import pytest

from pgj import tune


class _Library:
    """Records the shapes and plans in force; a launch's time is looked up in ``cost``."""

    def __init__(self, cost):
        self.cost, self.shape, self.plans, self.calls = cost, None, [0, 0, 0], []

    def pgj_hex8_set_shape(self, grid, L, es, *shape):
        self.shape = None if shape == (0, 0, 0, 0) else shape
        return 0

    def pgj_hex8_get_shape(self, grid, L, es, out):
        out[:5] = [*(self.shape or (1, 4, 32, 1)), 7]
        return 0

    def pgj_fft_set_plan(self, grid, es, pas, plan):
        self.plans[pas] = max(plan, 0)
        return 0


@pytest.fixture
def library(monkeypatch):
    def make(cost):
        lib = _Library(cost)
        monkeypatch.setattr(tune._lib, 'lib', lambda: lib)
        monkeypatch.setattr(tune, 'time_launch', lambda fn, reps: lib.cost(lib, fn))
        return lib
    return make


@pytest.mark.parametrize('es', [4, 8])
def test_default_shape_wins_and_stays_unset(library, es):
    lib = library(lambda l, fn: 1.0 if l.shape is None else 2.0)
    launches = []
    out = tune.tune_row_march(types.SimpleNamespace(nx=96), 3, es, lambda: launches.append(lib.shape))
    assert lib.shape is None and out == dict(shape=(1, 4, 32, 1), ms=1.0)
    assert launches == [None]      # one launch in the end, for the stages that follow


def test_explicit_shape_wins(library):
    lib = library(lambda l, fn: 0.5 if l.shape == (1, 1, 32, 1) else 2.0)
    out = tune.tune_row_march(types.SimpleNamespace(nx=96), 3, 8, lambda: None)
    assert lib.shape == out['shape'] == (1, 1, 32, 1)


def test_given_candidates_are_the_only_ones(library):
    lib = library(lambda l, fn: 1.0 if l.shape is None else 2.0)
    out = tune.tune_row_march(types.SimpleNamespace(nx=16), 3, 8, lambda: None, candidates=[(1, 2, 4, 0)])
    assert lib.shape == out['shape'] == (1, 2, 4, 0)


@pytest.mark.parametrize('n', [16, 20, 24, 32, 48, 64, 96, 128])
def test_default_plan_wins_and_stays_unset(library, n):
    lib = library(lambda l, fn: 1.0 + sum(l.plans))
    out = tune.tune_fft(types.SimpleNamespace(nx=n), 8, lambda stage: None)
    assert lib.plans == [0, 0, 0]
    assert all(out[k]['plan'] == 0 and '0' in out[k]['ms'] for k in ('fxy', 'fz', 'fxyi'))


def test_explicit_plan_wins(library):
    lib = library(lambda l, fn: 9.0 - sum(l.plans))
    out = tune.tune_fft(types.SimpleNamespace(nx=64), 8, lambda stage: None)
    assert lib.plans == [out[k]['plan'] for k in ('fxy', 'fz', 'fxyi')] == [3, 3, 3]


@pytest.mark.parametrize('gain, kept', [(0.04, True), (0.06, False)])
def test_noise_does_not_replace_the_default(library, gain, kept):
    lib = library(lambda l, fn: 1.0 - gain if l.shape == (1, 4, 8, 0) else 1.0)
    tune.tune_row_march(types.SimpleNamespace(nx=16), 1, 8, lambda: None)
    assert lib.shape == (None if kept else (1, 4, 8, 0))
