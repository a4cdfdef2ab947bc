"""UniformGrid.step calls a program's own fill_guards (a boundary of its own,
say) and hydro.compute_dt: without arguments, before the dt and again after the
detector.  The grid and the hydro unit are stand-ins, so this runs on the CPU."""
import types

import pytest

from flash5_amd import drivers as D
from flash5_amd.hydro import Hydro, HydroParams


class _Hydro(Hydro):
    def __init__(self, log):
        self.log = log

    def shock_detect_batch(self, U, deltas):
        self.log.append("detect")
        return types.SimpleNamespace(min_cell_cfl=0.0)

    def advance_batch(self, U, dt, deltas):
        self.log.append(("advance", dt))
        return types.SimpleNamespace(fallback_cfl=0.0)


def _grid(cls, hydro, log, detect=False):
    grid = object.__new__(cls)
    grid.__dict__.update(params=HydroParams(shokVar=10), hydro=hydro(log), U=None,
                         deltas=(0.1,) * 3, cfl=0.8, t=0.0, nsteps=0, detect=detect,
                         _cfl_next=0.8, log=log)
    grid._fill_guards_dt = lambda cfl: log.append(("fill and dt", cfl)) or 0.5
    return grid


class _OwnFill(D.UniformGrid):
    def fill_guards(self):
        self.log.append("own fill")


class _OwnDt(_Hydro):
    def compute_dt(self, U, deltas, cfl):
        self.log.append(("own dt", cfl))
        return 0.25


@pytest.mark.parametrize("detect", [False, True])
def test_own_fill_and_dt(detect):
    log = []
    assert _grid(_OwnFill, _OwnDt, log, detect).step() == 0.25
    mid = ["detect", "own fill"] if detect else []
    assert log == ["own fill", *mid, ("own dt", 0.8), ("advance", 0.25)]


def test_own_fill_set_on_the_object():
    log = []
    grid = _grid(D.UniformGrid, _OwnDt, log, True)
    grid.fill_guards = lambda: log.append("own fill")
    assert grid.step(dt_max=0.125) == 0.125
    assert log == ["own fill", "detect", "own fill", ("own dt", 0.8), ("advance", 0.125)]


def test_own_fill_set_on_the_class(monkeypatch):
    log = []
    monkeypatch.setattr(D.UniformGrid, "fill_guards", lambda self: log.append("own fill"))
    assert _grid(D.UniformGrid, _OwnDt, log).step() == 0.25
    assert log == ["own fill", ("own dt", 0.8), ("advance", 0.25)]


def test_own_dt_alone():
    log = []

    class Grid(D.UniformGrid):
        pass
    grid = _grid(Grid, _OwnDt, log)
    grid.lib = types.SimpleNamespace(fx_grid_fill_guards_var=lambda *a: log.append("fill"))
    import torch
    import numpy as np
    grid.U, grid.nbr = torch.zeros(2, 10, 9, 9, 9), np.zeros((2, 6), np.int32)
    assert grid.step() == 0.25
    assert log == ["fill", ("own dt", 0.8), ("advance", 0.25)]


def test_one_launch_without_them():
    log = []
    assert _grid(D.UniformGrid, _Hydro, log).step() == 0.5
    assert log == [("fill and dt", 0.8), ("advance", 0.5)]
