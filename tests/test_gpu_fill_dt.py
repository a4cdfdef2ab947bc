"""The guard fill that takes the CFL dt along, against the fill and the dt as
two calls, bit for bit; and captured runs, whose steps keep a dt each, against
eager steps over several replays."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest
import torch

from flash5_amd import drivers
from flash5_amd.hydro import HydroParams
from tests.test_gpu_fused_update import _batch

pytestmark = pytest.mark.gpu


def _grid(shape, nb, periodic, **kw):
    ndim = len(shape)
    s3 = tuple(shape) + (1,) * (3 - ndim)
    hp = HydroParams(ndim=ndim, nxb=s3[0], nyb=s3[1], nzb=s3[2], gamma=1.4, eintSwitch=1.0e-4, **kw)
    if kw.get("RiemannSolver") == "hybrid":
        hp.nunk, hp.shokVar = 11, 10
    U = _batch(hp, int(np.prod(nb)), 17)
    nbr = drivers.uniform_neighbors(nb, (periodic,) * ndim, ndim)
    return drivers.UniformGrid(hp, U, nbr, [1.0 / (n * b) for n, b in zip(shape, nb)]
                               + [1.0] * (3 - ndim), 0.4)


CASES = [((8, 8), (2, 2), True, {}), ((12, 10), (3, 2), False, {}),
         ((16, 16), (40, 40), True, {}),              # more blocks than compute units
         ((8, 8, 8), (2, 3, 2), False, {"RiemannSolver": "hybrid"}), ((64,), (5,), True, {})]


@pytest.mark.parametrize("shape,nb,periodic,kw", CASES)
def test_fill_with_dt_matches_two_calls(shape, nb, periodic, kw):
    grid = _grid(shape, nb, periodic, **kw)
    U0 = grid.U.clone()
    for scale in (1.0, 4.0, 0.25):                    # the minimum of one call is not the next one's
        grid.U.copy_(U0)
        grid.U[:, 1:4] *= scale
        two = grid.U.clone()
        dt = grid._fill_guards_dt(0.4)
        one, grid.U = grid.U, two
        grid.fill_guards()
        assert dt == grid.hydro.compute_dt(two, grid.deltas, 0.4)
        assert torch.equal(one, two)
        grid.U = one


@pytest.mark.parametrize("shape,nb,periodic,kw", CASES[:2] + CASES[3:4])
def test_captured_steps_match_eager_steps(shape, nb, periodic, kw):
    eager, graph = _grid(shape, nb, periodic, **kw), _grid(shape, nb, periodic, **kw)
    for steps, replays in ((3, 3), (70, 2)):          # more steps than one wavefront's lanes
        for _ in range(steps * replays):
            eager.step()
        t = graph.run_graph(steps, replays)
        torch.cuda.synchronize()
        assert torch.equal(eager.U, graph.U)
        assert t > 0.0 and graph.t == pytest.approx(eager.t, rel=1e-13)


def test_bad_arguments_are_refused():
    grid = _grid((8, 8), (2, 2), True)
    lib, st, dt = grid.lib, drivers.FxStatus(), C.c_double(0.0)
    U = C.cast(C.c_void_p(grid.U.data_ptr()), C.POINTER(C.c_double))
    bad = np.full_like(grid.nbr, 99)
    rc = lib.fx_grid_fill_guards_dt(U, grid.U.shape[0], grid.U[0].numel(),
                                    bad.ctypes.data_as(C.POINTER(C.c_int)),
                                    (C.c_double * 3)(*grid.deltas), 0.4, C.byref(dt), C.byref(st))
    assert rc == 3 and st.code == 3
