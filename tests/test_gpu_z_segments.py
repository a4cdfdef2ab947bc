"""Small 3-D batches, whose column tiles the march cuts along z, against the
same blocks in a batch large enough to take them whole, bit for bit, with the
same count of first-order states."""
from __future__ import annotations

import pytest
import torch

from flash5_amd import workloads as W
from flash5_amd.hydro import PREC_FP64, PREC_MIXED, Hydro, HydroParams
from tests.test_gpu_fused_update import _batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path", [0, 2])
@pytest.mark.parametrize("prec", [PREC_FP64, PREC_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("shape,nblocks,kw", [
    ((16, 16, 16), 1, {}),                                # as short as segments get
    ((16, 16, 16), 24, {}),
    ((16, 8, 17), 20, {"RiemannSolver": "hybrid"}),       # a shorter last segment
    ((8, 8, 8), 30, {"slopeLimiter": "mc"}),
    ((32, 32, 5), 3, {}),
    ((16, 16, 9), 10, {"use_steepening": True}),
    ((16, 16, 16), 10, {"hy_fPresInMomFlux": 0.5}),
    ((16, 16, 16), 10, {"RiemannSolver": "exact"}),
    ((8, 16, 2), 4, {}),
    ((12, 10, 14), 20, {}),                               # free tiles
    ((9, 7, 30), 20, {"use_3dFullCTU": False}),
])
def test_segments_match_whole_columns(shape, nblocks, kw, prec, path):
    hp = HydroParams(ndim=3, nxb=shape[0], nyb=shape[1], nzb=shape[2], gamma=1.4,
                     eintSwitch=1.0e-4, precision=prec, **kw)
    if hp.RiemannSolver == "hybrid":
        hp.nunk, hp.shokVar = 11, 10
    copies = -(-1100 // nblocks)
    U0 = _batch(hp, nblocks, 31)
    U0[:, 4] = U0[:, 4] * 0.02 + 0.001                    # cold: some states fall back
    W.eos_dens_pres(U0[:, :10], hp.gamma)
    dx = tuple(1.0 / n for n in shape)
    dt = W.cfl_dt(U0, 3, 4, dx, 0.3)
    hy = Hydro(hp)
    out = []
    try:
        hy.set_kernel_path(path)
        for n in (1, copies):
            U = U0.cuda().repeat(n, 1, 1, 1, 1)
            st = hy.advance_batch(U, dt, dx)
            out.append((U[:nblocks], st.code, st.fallbacks))
    finally:
        hy.set_kernel_path(0)
    assert out[0][1] == out[1][1] == 0
    assert out[0][2] * copies == out[1][2]
    assert torch.isfinite(out[0][0]).all()
    assert torch.equal(out[0][0], out[1][0])
    assert not torch.equal(out[0][0], U0.cuda())


@pytest.mark.parametrize("shape,nblocks", [((16, 16, 16), 1), ((8, 8, 17), 60), ((12, 10, 5), 7),
                                           ((8, 8, 2), 3), ((16, 16), 5)])
def test_detector_segments_match_whole_tiles(shape, nblocks):
    ndim = len(shape)
    s3 = tuple(shape) + (1,) * (3 - ndim)
    hp = HydroParams(ndim=ndim, nxb=s3[0], nyb=s3[1], nzb=s3[2], gamma=1.4,
                     RiemannSolver="hybrid", nunk=11, shokVar=10, shockLowerCFL=True)
    U0 = _batch(hp, nblocks, 41)
    gen = torch.Generator().manual_seed(3)
    U0[:, 4] *= 1.0 + 4.0 * (torch.rand(U0[:, 4].shape, generator=gen) < 0.3)
    U0[:, 1:4] *= 3.0
    copies = -(-1100 // nblocks)
    hy = Hydro(hp)
    out = []
    for n in (1, copies):
        U = U0.cuda().repeat(n, 1, 1, 1, 1)
        U[:, 10] = 7.0                                    # every cell is written
        st = hy.shock_detect_batch(U, tuple(1.0 / k for k in s3))
        out.append((U, st.min_cell_cfl))
    flags = out[0][0][:, 10]
    assert set(flags.unique().tolist()) == {0.0, 1.0}
    assert out[0][1] == out[1][1] > 0.0
    assert torch.equal(out[0][0].repeat(copies, 1, 1, 1, 1), out[1][0])
