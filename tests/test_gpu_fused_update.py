"""Batch steps whose update runs inside the column march, against the same
steps with the update as a kernel of its own (kernel path 2), bit for bit.

The shapes take every route: whole blocks per workgroup (one column tile and
several, the seam rows kept back), scratch and spread (wide blocks, small
batches, contact steepening, 2-D blocks of several tiles), and the separate
update that a pressure share below one in the momentum flux asks for.
"""
from __future__ import annotations

import pytest
import torch

from flash5_amd import workloads as W
from flash5_amd.hydro import PREC_FP64, PREC_MIXED, Hydro, HydroParams

pytestmark = pytest.mark.gpu


def _batch(hp: HydroParams, nblocks: int, seed: int):
    gen = torch.Generator().manual_seed(seed)
    _, nz, ny, nx = hp.block_shape()
    U = torch.zeros((nblocks, hp.nunk, nz, ny, nx), dtype=torch.float64)
    x = torch.arange(nx, dtype=torch.float64) / hp.nxb
    y = torch.arange(ny, dtype=torch.float64)[:, None] / hp.nyb
    z = torch.arange(nz, dtype=torch.float64)[:, None, None] / max(hp.nzb, 1)
    for v, base, amp in ((0, 1.0, 0.4), (1, 0.0, 0.8), (2, 0.0, 0.8), (3, 0.0, 0.8), (4, 1.0, 0.4)):
        k = torch.randint(1, 5, (nblocks, 3), generator=gen).double()
        ph = torch.rand(nblocks, generator=gen, dtype=torch.float64) * 6.0
        arg = ph[:, None, None, None] + 4.0 * (k[:, 0, None, None, None] * x
                                               + k[:, 1, None, None, None] * y
                                               + k[:, 2, None, None, None] * z)
        U[:, v] = base + amp * torch.sin(arg)
    W.eos_dens_pres(U[:, :10], hp.gamma)
    if hp.nunk == 11:                       # some flagged cells for the hybrid switch
        U[:, 10] = (torch.rand(U[:, 10].shape, generator=gen) < 0.2).double()
    return U


@pytest.mark.parametrize("prec", [PREC_FP64, PREC_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("shape,nblocks,kw", [
    ((16, 16, 16), 3, {}),                                # scratch: too few blocks
    ((16, 16, 16), 512, {}),                              # two tiles a workgroup
    ((16, 24, 10), 512, {"RiemannSolver": "hybrid"}),     # three tiles, short columns
    ((16, 8, 2), 5, {}),                                  # one tile, the shortest column
    ((8, 8, 8), 7, {"RiemannSolver": "hll"}),
    ((8, 32, 6), 512, {"use_auxEintEqn": False}),
    ((32, 16, 8), 4, {}),                                 # two tiles across x: scratch
    ((16, 16, 8), 512, {"use_steepening": True}),         # scratch: reads planes behind
    ((16, 16, 8), 512, {"hy_fPresInMomFlux": 0.5}),       # the update on its own
    ((8, 8, 8), 9, {"use_3dFullCTU": False, "use_flattening": False}),
    ((16, 16), 5, {}),                                    # 2-D, scratch
    ((8, 8), 5, {"RiemannSolver": "hybrid"}),             # 2-D, one tile
    ((8, 24), 300, {}),
])
def test_update_in_the_march_matches_the_separate_update(shape, nblocks, kw, prec):
    ndim = len(shape)
    shape = tuple(shape) + (1,) * (3 - ndim)
    hp = HydroParams(ndim=ndim, nxb=shape[0], nyb=shape[1], nzb=shape[2], gamma=1.4,
                     eintSwitch=1.0e-4, precision=prec, **kw)
    if hp.RiemannSolver in ("hll", "hybrid"):
        hp.nunk, hp.shokVar = 11, 10
    print("fused update:", shape, nblocks, kw, prec, flush=True)
    U0 = _batch(hp, nblocks, seed=11)
    deltas = tuple(1.0 / n for n in shape)
    dt = W.cfl_dt(U0, ndim, 4, deltas, 0.4)
    hy = Hydro(hp)
    out = []
    try:
        for path in (2, 0):
            hy.set_kernel_path(path)
            U = U0.cuda()
            for _ in range(2):
                st = hy.advance_batch(U, dt, deltas)
            assert st.code == 0
            out.append((U, st.fallbacks))
    finally:
        hy.set_kernel_path(0)
    assert out[0][1] == out[1][1]
    assert torch.isfinite(out[0][0]).all()
    assert torch.equal(out[0][0], out[1][0])
    assert not torch.equal(out[0][0], U0.cuda())
