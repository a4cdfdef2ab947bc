"""Batch steps of blocks whose extents are no multiples of 8, by column tiles
of free extents, against the three-kernel path (kernel path 1), bit for bit.

The shapes reach the edges of the tile layout: its widest rows, its tallest
columns, one column, blocks of one tile (updated in place) and of several
(the last one narrower or lower), each precision (the mixed mode keeps FP64
on these blocks).
"""
from __future__ import annotations

import pytest
import torch

from flash5_amd.hydro import PREC_FP64, PREC_MIXED, Hydro, HydroParams
from tests.test_gpu_fused_update import _batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,nblocks,kw", [
    ((12, 10, 14), 130, {}),                                  # one tile, in place
    ((16, 9, 6), 100, {"RiemannSolver": "hybrid"}),           # two tiles in y, 5 and 4 rows
    ((20, 20, 20), 50, {}),                                   # four tiles of 20 x 5
    ((19, 13, 7), 80, {"use_auxEintEqn": False}),             # 5 + 5 + 3 rows
    ((33, 7, 6), 80, {"RiemannSolver": "hll"}),               # three tiles in x
    ((6, 15, 9), 150, {}),                                    # the tallest tile
    ((18, 6, 5), 150, {"slopeLimiter": "minmod"}),
    ((24, 4, 6), 150, {"slopeLimiter": "hybrid"}),            # wide rows
    ((2, 2, 2), 9, {}),
    ((2, 2, 2), 3000, {}),
    ((12, 10, 8), 150, {"use_steepening": True}),             # scratch: reads planes behind
    ((12, 10, 8), 4, {"hy_fPresInMomFlux": 0.5}),             # the three kernels still
    ((9, 11, 6), 150, {"use_3dFullCTU": False, "use_flattening": False}),
    ((12, 10, 5), 300, {}),                                   # more blocks than compute units
    ((12, 10), 5, {}),                                        # 2-D
    ((20, 17), 5, {"RiemannSolver": "hybrid"}),
    ((7, 6), 300, {"use_steepening": True}),
])
@pytest.mark.parametrize("prec", [PREC_FP64, PREC_MIXED], ids=["fp64", "mixed"])
def test_free_tiles_match_the_three_kernels(shape, nblocks, kw, prec):
    ndim = len(shape)
    shape = tuple(shape) + (1,) * (3 - ndim)
    hp = HydroParams(ndim=ndim, nxb=shape[0], nyb=shape[1], nzb=shape[2], gamma=1.4,
                     eintSwitch=1.0e-4, precision=prec, **kw)
    if hp.RiemannSolver != "hllc":
        hp.nunk, hp.shokVar = 11, 10
    U0 = _batch(hp, nblocks, 5).cuda()
    dx = tuple(1.0 / n for n in shape)
    dt = 0.1 * min(dx[:ndim])
    out = []
    hy = Hydro(hp)
    try:
        for path in (0, 1):
            hy.set_kernel_path(path)
            U = U0.clone()
            for _ in range(2):
                st = hy.advance_batch(U, dt, dx)
            assert st.code == 0
            out.append((U, st.fallbacks))
    finally:
        hy.set_kernel_path(0)
    assert out[0][1] == out[1][1]
    assert not torch.equal(out[0][0], U0)
    assert torch.equal(out[0][0], out[1][0])
