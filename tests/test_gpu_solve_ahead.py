"""Exact-solver batch steps whose high faces are solved for several planes at a
time, at block heights around and between those groups, against the face
solve and the update as kernels of their own (kernel path 2), bit for bit."""
from __future__ import annotations

import pytest
import torch

from flash5_amd import learned as L
from flash5_amd import workloads as W
from flash5_amd.hydro import PREC_FP64, PREC_MIXED, Hydro, HydroParams
from tests.test_gpu_fused_update import _batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nblocks", [4, 260])        # apart as well, and in one kernel
@pytest.mark.parametrize("prec,gate", [(PREC_FP64, None), (PREC_MIXED, None), (PREC_MIXED, 0.05),
                                       (PREC_MIXED, 0.0), (PREC_FP64, 0.05)],
                         ids=["fp64", "mixed", "learned", "learned_all", "fp64_learned"])
@pytest.mark.parametrize("shape", [(16, 16, 2), (16, 16, 7), (16, 16, 8), (16, 16, 9),
                                   (16, 16, 17), (8, 16, 24), (16, 8, 5), (8, 8, 11)])
def test_solve_and_update_at_every_height(shape, prec, gate, nblocks):
    seeded = gate is not None
    hp = HydroParams(ndim=3, nxb=shape[0], nyb=shape[1], nzb=shape[2], gamma=1.4,
                     RiemannSolver="exact", precision=prec, learnedSeed=seeded)
    U0 = _batch(hp, nblocks, 23)
    dx = tuple(1.0 / n for n in shape)
    dt = W.cfl_dt(U0, 3, 4, dx, 0.4)
    hy = Hydro(hp)
    out = []
    try:
        if seeded:
            gen = torch.Generator().manual_seed(5)
            hy.set_seed_params((torch.randn(L.NPARAM, generator=gen) * 0.1).float().cuda())
            L.set_gate(gate)
        for path in (2, 0):
            hy.set_kernel_path(path)
            U = U0.cuda()
            for _ in range(2):
                st = hy.advance_batch(U, dt, dx)
                assert st.code == 0
            out.append((U, st.newton_iters, st.newton_fallbacks))
    finally:
        hy.set_kernel_path(0)
        if seeded:
            L.set_gate(0.2)
            hy.set_seed_params(None)
    assert torch.equal(out[0][0], out[1][0])
    assert out[0][1:] == out[1][1:]
    assert not torch.equal(out[0][0], U0.cuda())
