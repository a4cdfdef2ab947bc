"""The batch autotuner times the step that advance_batch runs: with the update
inside the march the whole step, whose only choice is the column-tile width;
else the flux stages.  It leaves the batch as it was, and the steps after it
have the bits of an untuned one."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("solver,path,wide,want", [
    ("HLLC", 0, 16, {(16, 0), (8, 0)}),
    ("hybrid", 0, 8, {(8, 0)}),
    ("HLLC", 2, 16, None), ("exact", 0, 16, None),   # None: the flux stages' candidates
])
def test_batch_autotuner_times_the_batch_step(solver, path, wide, want, prec):
    from flash5_amd import workloads as W
    from flash5_amd.hydro import PREC_FP64, PREC_MIXED, Hydro, HydroParams
    from tests.test_gpu_fused_update import _batch
    hp = HydroParams(ndim=3, nxb=wide, nyb=16, nzb=8, gamma=1.4, RiemannSolver=solver,
                     precision=PREC_FP64 if prec == "fp64" else PREC_MIXED)
    if solver == "hybrid":
        hp.nunk, hp.shokVar = 11, 10
    U0 = _batch(hp, 300, 23)
    deltas = (1.0 / wide, 1.0 / 16, 1.0 / 8)
    dt = W.cfl_dt(U0, 3, 4, deltas, 0.4)
    if want is None:
        want = {(tx, occ) for tx in (16, 8) for occ in ((0,) if prec == "fp64" else (0, 4))}
    hy = Hydro(hp)
    steps = []
    try:
        hy.set_kernel_path(path)
        for tuned in (False, True):
            U = U0.cuda()
            if tuned:
                res = hy.autotune_batch(U, dt, deltas, reps=2)
                print(solver, path, prec, res, flush=True)
                assert {(r["tile_x"], r["occupancy"]) for r in res} == want
                assert sum(r["chosen"] for r in res) == 1 and all(r["ms"] > 0 for r in res)
                assert torch.equal(U, U0.cuda())
            for _ in range(2):
                hy.advance_batch(U, dt, deltas)
            steps.append(U)
    finally:
        hy.autotune_reset()
        hy.set_kernel_path(0)
    assert torch.equal(steps[0], steps[1])
