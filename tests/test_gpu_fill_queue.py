"""Guard fills queued without a wait keep the neighbour table they were queued
with, also when the next call brings another table before they have run."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _grids():
    from flash5_amd.drivers import UniformGrid
    from flash5_amd.hydro import HydroParams
    p = HydroParams(ndim=2, nxb=8, nyb=8, nzb=1)
    rng = np.random.default_rng(3)
    out = []
    for nb in (20000, 300):
        U = torch.from_numpy(rng.standard_normal((nb,) + p.block_shape()))
        nbr = rng.integers(-2, nb, size=(nb, 6)).astype(np.int32)
        out.append(UniformGrid(p, U, nbr, (0.1, 0.1, 0.1)))
    return out


@pytest.mark.parametrize("own_stream", [False, True], ids=["default", "non-blocking"])
def test_queued_fills_keep_their_table(own_stream):
    a, b = _grids()
    for grid in (a, b):
        grid.fill_guards()
    want = [grid.U.clone() for grid in (a, b)]
    for grid in (a, b):                      # guard cells out of date again
        inner = grid.U[:, :, :, 4:-4, 4:-4].clone()
        grid.U.fill_(-1.0)
        grid.U[:, :, :, 4:-4, 4:-4] = inner
    torch.cuda.synchronize()
    stream = torch.cuda.Stream() if own_stream else None
    a.hydro.set_stream(stream)
    try:
        for _ in range(20):                  # the last of them behind the first ones
            a.fill_guards(wait=False)
        b.fill_guards(wait=False)
        a.fill_guards(wait=False)
        b.fill_guards(wait=False)
        torch.cuda.synchronize()
    finally:
        a.hydro.set_stream(None)
    assert torch.equal(a.U, want[0]) and torch.equal(b.U, want[1])
