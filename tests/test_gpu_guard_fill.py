"""The one-launch guard fill against three passes, one per axis, in numpy:
the same bits for every neighbour table (blocks, outflow, reflecting sides,
asymmetric ones), block shape and variable count, all variables or one."""
import itertools

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

NG = 4


def fill_passes(U, nbr, ndim, vel, only=None):
    """Axis by axis: later axes interior, earlier ones guard-inclusive."""
    U = U.copy()
    nb = U.shape[0]
    for axis in range(ndim):
        ax = 4 - axis                      # array axis of (b, v, z, y, x)
        n = U.shape[ax] - 2 * NG
        rows = [slice(None)] * 5
        for later in range(axis + 1, ndim):
            rows[4 - later] = slice(NG, U.shape[4 - later] - NG)
        old = U.copy()
        for b, side, gg in itertools.product(range(nb), (0, 1), range(1, NG + 1)):
            t = nbr[b, 2 * axis + side]
            d = NG + n - 1 + gg if side else NG - gg
            if t >= 0:
                s = NG + gg - 1 if side else NG + n - gg
            elif t == -2:
                s = NG + n - gg if side else NG + gg - 1
            else:
                s = NG + n - 1 if side else NG
            src, dst = list(rows), list(rows)
            src[0], src[ax] = (t if t >= 0 else b), s
            dst[0], dst[ax] = b, d
            val = old[tuple(src)].copy()
            if t == -2:
                val[vel[axis]] *= -1.0
            for v in (range(U.shape[1]) if only is None else [only]):
                U[tuple(dst)][v] = val[v]
    return U


@pytest.mark.parametrize("ndim,n,nunk", [(1, (5, 1, 1), 10), (2, (4, 4, 1), 10), (2, (16, 7, 1), 17),
                                         (3, (4, 4, 4), 11), (3, (12, 10, 14), 10),
                                         (3, (8, 16, 5), 25)])
def test_fill_equals_axis_passes(ndim, n, nunk):
    from flash5_amd.drivers import UniformGrid
    from flash5_amd.hydro import HydroParams
    nb = 7
    rng = np.random.default_rng(11 * nunk + n[0])
    p = HydroParams(ndim=ndim, nxb=n[0], nyb=n[1], nzb=n[2], nunk=nunk)
    shape = (nb, nunk) + tuple(n[a] + 2 * NG if a < ndim else 1 for a in (2, 1, 0))
    U = rng.standard_normal(shape)
    nbr = rng.integers(-2, nb, size=(nb, 6)).astype(np.int32)
    g = UniformGrid(p, U, nbr, (0.1, 0.1, 0.1))
    vel = [p.var[1], p.var[2], p.var[3]]
    g.fill_guards(nunk - 1)
    torch.cuda.synchronize()
    want = fill_passes(U, nbr, ndim, vel, only=nunk - 1)
    assert np.array_equal(g.U.cpu().numpy(), want)
    g.fill_guards()
    torch.cuda.synchronize()
    assert np.array_equal(g.U.cpu().numpy(), fill_passes(want, nbr, ndim, vel))
