"""The FP64 exact solver's two builds, quotients without range handling inside
a window of states and plain ones outside it, bit for bit.  A wavefront with one
problem scaled out of the window takes the plain build as a whole, so its other
problems have to give what they give without it, iterations included; and a
block whose densities and pressures are scaled by a power of two goes through
the same arithmetic with other exponents."""
import pytest
import torch

from flash5_amd import learned, workloads as W
from flash5_amd.hydro import Hydro, HydroParams

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("a,b", [(0, 0), (80, 80), (120, 120), (-120, 0), (-100, 100), (0, 140)])
@pytest.mark.parametrize("seeded", [False, True])
def test_a_problem_outside_changes_no_other(a, b, seeded):
    S = learned.sample_interfaces(5000, seed=3)
    net = learned.init_params(4) if seeded else None
    scale = torch.tensor([2.0 ** a, 2.0 ** ((b - a) // 2), 2.0 ** b] * 2, dtype=torch.float64,
                         device="cuda")[:, None]
    p0, it0 = learned.solve(S, 1.4, net)[:2]
    p1, it1 = learned.solve((S * scale).contiguous(), 1.4, net)[:2]
    # one problem outside among those inside
    M = S.clone()
    M[:, ::64] = (S * scale)[:, ::64]
    p2, it2 = learned.solve(M.contiguous(), 1.4, net)[:2]
    want, itw = p0.clone(), it0.clone()
    want[::64], itw[::64] = p1[::64], it1[::64]
    assert torch.equal(p2, want) and torch.equal(it2, itw)


@pytest.mark.parametrize("shape,path", [((16, 16, 8), 0), ((16, 16, 8), 2), ((12, 10, 6), 0),
                                        ((16, 16, 1), 0)])
def test_scaled_blocks_step_alike(shape, path):
    ndim = 3 if shape[2] > 1 else 2
    hp = HydroParams(ndim=ndim, nxb=shape[0], nyb=shape[1], nzb=shape[2], gamma=1.4,
                     RiemannSolver="exact")
    gen = torch.Generator().manual_seed(5)
    U = torch.zeros((6,) + tuple(hp.block_shape()), dtype=torch.float64)
    for v, base, amp in ((0, 1.0, 0.4), (1, 0.0, 0.8), (2, 0.0, 0.8), (3, 0.0, 0.8), (4, 1.0, 0.4)):
        U[:, v] = base + amp * (2 * torch.rand(U[:, v].shape, generator=gen, dtype=torch.float64) - 1)
    W.eos_dens_pres(U[:, :10], hp.gamma)
    out = []
    for e in (0, 120):
        V = U.clone()
        V[:, [0, 4]] *= 2.0 ** e
        V = V.cuda()
        h = Hydro(hp)
        h.set_kernel_path(path)
        h.advance_batch(V, 1e-3, (0.1, 0.1, 0.1))
        h.set_kernel_path(0)
        V[:, [0, 4]] *= 2.0 ** -e
        out.append(V.cpu())
    assert torch.equal(out[0], out[1])
