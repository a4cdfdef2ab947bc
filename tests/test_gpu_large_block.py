"""A block whose array is longer than 2 GiB, past the column march's byte
offsets: a step of it has the bits of the same cells as two blocks of half the
size (with each other's cells as guards), which the march takes."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def test_block_past_two_gib_matches_its_halves():
    from flash5_amd import workloads as W
    from flash5_amd.hydro import FxError, Hydro, HydroParams
    nx, ny, ng = 8192, 4096, 4
    big = HydroParams(ndim=2, nxb=nx, nyb=ny, nzb=1, gamma=1.4)
    half = HydroParams(ndim=2, nxb=nx, nyb=ny // 2, nzb=1, gamma=1.4)
    U = torch.zeros((1,) + big.block_shape(), dtype=torch.float64, device="cuda")
    assert U.numel() * 8 > 2 ** 31 and U.numel() * 4 < 2 ** 31
    x = torch.arange(nx + 2 * ng, dtype=torch.float64, device="cuda") * 0.37
    y = torch.arange(ny + 2 * ng, dtype=torch.float64, device="cuda")[:, None] * 0.29
    for v, base, amp, ph in ((0, 1.0, 0.4, 0.1), (1, 0.0, 0.8, 1.3), (2, 0.0, 0.8, 2.9),
                             (4, 1.0, 0.4, 4.1)):
        U[:, v] = base + amp * torch.sin(x + ph) * torch.cos(y - ph)
    W.eos_dens_pres(U, big.gamma)
    rows = ny // 2 + 2 * ng
    H = torch.cat([U[:, :, :, :rows], U[:, :, :, ny // 2:]]).contiguous()
    deltas = (1.0 / nx, 1.0 / ny, 1.0)
    dt = 2.0e-5
    print("large block:", tuple(U.shape), flush=True)
    st = Hydro(half).advance_batch(H, dt, deltas)
    hy = Hydro(big)
    sb = hy.advance_batch(U, dt, deltas)
    assert sb.code == st.code == 0
    got = U[0, :, :, ng:-ng, ng:-ng]
    for k in (0, 1):
        want = H[k, :, :, ng:-ng, ng:-ng]
        assert torch.equal(got[:, :, k * (ny // 2):(k + 1) * (ny // 2)], want)
    with pytest.raises(FxError):             # classes take the march alone
        hy.set_block_classes([(nx, ny)])
