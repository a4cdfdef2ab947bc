"""The network gradient's sums over samples: at sizes around a wavefront's 32
and a workgroup's 128 samples, and past one set per workgroup, the gradient is
the sum of the single samples' gradients.  Each sample's terms are the same
FP32 numbers in both (bf16 products are exact in FP32), so the two differ by
the FP32 additions alone: at most some 200 a parameter (128 of a set, the sets
of a workgroup, a quarter of 256 rows and 4 parts), of rounding or truncation
2^-23 each."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 31, 33, 129, 300, 256 * 128 + 77])
def test_gradient_is_the_sum_of_samples(n):
    from flash5_amd.learned import NPARAM, SeedNet, _fp
    gen = torch.Generator(device="cuda").manual_seed(n)
    net = SeedNet(seed=3)
    x = torch.randn(n, 6, generator=gen, device="cuda")
    t = torch.randn(n, generator=gen, device="cuda")
    scale = 2.0 ** -10

    def grad(a, b, g):
        rc = net.lib.fx_mlp_grad(_fp(net.params), _fp(a), _fp(b), a.shape[0], scale,
                                 _fp(g), _fp(g[NPARAM:]))
        assert rc == 0

    got = torch.zeros(NPARAM + 1, device="cuda")
    grad(x, t, got)
    want = torch.zeros(NPARAM + 1, dtype=torch.float64, device="cuda")
    size = torch.zeros_like(want)
    for i in range(0, n, 4096):
        m = min(4096, n - i)
        one = torch.zeros(m, NPARAM + 1, device="cuda")
        for k in range(m):
            grad(x[i + k:i + k + 1], t[i + k:i + k + 1], one[k])
        want += one.double().sum(0)
        size += one.double().abs().sum(0)
    assert (got.double() - want).abs().le(200 * 2.0 ** -23 * size).all()
    # a second call adds to what is there
    again = got.clone()
    grad(x, t, again)
    assert torch.allclose(again, 2 * got, rtol=1e-6, atol=0)
