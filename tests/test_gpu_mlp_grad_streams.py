"""Gradient calls that overlap: queued on two streams without a wait, and
replayed from a graph beside eager calls.  Sums in one stream's order have the
bits of waiting calls; sums whose order is open differ by the roundings of
their additions alone, at most 2^-23 of the terms' magnitudes each."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

N, CALLS = 131072, 12


@pytest.fixture
def nets():
    from flash5_amd.learned import SeedNet
    gen = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(2, N, 6, generator=gen, device="cuda")
    t = torch.randn(2, N, generator=gen, device="cuda")
    net = SeedNet(seed=3)
    yield net, x, t
    net.lib.fx_hydro_set_stream(None)
    net.lib.fx_hydro_set_async(0)


def _grad(net, x, t, g):
    from flash5_amd.learned import NPARAM, _fp
    assert net.lib.fx_mlp_grad(_fp(net.params), _fp(x), _fp(t), x.shape[0], 2.0 ** -17, _fp(g),
                               _fp(g[NPARAM:])) == 0


def _queue(net, calls):
    """calls: (stream, x, t, gradient), queued without a wait between them"""
    torch.cuda.synchronize()
    net.lib.fx_hydro_set_async(1)
    for stream, x, t, g in calls:
        net.lib.fx_hydro_set_stream(stream.cuda_stream)
        _grad(net, x, t, g)
    torch.cuda.synchronize()
    net.lib.fx_hydro_set_async(0)
    net.lib.fx_hydro_set_stream(None)


def _zeros(*shape):
    from flash5_amd.learned import NPARAM
    return torch.zeros(*shape, NPARAM + 1, device="cuda")


def test_two_streams_with_gradients_of_their_own(nets):
    net, x, t = nets
    want, got, s = _zeros(2), _zeros(2), [torch.cuda.Stream(), torch.cuda.Stream()]
    for k in range(2):
        for _ in range(CALLS):
            _grad(net, x[k], t[k], want[k])
    _queue(net, [(s[k], x[k], t[k], got[k]) for _ in range(CALLS) for k in range(2)])
    assert torch.equal(got, want)
    _grad(net, x[0], t[0], want[0])          # a waiting call behind them
    _grad(net, x[0], t[0], got[0])
    assert torch.equal(got, want)


def test_two_streams_add_to_one_gradient(nets):
    net, x, t = nets
    one, got, s = _zeros(2), _zeros(), [torch.cuda.Stream(), torch.cuda.Stream()]
    for k in range(2):
        _grad(net, x[k], t[k], one[k])
    _queue(net, [(s[k], x[k], t[k], got) for _ in range(CALLS) for k in range(2)])
    want = CALLS * one.double().sum(0)
    assert (got - want).abs().le(2 * CALLS * 2.0 ** -23 * CALLS * one.double().abs().sum(0)).all()


def test_replays_beside_eager_calls(nets):
    net, x, t = nets
    xs, ts = x[0, :384], t[0, :384]          # three workgroups
    part, one, got = _zeros(3), _zeros(), _zeros()
    for k in range(3):
        _grad(net, xs[128 * k:128 * k + 128], ts[128 * k:128 * k + 128], part[k])
    _grad(net, x[1], t[1], one)
    s = [torch.cuda.Stream(), torch.cuda.Stream()]
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    net.lib.fx_hydro_set_async(1)
    net.lib.fx_hydro_set_stream(s[0].cuda_stream)
    with torch.cuda.graph(graph, stream=s[0]):
        _grad(net, xs, ts, got)
    net.lib.fx_hydro_set_stream(s[1].cuda_stream)
    for n in (1, 2, 3):                      # so many replays and eager calls by then
        with torch.cuda.stream(s[0]):
            graph.replay()
        _grad(net, x[1], t[1], got)
        torch.cuda.synchronize()
        want = n * (part.double().sum(0) + one.double())
        size = n * (part.double().abs().sum(0) + one.double().abs())
        assert (got - want).abs().le(4 * n * 2.0 ** -23 * size).all(), n
