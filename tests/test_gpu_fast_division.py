"""The FP64 quotients and roots that the device forms without range handling
(recip_rn, quot, quot_r, sqrt_fast) on the device itself, against IEEE division
and root, bit for bit.  The correction steps round correctly from any start
near enough, save for divisors whose significand is all ones: there 1/y lies a
hair above the midpoint of two doubles and the start has to lie above it, which
only the hardware's estimate can show.  An estimate depends on the significand
alone, so every exponent is tried with that one and its neighbours."""
import ctypes as C
import os

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cdiv", "libdevice_div.so")


def _double(sign, exp, sig):
    b = (sign.astype(np.uint64) << np.uint64(63)) | (sig.astype(np.uint64))
    b |= (exp + 1023).astype(np.uint64) << np.uint64(52)
    return b.view(np.float64)


def _random(rng, n, span):
    """significands random, at both ends of the binade, or short; both signs"""
    sig = rng.integers(0, 1 << 52, n)
    kind = rng.integers(0, 8, n)
    sig = np.where(kind == 0, (1 << 52) - 1 - (sig & 15), sig)
    sig = np.where(kind == 1, sig & 15, sig)
    sig = np.where(kind == 2, sig & 0xFFFFFFFF00000, sig)
    return _double(rng.integers(0, 2, n), rng.integers(-span, span + 1, n), sig)


def _top(rng, reps):
    """every exponent to +-900 and both signs with the 16 highest significands"""
    exp, low, sign = np.meshgrid(np.arange(-900, 901), np.arange(16), [0, 1])
    y = _double(sign.ravel(), exp.ravel(), (1 << 52) - 1 - low.ravel())
    return np.tile(y, reps)


@pytest.mark.parametrize("which", ["all-ones", "random"])
def test_device_quotients_and_roots_are_ieee(which):
    lib = C.CDLL(LIB)
    lib.fx_test_div.argtypes = [C.c_void_p, C.c_void_p, C.c_long, C.c_void_p]
    rng = np.random.default_rng(7)
    if which == "all-ones":
        y = _top(rng, 40)
        x = _random(rng, y.size, 50)
    else:
        x, y = _random(rng, 1 << 23, 400), _random(rng, 1 << 23, 400)
    n = y.size
    dx, dy = torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda()
    out = torch.empty(4, n, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    assert lib.fx_test_div(dx.data_ptr(), dy.data_ptr(), n, out.data_ptr()) == 0
    got = out.cpu().numpy().view(np.uint64)
    want = np.stack([1.0 / y, x / y, x / y, np.sqrt(np.abs(y))]).view(np.uint64)
    for name, a, b in zip(("recip_rn", "quot", "quot_r", "sqrt_fast"), got, want):
        bad = np.flatnonzero(a != b)
        print(which, name, n, bad.size, [(x[i].hex(), y[i].hex()) for i in bad[:4]], flush=True)
        assert bad.size == 0, name
