"""The FP64 quotients and roots that the device code forms without range
handling (recip_fast, recip_rn, quot_r, sqrt_fast in
flash5_amd/csrc/fx_device.hpp) against IEEE division and square root, on the
CPU: the same steps from starts as far off as the hardware's estimates (and
farther) must give the IEEE bits over the exponent window they are used in.
glibc's fma is correctly rounded, as the device's v_fma_f64 is."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("gcc") is None, reason="needs gcc")
def test_fast_quotients_and_roots_match_ieee(tmp_path):
    exe = str(tmp_path / "fdc")
    subprocess.run(["gcc", "-O2", "-ffp-contract=off", "-o", exe,
                    os.path.join(HERE, "cdiv", "fast_div_check.c"), "-lm"], check=True)
    out = subprocess.run([exe, "10000000"], capture_output=True, text=True, check=False)
    rows = [line.split() for line in out.stdout.strip().splitlines()]
    assert [r[0] for r in rows] == ["recip_rn", "quot", "quot_shared", "sqrt"]
    for name, tried, bad in rows:
        assert int(tried) == 10_000_000 and int(bad) == 0, (name, tried, bad)
    assert out.returncode == 0
