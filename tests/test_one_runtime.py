"""A process that loads the library before torch has one HIP runtime."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_library_before_torch_shares_its_runtime():
    code = ("from flash5_amd import hydro\n"
            "hydro.load_library()\n"
            "import torch\n"
            "torch.zeros(1)\n"
            "print(len({l.split()[-1] for l in open('/proc/self/maps') if 'libamdhip64' in l}))\n")
    out = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True,
                         check=True)
    assert out.stdout.split() == ["1"], out.stdout
