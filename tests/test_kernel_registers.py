"""Registers of the built library's kernels that are asked to leave room for a
number of wavefronts: the FP64 face solve fits its three (168 registers) with
next to no spills.  With 14 it took 8.8 instead of 5.7 ms on a grid of 94M faces.
Read from the metadata notes of the library's gfx950 code objects."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from flash5_amd import hydro

READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"


def _code_objects(path):
    data = open(path, "rb").read()
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data):
        base, pos = m.start(), m.end()
        n = struct.unpack_from("<Q", data, pos)[0]
        pos += 8
        for _ in range(n):
            off, size, name = struct.unpack_from("<QQQ", data, pos)
            pos += 24 + name
            if size and b"gfx950" in data[pos - name:pos]:
                yield data[base + off:base + off + size]


@pytest.mark.skipif(not os.path.exists(READELF), reason="needs llvm-readelf")
def test_face_solve_fits_three_waves(tmp_path):
    spills = {}
    for k, obj in enumerate(_code_objects(hydro.LIB_PATH)):
        f = tmp_path / f"{k}.elf"
        f.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(f)], capture_output=True, text=True,
                               check=True).stdout
        for kernel in notes.split("  - .agpr_count:")[1:]:
            name = re.search(r"\.name:\s+(\S+)", kernel)[1]
            spills[name] = int(re.search(r"\.vgpr_spill_count:\s+(\d+)", kernel)[1])
    face = {multi: [v for n, v in spills.items() if f"k_face_solveILb0ELb{multi}Ed" in n]
            for multi in (0, 1)}
    assert face[0] == [0], face
    assert len(face[1]) == 1 and face[1][0] <= 2, face
