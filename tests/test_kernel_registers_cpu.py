"""Tiles of csrc/kernels/gemm_lds_kernel.h keep their accumulators in registers: a tile that spills took five times its time, with the
right results.  Read from the kernels' metadata in the built library."""
import os
import re
import shutil
import subprocess

import pytest

from shai_amd import native

READELF = shutil.which("llvm-readelf", path="/opt/rocm/llvm/bin")
if READELF is None or not os.path.exists(native.KERNELS_LIB):
    pytest.skip("needs the native library and llvm-readelf", allow_module_level=True)


def spills(tmp_path):
    """{kernel: registers spilled} over the device objects of the library."""
    data, out = open(native.KERNELS_LIB, "rb").read(), {}
    at = [m.start() for m in re.finditer(b"\x7fELF", data)][1:]     # behind the library's own header
    for i, (a, b) in enumerate(zip(at, at[1:] + [len(data)])):
        f = tmp_path / f"{i}.o"
        f.write_bytes(data[a:b])
        notes = subprocess.run([READELF, "--notes", str(f)], capture_output=True, text=True).stdout
        for name, n in re.findall(r"\.name:\s+(_Z\w+).*?\.vgpr_spill_count:\s+(\d+)", notes, re.S):
            out[name] = int(n)
    return out


def test_gemm_tiles_do_not_spill(tmp_path):
    tiles = {k: n for k, n in spills(tmp_path).items() if "gemm2_kernel" in k}
    assert len(tiles) > 100
    assert not {k: n for k, n in tiles.items() if n}
