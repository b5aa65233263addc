"""Kernels that must keep their values in registers: a GEMM tile that spilled took five times its time, a norm with a convolution twice,
with the right results.  Read from the kernels' metadata in the built libraries."""
import os
import re
import shutil
import subprocess

import pytest

from shai_amd import native

READELF = shutil.which("llvm-readelf", path="/opt/rocm/llvm/bin")
if READELF is None or not os.path.exists(native.KERNELS_LIB) or not os.path.exists(native.LM_LIB):
    pytest.skip("needs the native libraries and llvm-readelf", allow_module_level=True)


def spills(lib, tmp_path, what="vgpr_spill_count"):
    """{kernel: registers spilled} over the device objects of a library; ``what``: another of the counts."""
    data, out = open(lib, "rb").read(), {}
    at = [m.start() for m in re.finditer(b"\x7fELF", data)][1:]     # behind the library's own header
    for i, (a, b) in enumerate(zip(at, at[1:] + [len(data)])):
        f = tmp_path / f"{i}.o"
        f.write_bytes(data[a:b])
        notes = subprocess.run([READELF, "--notes", str(f)], capture_output=True, text=True).stdout
        for name, n in re.findall(rf"\.name:\s+(_Z\w+).*?\.{what}:\s+(\d+)", notes, re.S):
            out[name] = int(n)
    return out


def test_gemm_tiles_do_not_spill(tmp_path):
    tiles = {k: n for k, n in spills(native.KERNELS_LIB, tmp_path).items() if "gemm2_kernel" in k}
    assert len(tiles) > 100
    assert not {k: n for k, n in tiles.items() if n}


def test_norms_do_not_spill(tmp_path):
    """Without a convolution; with one of two taps, rows up to 4096 columns."""
    norms = {k: n for k, n in spills(native.LM_LIB, tmp_path).items() if "residual_norm_kernel" in k}
    plain = [k for k in norms if "ELi0ELb" in k]
    conv = [k for k in norms if re.search(r"Li(256|512)ELi[12]ELi2ELb", k)]
    assert len(plain) >= 15 and len(conv) >= 9
    assert not {k: norms[k] for k in plain + conv if norms[k]}


def test_joined_and_fused_kernels_do_not_spill(tmp_path):
    """Kernels that hold the work of two: attention beside a delta rule, a norm in its product, attention with its projection, products whose
    tiles follow each other, the four-wave tile."""
    a, b = spills(native.KERNELS_LIB, tmp_path), spills(native.LM_LIB, tmp_path)
    for lib, name, least in ((b, "attn_rule_kernel", 20), (b, "normed_gemm_kernel", 6), (a, "attn_proj_kernel", 9), (b, "gemm_wide_kernel", 1),
                             (a, "gemm_w4_kernel", 10), (a, "fold_norm_kernel", 6), (a, "skinny3_kernel", 1)):
        found = {k: n for k, n in lib.items() if name in k}
        assert len(found) >= least, name
        assert not {k: n for k, n in found.items() if n}


def test_two_workgroups_a_cu(tmp_path):
    """A norm in its product: the grid is two workgroups of eight waves a CU, which have 128 registers a lane."""
    found = {k: n for k, n in spills(native.LM_LIB, tmp_path, "vgpr_count").items() if "normed_gemm_kernel" in k}
    assert len(found) >= 6 and max(found.values()) <= 128
