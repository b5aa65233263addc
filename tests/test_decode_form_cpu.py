"""Which decode attention kernel a launch takes (csrc/kernels/attention.hip), and the switches that force one."""
import os
import subprocess
import sys

import pytest

from shai_amd import native

if not os.path.exists(native.KERNELS_LIB):
    pytest.skip("the native library is not built", allow_module_level=True)

# (rows, query heads, KV heads, head size, splits): one split; up to four workgroups for each of 256 CUs and one more; another group or head size
CALLS = [(1, 32, 8, 128, 1), (300, 32, 8, 128, 1), (2, 32, 8, 128, 64), (3, 32, 8, 128, 64), (32, 32, 8, 128, 4), (33, 32, 8, 128, 4),
         (1, 16, 8, 128, 8), (1, 32, 8, 64, 9), (1, 8, 8, 128, 1)]


def forms(**env):
    code = f"""
from shai_amd import native
print([native.ops().decode_attn_form(*c) for c in {CALLS}])
"""
    own = {k: v for k, v in os.environ.items() if k not in ("SHAI_DECODE_WB", "SHAI_DECODE_PERSIST")}
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = subprocess.run([sys.executable, "-c", code], env={**own, **env, "HIP_VISIBLE_DEVICES": ""}, cwd=root, check=True,
                         capture_output=True, text=True, timeout=300).stdout
    return eval(out.strip().splitlines()[-1])


@pytest.mark.parametrize("env,want", [
    ({}, ["waves", "waves", "waves", "walk", "waves", "items", "items", "walk", "items"]),
    ({"SHAI_DECODE_PERSIST": "1"}, ["waves", "waves", "walk", "walk", "walk", "walk", "walk", "walk", "walk"]),
    ({"SHAI_DECODE_PERSIST": "0"}, ["waves", "waves", "items", "items", "items", "items", "items", "items", "items"]),
    ({"SHAI_DECODE_WB": "0"}, ["items", "items", "walk", "walk", "items", "items", "items", "walk", "items"])])
def test_form_and_switches(env, want):
    assert forms(**env) == want
