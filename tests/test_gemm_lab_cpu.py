"""The GEMM lab's scripts name every source that they have to link: those that define what the listed ones launch."""
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
KERNELS = os.path.join(ROOT, "csrc", "kernels")


def text(name):
    return open(os.path.join(KERNELS, name)).read()


@pytest.mark.parametrize("script", ["build.sh", "build_decode.sh"])
def test_sources_are_listed(script):
    listed = re.search(r"for src in ([\w ]+);", open(os.path.join(ROOT, "tools", "gemm_lab", script)).read())[1].split()
    defined = {}
    for name in os.listdir(KERNELS):
        if name.endswith(".hip"):
            for f in re.findall(r"^(?:hipError_t|void|int|bool) (launch_gemm\w*)\(.*\{$", text(name), re.M):
                defined[f] = name[:-4]
    for src in listed:
        if src.startswith("gemm"):
            for f in re.findall(r"\b(launch_gemm\w*)\(", text(src + ".hip")):
                assert defined.get(f, src) in listed, (src, f, defined[f])
