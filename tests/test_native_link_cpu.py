"""The in-tree native libraries must dlopen (all symbols resolved) -- catches e.g. kernel launch stubs a
host pass silently dropped, which otherwise only shows up as a load failure on the GPU box."""
import ctypes
import os

import pytest

from shai_amd import native


@pytest.mark.parametrize("lib", [native.KERNELS_LIB, native.LM_LIB, native.RUNTIME_LIB, native.COMM_LIB])
def test_native_library_links(lib):
    if not os.path.exists(lib):
        pytest.skip(f"{lib} not built (python csrc/build.py)")
    if lib == native.COMM_LIB:
        import torch.cuda  # noqa: F401  (resolves libamdhip64 the way native.comm() does)
    ctypes.CDLL(lib, mode=ctypes.RTLD_GLOBAL)


@pytest.mark.skipif(not os.path.exists(native.KERNELS_LIB), reason="kernels are not built")
def test_launchers_say_what_they_do_not_launch():
    """The one-launch GroupNorm of an image whose groups it does not take (here of 3 channels, and of one pixel too many for a fold's
    registers) and a fold of rows that are too wide are errors of the launch; nothing to do is none.  No device is reached."""
    lib, P, INVALID = ctypes.CDLL(native.KERNELS_LIB, mode=ctypes.RTLD_GLOBAL), ctypes.c_void_p, 1

    class GnOne(ctypes.Structure):
        _fields_ = [("x", P), ("x2", P), ("C1", ctypes.c_int), ("parts", P), ("splits", ctypes.c_int), ("bias", P), ("bias2d", P),
                    ("bias2d_ld", ctypes.c_long), ("residual", P), ("res_alpha", ctypes.c_float), ("raw", P), ("gamma", P), ("beta", P),
                    ("out", P), ("N", ctypes.c_int), ("HW", ctypes.c_int), ("C", ctypes.c_int), ("G", ctypes.c_int), ("eps", ctypes.c_float),
                    ("silu", ctypes.c_int)]

    class FoldNorm(ctypes.Structure):
        _fields_ = [("parts", P), ("bias", P), ("residual", P), ("y", P), ("gamma", P), ("beta", P), ("out", P), ("splits", ctypes.c_int),
                    ("rows", ctypes.c_int), ("D", ctypes.c_int), ("rms", ctypes.c_int), ("ldr", ctypes.c_long), ("res_alpha", ctypes.c_float),
                    ("eps", ctypes.c_float)]
    gn, fold = lib._ZN4shai13launch_gn_oneERKNS_9GnOneArgsEP12ihipStream_t, lib._ZN4shai16launch_fold_normERKNS_12FoldNormArgsEP12ihipStream_t
    for f in (gn, fold):
        f.restype, f.argtypes = ctypes.c_int, [P, P]
    one = lambda **a: gn(ctypes.byref(GnOne(**a)), None)  # noqa: E731
    assert one(N=1, HW=64, C=96, G=32) == INVALID and one(N=1, HW=0, C=128, G=32) == INVALID
    assert one(N=1, HW=8193, C=128, G=32, parts=16) == INVALID
    assert one(N=0, HW=64, C=96, G=32) == 0
    assert fold(ctypes.byref(FoldNorm(rows=1, D=2056)), None) == INVALID and fold(ctypes.byref(FoldNorm(rows=0, D=2056)), None) == 0
