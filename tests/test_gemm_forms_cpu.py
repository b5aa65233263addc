"""Which kernel a product of a decoder block runs on, at the borders of the rules in csrc/lm: those sizes were measured on both sides."""
import os

import pytest

from shai_amd import native
from shai_amd.ops import lm

if not os.path.exists(native.LM_LIB):
    pytest.skip("the native library is not built", allow_module_level=True)


def form(*args):
    return native.lm_ops().lm_gemm_form(*args)


@pytest.mark.parametrize("M,N,K,want", [
    (8, 8192, 2048, "stream"), (9, 5120, 2048, "ring"), (9, 7232, 2048, "stream"), (12, 17424, 2048, "ring"),      # many columns
    (16, 2048, 2048, "stream"), (17, 2048, 2048, "ring"), (17, 4096, 1024, "stream"), (24, 4096, 1024, "ring"),    # few columns
    (32, 512, 768, "ring"), (33, 2048, 8192, "stream"), (33, 2304, 512, "ring"), (64, 508, 4096, "stream"), (64, 4096, 448, "stream"),
    (32, 32768, 2048, "stream"), (32, 32768, 3072, "ring"), (33, 32768, 512, "ring")])                             # more than a round
def test_few_rows(M, N, K, want):
    assert form(M, N, K) == want


@pytest.mark.parametrize("M,N,K,splits,want", [
    (16, 1024, 2048, 4, "stream"), (17, 1024, 2048, 4, "ring"), (1, 2048, 8192, 8, "ring"), (8, 2048, 4096, 8, "stream"),
    (9, 2048, 4096, 8, "ring"), (1, 2304, 4096, 4, "ring"), (1, 3072, 4032, 4, "stream"), (16, 1024, 4096, 4, "stream"),
    (1, 8192, 4096, 4, "stream"), (32, 8192, 512, 4, "stream"), (33, 8192, 512, 4, "ring"),
    (9, 2048, 4096, 4, "ring"), (8, 2048, 8128, 4, "stream"), (1, 1792, 8192, 4, "ring"), (16, 1728, 8192, 4, "stream"),
    (16, 512, 8192, 8, "stream"), (17, 512, 8192, 8, "ring"), (16, 832, 8192, 8, "stream"), (1, 896, 8192, 8, "ring")])
def test_parts(M, N, K, splits, want):
    assert form(M, N, K, splits) == want


# partial sums: eight where four would leave CUs idle, and of many rows and a long K; a norm pays for every one of them
@pytest.mark.parametrize("M,N,K,want", [
    (1, 2048, 8448, 4), (24, 2048, 12544, 4), (25, 2048, 9216, 8), (64, 2048, 9152, 4), (64, 2056, 12544, 4), (1, 1792, 8448, 4),
    (1, 1784, 4096, 8), (1, 1784, 4032, 4), (16, 1024, 5056, 4), (16, 1024, 5120, 8), (17, 1024, 4096, 8), (1, 512, 4096, 8), (1, 8192, 512, 4),
    (1, 8193, 512, 1), (1, 2048, 448, 1), (65, 2048, 8448, 4), (600, 8192, 4096, 1)])
def test_number_of_parts(M, N, K, want):
    assert lm.parts(M, N, K) == want


# 64 x 64 tiles up to two for each CU, more with a K of 2048; 128 x 128 up to one; 256 x 256 from 192 on
@pytest.mark.parametrize("M,N,K,splits,want", [
    (512, 4096, 512, 1, "64x64 of 4"), (600, 4096, 1984, 1, "64x64"), (600, 4096, 2048, 1, "64x64 of 4"), (600, 4096, 2112, 1, "128x128 of 4"),
    (1024, 4096, 512, 1, "128x128 of 4"), (1025, 4096, 512, 1, "128x128"), (600, 2048, 8192, 3, "128x128 of 4"),
    (600, 2048, 8192, 4, "128x128"), (4096, 3072, 1600, 1, "wide"), (4096, 3072, 1536, 1, "128x128"), (4096, 3008, 1600, 1, "wide"),
    (4096, 2816, 1600, 1, "128x128"), (8192, 128, 4096, 1, "128x128 of 4")])
def test_tiles(M, N, K, splits, want):
    assert form(M, N, K, splits) == want


# grouped rows in tiles of 256: the wide form from a K of 1600 on
@pytest.mark.parametrize("N,K,want", [(1024, 1600, "wide"), (1024, 4096, "wide"), (1536, 512, "256x256"), (1536, 1536, "256x256")])
def test_grouped(N, K, want):
    assert form(5000, N, K, 1, 27) == want


# tiles one after the other in a workgroup: all whole rounds; with side columns all tiles without them where the whole rounds reach into
# theirs, as many as an eighth; not a single round, a width or a K that it does not take
@pytest.mark.parametrize("M,N,K,side,want", [
    (7700, 14848, 2048, 0, 1792), (8192, 8192, 8192, 0, 1024), (7700, 17424, 2048, 16, 2048), (7700, 14624, 2048, 32, 31 * 57),
    (8192, 17424, 2048, 16, 32 * 68), (4096, 8192, 2048, 1024, 16 * 28), (4096, 8192, 2048, 1032, 0), (7700, 2048, 4096, 0, 0),
    (4096, 4104, 2048, 8, 0), (4352, 4104, 2048, 8, 0), (6400, 4104, 2048, 8, 25 * 16), (7700, 14624, 64, 32, 0), (7700, 14624, 128, 32, 31 * 57), (7700, 14628, 2048, 0, 0)])
def test_chained_tiles(M, N, K, side, want):
    assert native.lm_ops().lm_gemm_chained(M, N, K, side) == want
