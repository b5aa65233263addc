"""The counts of parts of K that the tuner tries (csrc/kernels/gemm_lds.hip): by a rule on sizes, the same for every image and batch."""
import json
import os
import re

import pytest

from shai_amd import native

if not os.path.exists(native.KERNELS_LIB):
    pytest.skip("the native library is not built", allow_module_level=True)

# tile rows and columns of some configs
TILES = {1: (256, 256), 3: (128, 128), 4: (128, 64), 9: (256, 256), 10: (256, 320), 16: (64, 64), 17: (128, 64), 18: (128, 128), 21: (192, 128)}


def counts(M, N, K, cfg):
    return native.ops().gemm_split_counts(M, N, K, cfg)


@pytest.mark.parametrize("cfg", sorted(TILES))
@pytest.mark.parametrize("M,N,K", [(126, 1280, 11520), (120, 1280, 23040), (2048, 640, 17280), (504, 640, 5760), (8064, 4, 2880), (77, 320, 520),
                                   (2, 8, 64), (18432, 320, 8640), (110, 4096, 4096)])
def test_counts_fill_rounds(M, N, K, cfg):
    """From each of four ranges the count whose last round is the fullest, no more of them than powers of two, no part empty or short."""
    bm, bn = TILES[cfg]
    tiles, kt = -(-M // bm) * -(-N // bn), -(-K // 64)
    fill = lambda s: tiles * s / (-(-tiles * s // 256) * 256)
    got, want = counts(M, N, K, cfg), [1]
    for lo, hi, power in ((2, 3, 2), (4, 6, 4), (7, 12, 8), (13, 16, 16)):
        fit = [s for s in range(lo, hi + 1) if kt // s >= 4 and -(-kt // -(-kt // s)) == s]
        if fit and kt // power >= 4:
            want.append(max(fit, key=lambda s: (round(fill(s), 9), -s)))
    assert got == want and len(got) <= 5


def test_a_part_for_every_cu():
    """Workgroups that share a CU do not hide counts that give every CU one."""
    assert 2 in counts(110, 4096, 4096, 16) and 4 in counts(110, 4096, 4096, 17)


def test_unsplit_tiles():
    for cfg in (13, 14, 15):
        assert counts(512, 1280, 11520, cfg) == [1]


def test_shipped_choices_are_the_tuners():
    """A shipped choice with another count than a power of two is one that the tuner tries, for its size as for any other."""
    path = os.path.join(os.path.dirname(native.DEFAULT_TUNE_FILE), "gemm_tuning_mi355x.json")
    seen = 0
    for entry in json.load(open(path)):
        key, cfg, parts = re.match(r"(.*)=(\d+),(\d+)$", entry).groups()
        cfg, parts = int(cfg), int(parts)
        if cfg < 1000 and parts & (parts - 1):
            M, N, K = (int(v) for v in re.match(r"\d:(\d+),(\d+),(\d+),", key).groups())
            assert parts in counts(M, N, K, cfg), entry
            seen += 1
    assert seen
