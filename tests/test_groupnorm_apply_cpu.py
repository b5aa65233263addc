"""How many vectors a thread of GroupNorm's apply pass has: by size alone, so that images of neighbouring sizes are made alike."""
import os

import pytest

from shai_amd import native

if not os.path.exists(native.KERNELS_LIB):
    pytest.skip("the native library is not built", allow_module_level=True)


def each(N, HW, C):
    """Vectors of 8 channels a thread, rounded."""
    return round(N * HW * C / 8 / 256 / native.ops().groupnorm_apply_blocks(N, HW, C))


@pytest.mark.parametrize("N,HW,C,want", [
    (1, 4096, 320, 1), (2, 4096, 384, 1), (1, 16383, 256, 1), (1, 16384, 256, 2), (1, 24575, 256, 2), (1, 24576, 256, 3), (2, 147456, 256, 3),
    (3, 4096, 960, 2), (3, 1024, 1280, 1), (4, 65536, 256, 2), (5, 65536, 256, 1), (16, 4096, 640, 1)])
def test_by_size_and_images(N, HW, C, want):
    assert each(N, HW, C) == want


@pytest.mark.parametrize("C,sides", [(256, (512, 512, 448, 576)), (128, (1024, 1024, 1000, 1040)), (512, (256, 256, 224, 288)), (512, (128, 256, 136, 248))])
def test_sizes_with_odd_sides_alike(C, sides):
    """Images of 2^k pixels and of about as many."""
    h, w, h2, w2 = sides
    assert each(1, h * w // 4, C) == each(1, h2 * w2 // 4, C) == each(1, h * w // 4 + 1, C)


@pytest.mark.parametrize("C", [8, 264, 320, 960, 1280])
def test_a_channel_vector_to_a_thread(C):
    """The grid's threads are a multiple of the vectors of a pixel."""
    for HW in (1, 77, 5000, 300000):
        assert native.ops().groupnorm_apply_blocks(1, HW, C) * 256 % (C // 8) == 0
