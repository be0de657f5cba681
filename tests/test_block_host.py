"""What the launch of a residual block reads of LDS, without a GPU."""
import ctypes

import pytest

from mxnet_amd import _lib


def lds(*shape):
    have, reach = ctypes.c_int(), ctypes.c_int()
    _lib.check(_lib.lib.mxq_test_block_lds(*shape, ctypes.byref(have), ctypes.byref(reach)))
    return have.value, reach.value


# one piece a row and many; the channels that a kernel instance is made for, and others; planes in
# rectangles, as runs and of several images a tile
@pytest.mark.parametrize("tile", [32, 64])
@pytest.mark.parametrize("n, h, w", [(1, 1, 1), (3, 4, 4), (2, 7, 7), (64, 14, 14), (5, 6, 11),
                                     (64, 28, 28), (64, 56, 56), (1, 2, 500)])
def test_block_reads_only_the_lds_it_has(n, h, w, tile):
    some = 0
    for c in (16, 32, 64, 96, 128, 256, 272):
        for mid in (16, 48, 64, 80, 128, 144, 256):
            for out in (16, 32, 48, 112, 256, 512, 1024):
                for after in (0, 16, 48, 64, 256):
                    have, reach = lds(n, h, w, c, mid, out, after, tile)
                    assert reach <= have, (c, mid, out, after)
                    some += have > 0
    assert some > 100


# within 608 bytes of what a tile of 64 pixels may have: of all LDS, and of half of it
@pytest.mark.parametrize("shape, most", [
    ((64, 7, 7, 128, 256, 2048, 256), 160 * 1024), ((64, 15, 15, 96, 192, 2048, 0), 160 * 1024),
    ((64, 10, 10, 1232, 112, 768, 0), 160 * 1024), ((64, 4, 4, 704, 256, 512, 256), 160 * 1024),
    ((64, 11, 11, 528, 112, 512, 0), 80 * 1024), ((64, 17, 17, 320, 128, 256, 0), 160 * 1024 // 3)])
def test_block_tables_take_no_more_lds_than_a_word_a_pixel(shape, most):
    have, reach = lds(*shape, 64)
    assert 0 < have <= most and reach <= have
