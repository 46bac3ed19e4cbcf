"""Where a convolution's filter goes through LDS (csrc/kernels/conv.hip; no GPU: the rule is asked).  The times behind the lines
stand at convStagedWaves."""
import ctypes

import pytest

from test_index_bounds import internal


@pytest.mark.parametrize("win,stride,tiles,IC,OC,OW,waves", [
    (3, 1, 256, 64, 32, 32, 8),
    (3, 1, 256, 72, 32, 32, 0),
    (3, 1, 256, 128, 32, 32, 8),
    (3, 1, 256, 62, 32, 32, 0),
    (3, 1, 230, 128, 16, 32, 8),
    (3, 1, 230, 256, 16, 32, 8),
    (3, 1, 230, 256, 8, 32, 0),
    (3, 2, 230, 80, 32, 4, 8),
    (3, 1, 230, 80, 32, 64, 0),
    (3, 1, 384, 40, 64, 64, 0),
    (3, 1, 450, 40, 64, 64, 4),
    (3, 1, 450, 72, 64, 64, 8),
    (3, 1, 512, 160, 32, 32, 8),
    (3, 1, 513, 160, 32, 32, 4),
    (3, 1, 750, 40, 32, 32, 4),
    (3, 1, 768, 40, 64, 32, 4),
    (3, 1, 770, 40, 64, 32, 0),
    (3, 1, 1500, 64, 32, 64, 4),
    (3, 1, 1500, 48, 32, 64, 0),
    (3, 1, 2048, 64, 32, 64, 4),
    (3, 1, 2049, 64, 32, 64, 0),
    (3, 1, 450, 129, 32, 32, 0),
    (5, 1, 256, 32, 32, 32, 8),
    (5, 1, 257, 32, 32, 32, 4),
    (5, 1, 256, 40, 32, 32, 8),
    (5, 2, 256, 40, 32, 8, 8),
    (5, 1, 256, 30, 32, 8, 0),
    (5, 1, 330, 16, 32, 32, 4),
    (5, 1, 330, 14, 32, 32, 0),
    (5, 2, 1020, 32, 32, 32, 4),
    (5, 1, 1020, 24, 32, 32, 0),
    (5, 2, 1220, 16, 32, 8, 4),
    (5, 1, 1200, 32, 64, 32, 0),
    (7, 1, 256, 16, 32, 32, 8),
    (7, 1, 257, 16, 32, 32, 4),
    (7, 1, 256, 14, 32, 32, 0),
    (7, 1, 256, 18, 8, 32, 0),
    (7, 1, 1020, 18, 32, 32, 4),
    (7, 1, 1020, 18, 64, 32, 0),
    (1, 1, 256, 256, 32, 32, 0),
])
def test_wavefronts_a_tile(pkg, win, stride, tiles, IC, OC, OW, waves):
    """On either side of the lines on tiles, channel groups, channels a tile, whole lines of the filter, stride and short rows."""
    ask = internal(pkg, "_ZN4mgpu15convStagedWavesEillllll", ctypes.c_int, ctypes.c_int, *[ctypes.c_int64] * 6)
    assert ask(win, stride, tiles // -(-OC // 32) * 32, IC, OC, OW, 256) == waves


@pytest.mark.parametrize("win,stride,tiles,rowTiles,IC,OC,OW,patches", [
    (5, 1, 1, 1, 1, 8, 16, True),         # from one channel, if half of a row's tiles are filled
    (5, 1, 1, 1, 1, 8, 15, False),
    (7, 2, 1, 2, 1, 8, 33, True),
    (7, 1, 1, 1, 3, 8, 32, True),
    (5, 1, 256, 300, 3, 64, 28, False),   # few tiles
    (5, 1, 257, 300, 3, 64, 28, True),
    (5, 2, 400, 500, 3, 96, 28, False),
    (5, 2, 401, 500, 3, 96, 28, True),
    (7, 2, 256, 300, 3, 96, 28, True),
    (7, 1, 1024, 1025, 3, 96, 28, False), # another round of the SIMDs
    (7, 1, 1025, 1026, 3, 96, 28, True),
    (7, 1, 1024, 1025, 3, 64, 28, True),  # instead of 64 x 64 tiles
    (5, 1, 2048, 3072, 3, 96, 28, True),  # three for two
    (5, 2, 2048, 3072, 3, 96, 28, False),
    (7, 3, 9000, 9000, 3, 96, 64, False),
    (3, 1, 9000, 9000, 3, 96, 64, False),
    (7, 1, 9000, 9000, 2, 96, 64, False),
])
def test_patches_of_input_rows(pkg, win, stride, tiles, rowTiles, IC, OC, OW, patches):
    ask = internal(pkg, "_ZN4mgpu13convByPatchesEiillllll", ctypes.c_bool, ctypes.c_int, ctypes.c_int, *[ctypes.c_int64] * 6)
    assert ask(win, stride, tiles, rowTiles, IC, OC, OW, 256) is patches
