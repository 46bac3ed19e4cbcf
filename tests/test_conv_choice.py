"""Where a convolution's filter goes through LDS (csrc/kernels/conv.hip; no GPU: the rule is asked).  The times behind the lines
stand at convStagedWaves."""
import ctypes

import pytest

from test_index_bounds import internal


@pytest.mark.parametrize("win,tiles,IC,OC,waves", [
    (3, 256, 64, 32, 8),     # a round of the CUs, rows of the filter of whole lines
    (3, 256, 72, 32, 0),
    (3, 256, 32, 32, 0),
    (3, 230, 128, 16, 0),    # half of a tile's channels at most
    (3, 230, 256, 16, 8),
    (3, 450, 32, 24, 4),
    (3, 450, 48, 32, 0),
    (3, 450, 96, 32, 8),
    (3, 450, 144, 32, 8),
    (3, 450, 40, 64, 4),     # instead of 64 x 64 tiles
    (3, 450, 72, 64, 8),
    (3, 384, 40, 64, 0),
    (3, 512, 96, 16, 0),
    (3, 512, 192, 16, 8),
    (3, 750, 40, 32, 4),     # three tiles a CU
    (3, 750, 40, 16, 0),
    (3, 750, 64, 16, 4),
    (3, 769, 40, 32, 0),
    (3, 1500, 64, 32, 4),
    (3, 1500, 64, 16, 0),
    (3, 1500, 64, 64, 0),
    (3, 2049, 64, 32, 0),
    (3, 450, 33, 32, 0),
    (5, 230, 32, 32, 8),
    (5, 230, 40, 32, 0),
    (5, 230, 48, 32, 8),
    (5, 230, 48, 16, 0),
    (5, 330, 16, 32, 4),
    (5, 330, 24, 16, 0),
    (5, 750, 24, 16, 4),
    (5, 1020, 32, 32, 4),
    (5, 1020, 40, 32, 0),
    (5, 1200, 24, 32, 4),
    (5, 1500, 24, 32, 0),
    (5, 10125, 32, 32, 4),
    (7, 230, 18, 32, 8),
    (7, 230, 18, 16, 0),
    (7, 750, 32, 16, 4),
    (7, 1020, 32, 16, 0),
    (7, 1020, 18, 32, 4),
    (7, 1020, 18, 64, 0),
])
def test_wavefronts_a_tile(pkg, win, tiles, IC, OC, waves):
    ask = internal(pkg, "_ZN4mgpu15convStagedWavesEillll", ctypes.c_int, ctypes.c_int, *[ctypes.c_int64] * 4)
    assert ask(win, tiles, IC, OC, 256) == waves


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
