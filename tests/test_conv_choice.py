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
