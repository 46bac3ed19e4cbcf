"""Which kernel serves a 16-bit product (csrc/kernels/gemm.cpp; no GPU: the rule is asked, for the 256 compute units it
assumes without one), on either side of each of its lines.  The times behind the lines stand at libraryAhead."""
import ctypes

import pytest

from test_index_bounds import internal

LIBRARY, MFMA, KSPLIT, F32_SMALL, WIDE, ROUND = range(6)
NONE, RELU, GELU = range(3)


@pytest.mark.parametrize("M,N,K,act,kernel", [
    (2048, 2048, 6144, NONE, ROUND),     # one round of tiles, however deep
    (2000, 2000, 4096, RELU, ROUND),
    (2000, 2000, 4104, NONE, ROUND),     # filled up to a multiple of 64
    (2000, 2000, 4100, NONE, LIBRARY),   # rows off the 16-byte grid
    (512, 3072, 72, NONE, ROUND),
    (2304, 2048, 2560, NONE, WIDE),      # beyond one round
    (4000, 2048, 768, RELU, WIDE),
    (5250, 1024, 4192, NONE, WIDE),
    (3000, 2048, 4096, GELU, WIDE),
    (3200, 2048, 64, NONE, MFMA),        # 400 tiles, too shallow for gemm_wide
    (3200, 2056, 64, NONE, LIBRARY),     # 425 that overhang
    (3968, 2048, 64, NONE, MFMA),        # 496 whole ones
    (4096, 3072, 64, GELU, MFMA),
    (19200, 19200, 64, GELU, LIBRARY),
    (32, 20000, 512, NONE, ROUND),       # few rows
    (32, 20000, 1024, NONE, LIBRARY),
    (100, 40000, 256, NONE, WIDE),
    (127, 40000, 1024, GELU, MFMA),
    (127, 600000, 512, GELU, LIBRARY),
    (8, 16384, 1024, NONE, KSPLIT),
    (77, 2304, 768, NONE, KSPLIT),
    (768, 1152, 32, NONE, MFMA),         # 54 tiles of 32 deep
    (768, 1152, 32, GELU, KSPLIT),
    (256, 1152, 32, NONE, KSPLIT),
    (768, 1152, 64, NONE, KSPLIT),
    (26, 18248, 32, NONE, MFMA),         # two rounds of gemm_ksplit's
    (1, 23560, 96, NONE, MFMA),
    (83, 6128, 96, NONE, KSPLIT),        # one
    (2209, 488, 96, NONE, MFMA),         # shallow
    (5504, 3552, 96, RELU, MFMA),
    (500, 2000, 1000, NONE, KSPLIT),
    (1024, 1024, 2048, NONE, KSPLIT),
])
def test_kernel_of_a_product(pkg, M, N, K, act, kernel):
    served = internal(pkg, "_ZN4mgpu13gemmKernelForENS_5DTypeElllbibb", ctypes.c_int, ctypes.c_int, *[ctypes.c_int64] * 3,
                      ctypes.c_bool, ctypes.c_int, ctypes.c_bool, ctypes.c_bool)
    for dtype in (1, 2):
        assert served(dtype, M, N, K, True, act, False, False) == kernel


@pytest.mark.parametrize("M,N,K,act,wanted", [
    (3072, 2048, 2048, RELU, False),   # gemm_wide's
    (2304, 2048, 768, NONE, False),
    (2048, 2048, 2048, NONE, False),   # gemm_round's
    (512, 3000, 1000, NONE, False),    # ... of a depth that it fills up
    (240, 768, 768, NONE, False),      # gemm_ksplit's
    (240, 770, 768, NONE, True),       # the library's
    (240, 770, 256, GELU, True),
    (32, 20000, 1024, NONE, True),     # few rows: the library's either way
    (64, 20000, 512, GELU, False),
])
def test_layout_of_a_weight_that_is_cast_per_call(pkg, M, N, K, act, wanted):
    wants = internal(pkg, "_ZN4mgpu19gemmWantsKMajorCastENS_5DTypeElllbib", ctypes.c_bool, ctypes.c_int, *[ctypes.c_int64] * 3,
                     ctypes.c_bool, ctypes.c_int, ctypes.c_bool)
    assert wants(1, M, N, K, True, act, False) is wanted


@pytest.mark.parametrize("M,N,K,act,kernel", [
    (64, 40000, 128, NONE, MFMA),   # tiles of 256 rows three quarters empty
    (65, 40000, 128, NONE, WIDE),
    (100, 40000, 96, NONE, MFMA),
    (127, 40000, 256, GELU, MFMA),
    (128, 40000, 256, GELU, MFMA),  # shallow: 12.4 us on gemm_wide, 11.0 here
    (128, 40000, 512, GELU, WIDE),
    (1395, 648, 32, RELU, MFMA),    # one round, shallow, no whole lines
    (2209, 488, 96, NONE, MFMA),
    (2209, 488, 128, NONE, ROUND),
    (300, 3000, 160, NONE, MFMA),
    (300, 3000, 224, NONE, ROUND),
    (2304, 576, 96, NONE, MFMA),    # whole lines
    (2304, 576, 64, NONE, ROUND),
    (2304, 576, 160, NONE, ROUND),
    (5504, 3552, 96, NONE, MFMA),   # more rounds: by the estimates
    (5504, 3552, 128, NONE, WIDE),
    (14080, 2888, 96, GELU, MFMA),
    (14080, 2888, 128, NONE, WIDE),
    (5504, 3552, 320, GELU, WIDE),  # beyond 256 deep
    (128, 40000, 64, GELU, MFMA),   # too shallow for gemm_wide
    (127, 32768, 256, GELU, ROUND),
    (4096, 768, 768, NONE, ROUND),
    (2000, 1024, 512, NONE, ROUND),
])
def test_kernel_behind_gemm_mfma(pkg, M, N, K, act, kernel):
    """gemm_mfma's launcher hands products to gemm_round and gemm_wide; not those whose rows would leave their tiles empty."""
    ask = internal(pkg, "_ZN4mgpu14gemmMfmaKernelENS_5DTypeEPKvS2_S2_S2_S2_llliPi", ctypes.c_int, ctypes.c_int, *[ctypes.c_void_p] * 5,
                   *[ctypes.c_int64] * 3, ctypes.c_int, ctypes.POINTER(ctypes.c_int))
    got = ctypes.c_int()
    for dtype in (1, 2):
        assert ask(dtype, 4096, 4096, 4096, None, 4096, M, N, K, act, got) == kernel
        assert got.value in ((128, 192, 256) if kernel == WIDE else (96, 128))


@pytest.mark.parametrize("M,N,K,act,prefers", [
    (2000, 768, 3072, NONE, False),   # up to one round of tiles, ragged: gemm_round
    (1368, 768, 3072, NONE, False),   # ... split over blocks
    (774, 3072, 768, GELU, False),
    (4096, 768, 3072, NONE, False),
    (77, 768, 768, NONE, False),      # gemm_ksplit
    (4096, 6144, 2048, NONE, False),  # gemm_wide
    (774, 770, 768, NONE, True),      # no multiple of 8: the library
    (774, 768, 3070, GELU, True),
    (32, 20000, 1024, RELU, True),
])
def test_layout_of_a_weight_that_is_kept(pkg, M, N, K, act, prefers):
    """K-major exactly where the [K, N] weight would be the library's, be it for where it lies."""
    ask = internal(pkg, "_ZN4mgpu17gemmPrefersKMajorENS_5DTypeEPKvS2_lllbib", ctypes.c_bool, ctypes.c_int, *[ctypes.c_void_p] * 2,
                   *[ctypes.c_int64] * 3, ctypes.c_bool, ctypes.c_int, ctypes.c_bool)
    served = internal(pkg, "_ZN4mgpu13gemmKernelForENS_5DTypeElllbibb", ctypes.c_int, ctypes.c_int, *[ctypes.c_int64] * 3,
                      ctypes.c_bool, ctypes.c_int, ctypes.c_bool, ctypes.c_bool)
    assert ask(1, 4096, 4096, M, N, K, True, act, False) is prefers
    assert (served(1, M, N, K, True, act, False, False) == LIBRARY) is prefers
    assert ask(1, 4098, 4096, M, N, K, True, act, False) and ask(1, 4096, 4098, M, N, K, True, act, False)
