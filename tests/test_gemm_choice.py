"""Which kernel serves a 16-bit product (csrc/kernels/gemm.cpp; no GPU: the rule is asked, for the 256 compute units it
assumes without one), on either side of each of its lines.  The times behind the lines stand at libraryAhead."""
import ctypes

import pytest

from test_index_bounds import internal

LIBRARY, MFMA, KSPLIT, F32_SMALL, WIDE, ROUND = range(6)
NONE, RELU, GELU = range(3)


@pytest.mark.parametrize("M,N,K,act,kernel", [
    (2048, 2048, 6144, NONE, MFMA),      # one round of tiles, however deep
    (2000, 2000, 4096, RELU, MFMA),
    (2304, 2048, 2048, NONE, MFMA),      # 288 tiles
    (2304, 2048, 2560, NONE, LIBRARY),
    (3072, 2048, 1536, RELU, MFMA),      # 384 tiles
    (3072, 2048, 2048, NONE, LIBRARY),
    (3000, 2048, 2048, RELU, LIBRARY),   # the same, ragged
    (2500, 2304, 768, NONE, MFMA),
    (5250, 1024, 4096, NONE, MFMA),      # 336 tiles, M at least twice N
    (5250, 1024, 4192, RELU, LIBRARY),
    (2047, 1024, 1536, NONE, MFMA),
    (4096, 2048, 1024, NONE, MFMA),      # 512 whole tiles
    (4096, 2048, 1056, NONE, LIBRARY),
    (4000, 2048, 768, NONE, LIBRARY),    # 512 tiles that overhang
    (3000, 2048, 3072, GELU, MFMA),      # a GELU to fuse
    (3000, 2048, 4096, GELU, LIBRARY),
    (4096, 3072, 1536, GELU, MFMA),
    (5000, 3072, 1536, GELU, LIBRARY),
    (32, 20000, 512, NONE, MFMA),        # few rows
    (32, 20000, 1024, NONE, LIBRARY),
    (8, 16384, 1024, NONE, KSPLIT),
    (77, 2304, 768, NONE, KSPLIT),
    (1024, 1024, 2048, NONE, KSPLIT),
])
def test_kernel_of_a_product(pkg, M, N, K, act, kernel):
    served = internal(pkg, "_ZN4mgpu13gemmKernelForENS_5DTypeElllbibb", ctypes.c_int, ctypes.c_int, *[ctypes.c_int64] * 3,
                      ctypes.c_bool, ctypes.c_int, ctypes.c_bool, ctypes.c_bool)
    for dtype in (1, 2):
        assert served(dtype, M, N, K, True, act, False, False) == kernel


@pytest.mark.parametrize("M,N,K,act,wanted", [
    (3072, 2048, 2048, RELU, True),    # a decoding layer of 3072 tokens at d_model 2048
    (3072, 6144, 2048, NONE, True),
    (2304, 2048, 2048, NONE, True),    # although the [K, N] weight would be gemm_mfma's
    (2304, 2048, 768, NONE, False),
    (2048, 2048, 2048, NONE, False),   # one round
    (3072, 2048, 2048, GELU, False),
    (4096, 2304, 768, NONE, False),    # a row of the table
    (240, 768, 768, NONE, False),
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
    (128, 40000, 256, GELU, WIDE),
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
