"""gemm_wide and gemm_round (csrc/kernels): every tile width, where tiles end inside the shape and where they fit, from the
fewest reduction steps on, each epilogue, both types; nothing stored outside the output."""
import ctypes

import pytest

from test_index_bounds import internal

SHAPES = [
    (1, 8, 128),       # one row, one chunk of columns; gemm_wide: no pass of the loop
    (256, 768, 192),   # whole tiles of every width; gemm_wide: one pass
    (257, 520, 256),   # gemm_round: as many steps as are kept ahead
    (300, 1000, 320),
    (511, 248, 1088),
    (2300, 136, 704),  # more tile rows than a group
]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("name,width,M,N,K", [("8gemmWide", w, *s) for w in (128, 192, 256) for s in SHAPES] +
                         [("9gemmRound", w, *s) for w in (96, 128) for s in SHAPES + [(130, 104, 64)]])
def test_against_float64(pkg, gpu, dtype, name, width, M, N, K):
    import torch
    t, code, ulp = (torch.float16, 1, 2.0**-11) if dtype == "f16" else (torch.bfloat16, 2, 2.0**-8)
    g = torch.Generator(device=gpu).manual_seed(M + N + K)
    r = lambda *s: torch.randn(s, generator=g, device=gpu)
    x, w, b, res = r(M, K).to(t), (r(K, N) / K**0.5).to(t), r(N).to(t), r(M, N).to(t)
    gemm = internal(pkg, "_ZN4mgpu" + name + "ENS_5DTypeEPKvS2_S2_S2_PvllliiP12ihipStream_t", None, ctypes.c_int, *[ctypes.c_void_p] * 5, *[ctypes.c_int64] * 3, ctypes.c_int, ctypes.c_int, ctypes.c_void_p)
    X, W = x.double().cpu(), w.double().cpu()
    prod, size = X @ W, X.abs() @ W.abs()
    B, R = b.double().cpu(), res.double().cpu()
    for bias, act, residual in ((None, 0, None), (b, 1, None), (b, 2, None), (b, 0, res)):
        out = torch.full((M + 2, N), 7.0, dtype=t, device=gpu)  # a row before and one behind
        gemm(code, x.data_ptr(), w.data_ptr(), bias.data_ptr() if bias is not None else None, residual.data_ptr() if residual is not None else None,
             out[1:].data_ptr(), M, N, K, act, width, torch.cuda.current_stream().cuda_stream)
        got = out.double().cpu()
        ref = prod + (B if bias is not None else 0)
        ref = ref.relu() if act == 1 else 0.5 * ref * torch.erfc(-ref / 2**0.5) if act == 2 else ref
        ref = ref + R if residual is not None else ref
        # one rounding of the result (and the smallest number), K + 2 fp32 roundings of partial sums no larger than |x||w| + |b|,
        # through a GELU whose slope stays below 1.13 and whose own error is below 3e-6
        bound = 1.05 * ulp * ref.abs() + 2.0**-25 + 1.13 * (K + 2) * 2.0**-24 * (size + B.abs()) + 3e-6 * ref.abs()
        assert ((got[1:-1] - ref).abs() <= bound).all(), (act, ((got[1:-1] - ref).abs() / bound).max())
        assert (got[0] == 7).all() and (got[-1] == 7).all()


RAGGED = [
    (3, 8, 72),        # the shortest of gemm_wide: a chunk of the second buffer, no pass of the loop
    (256, 384, 136),
    (257, 520, 184),   # the last slice of 32 all filler, and one chunk short of whole
    (300, 1000, 232),
    (513, 248, 1096),
    (2300, 136, 680),
]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("name,width,M,N,K", [("8gemmWide", w, *s) for w in (128, 192, 256) for s in RAGGED] +
                         [("9gemmRound", w, *s) for w in (96, 128) for s in RAGGED + [(130, 104, 8), (129, 200, 56), (64, 96, 296)]])
def test_depths_that_are_no_multiple_of_64(pkg, gpu, dtype, name, width, M, N, K):
    """As above; and what lies behind the end of a row or of the weight has no part in the result, whatever it is."""
    import torch
    test_against_float64(pkg, gpu, dtype, name, width, M, N, K)
    t, code = (torch.float16, 1) if dtype == "f16" else (torch.bfloat16, 2)
    x, w = torch.full((M + 1, K), float("inf"), dtype=t, device=gpu), torch.full((K + 64, N), float("nan"), dtype=t, device=gpu)
    x[0:M:2], w[:K] = 1.0, 2.0**-4  # every other row is infinite
    out = torch.zeros((M, N), dtype=t, device=gpu)
    gemm = internal(pkg, "_ZN4mgpu" + name + "ENS_5DTypeEPKvS2_S2_S2_PvllliiP12ihipStream_t", None, ctypes.c_int, *[ctypes.c_void_p] * 5,
                    *[ctypes.c_int64] * 3, ctypes.c_int, ctypes.c_int, ctypes.c_void_p)
    gemm(code, x.data_ptr(), w.data_ptr(), None, None, out.data_ptr(), M, N, K, 0, width, torch.cuda.current_stream().cuda_stream)
    assert (out[0::2].float() == torch.tensor(K / 16).to(t).float().item()).all() and (out[1::2] == float("inf")).all()


@pytest.mark.gpu
@pytest.mark.parametrize("width", [128, 192, 256])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_fp32_result_against_float64(pkg, gpu, width, M, N, K):
    import torch
    g = torch.Generator(device=gpu).manual_seed(M + N + K)
    r = lambda *s: torch.randn(s, generator=g, device=gpu)
    x, w, b, res = r(M, K).half(), (r(K, N) / K**0.5).half(), r(N).half(), r(M, N).half()
    gemm = internal(pkg, "_ZN4mgpu19gemmWideResidualF32EPKvS1_S1_S1_PfllliP12ihipStream_t", None, *[ctypes.c_void_p] * 5,
                    *[ctypes.c_int64] * 3, ctypes.c_int, ctypes.c_void_p)
    out = torch.full((M + 2, N), 7.0, device=gpu)  # a row before and one behind
    gemm(x.data_ptr(), w.data_ptr(), b.data_ptr(), res.data_ptr(), out[1:].data_ptr(), M, N, K, width, torch.cuda.current_stream().cuda_stream)
    got, X, W, B, R = [t.double().cpu() for t in (out, x, w, b, res)]
    # K + 2 fp32 roundings of partial sums no larger than |x||w| + |b| + |residual|
    bound = (K + 2) * 2.0**-24 * (X.abs() @ W.abs() + B.abs() + R.abs())
    assert ((got[1:-1] - (X @ W + B + R)).abs() <= bound).all()
    assert (got[0] == 7).all() and (got[-1] == 7).all()


@pytest.mark.gpu
@pytest.mark.parametrize("width,M,N,K,parts", [(96, 300, 200, 512, 2), (128, 131, 264, 1088, 4), (96, 128, 96, 832, 3)])
def test_planes_of_partial_sums(pkg, gpu, width, M, N, K, parts):
    """Shares of unequal length; the planes add up to the product."""
    import torch
    g = torch.Generator(device=gpu).manual_seed(K)
    x, w = torch.randn((M, K), generator=g, device=gpu).half(), torch.randn((K, N), generator=g, device=gpu).half()
    gemm = internal(pkg, "_ZN4mgpu19gemmRoundPartialF16EPKvS1_PfllliiP12ihipStream_t", None, *[ctypes.c_void_p] * 3, *[ctypes.c_int64] * 3,
                    ctypes.c_int, ctypes.c_int, ctypes.c_void_p)
    planes = torch.full((parts + 1, M, N), 7.0, device=gpu)
    gemm(x.data_ptr(), w.data_ptr(), planes.data_ptr(), M, N, K, width, parts, torch.cuda.current_stream().cuda_stream)
    X, W = x.double().cpu(), w.double().cpu()
    got = planes[:parts].double().cpu().sum(0)
    assert ((got - X @ W).abs() <= (K + parts) * 2.0**-24 * (X.abs() @ W.abs())).all()
    assert (planes[parts] == 7).all()


@pytest.mark.parametrize("M,N,K,act,residual,width", [
    (4096, 3072, 768, 2, False, 192),    # a round of tiles of 192
    (4096, 6144, 2048, 0, False, 192),
    (8192, 8192, 8192, 0, False, 256),
    (4096, 2048, 2048, 0, True, 128),
    (2304, 2048, 2560, 0, False, 128),   # beyond one round of 128 x 128 tiles, however deep
    (2049, 2048, 128, 0, False, None),   # (whatever the width)
    (4096, 2048, 72, 0, False, None),    # filled up to the fewest steps its loop is built for
    (4096, 2048, 64, 0, False, 0),
    (4096, 2048, 1048, 0, False, None),
    (4096, 2048, 1052, 0, False, 0),     # rows off the 16-byte grid
    (4096, 2044, 1024, 0, False, 0),
    (127, 40000, 1024, 0, False, 0),
    (4096, 768, 3072, 0, False, 0),      # up to one round of 128 x 128 tiles
    (77, 768, 768, 0, False, 0),
])
def test_what_it_serves(pkg, M, N, K, act, residual, width):
    served = internal(pkg, "_ZN4mgpu13gemmWideWidthENS_5DTypeElllib", ctypes.c_int, ctypes.c_int, *[ctypes.c_int64] * 3, ctypes.c_int, ctypes.c_bool)
    for dtype in (1, 2):
        got = served(dtype, M, N, K, act, residual)
        assert got == width if width is not None else got in (128, 192, 256)
    assert served(0, M, N, K, act, residual) == 0  # fp32


def test_tiles_stay_inside_a_grid_and_rows_inside_an_int(pkg):
    supports = internal(pkg, "_ZN4mgpu16gemmWideSupportsENS_5DTypeEPKvS2_S2_S2_S2_lll", ctypes.c_bool, ctypes.c_int,
                        *[ctypes.c_void_p] * 5, *[ctypes.c_int64] * 3)

    def ask(M, N, K, out=4096):
        return supports(1, 4096, 4096, 4096, None, out, M, N, K)

    assert ask(300, 104, 128) and not ask(300, 104, 128, out=4104)
    for N in (8, 128, 136, 1024, 2**20):
        for M in (2**24, 2**30, 2**31 - 256, 2**31 - 255, 2**31, 2**33 + 5):
            if ask(M, N, 128):
                assert -(-M // 256) * 256 < 2**31 and -(-M // 256) * -(-N // 128) * 512 < 2**32, (M, N)
    assert ask(2**31 - 256, 8, 128) and not ask(2**31 - 255, 8, 128)
