"""The epilogues that widen a layer's fp16 result to fp32, and the one launch that casts a layer's weights beside its input's
LayerNorm, against the separate kernels."""
import ctypes

import pytest
import torch

from conftest import to_dev
from test_gemm_choice import KSPLIT, NONE, ROUND
from test_index_bounds import internal

pytestmark = pytest.mark.gpu
STREAM = ctypes.c_void_p


def ptr(t):
    return ctypes.c_void_p(t.data_ptr())


@pytest.mark.parametrize("M,N,K,kernel", [
    (1, 8, 8, KSPLIT), (33, 40, 72, KSPLIT),     # 32 x 32 tiles that overhang either way
    (186, 768, 768, KSPLIT), (300, 1032, 264, KSPLIT),
    (1194, 512, 1024, KSPLIT), (2001, 968, 448, ROUND),  # last rows and columns of a tile
    (2001, 968, 520, ROUND), (4096, 768, 3080, ROUND),   # a depth filled up to 64
])
def test_product_with_a_residual_in_fp32(pkg, gpu, M, N, K, kernel):
    pkg.ops()
    run = internal(pkg, "_ZN4mgpu17matmulResidualF32EPKvS1_S1_S1_PflllbP12ihipStream_t", ctypes.c_bool, *[ctypes.c_void_p] * 5,
                   *[ctypes.c_int64] * 3, ctypes.c_bool, STREAM)
    served = internal(pkg, "_ZN4mgpu13gemmKernelForENS_5DTypeElllbibb", ctypes.c_int, ctypes.c_int, *[ctypes.c_int64] * 3,
                      ctypes.c_bool, ctypes.c_int, ctypes.c_bool, ctypes.c_bool)
    assert served(1, M, N, K, True, NONE, True, False) == kernel
    gen = torch.Generator(device=gpu).manual_seed(M)
    x, w, b, r = (torch.randn(s, device=gpu, generator=gen).half() for s in ((M, K), (K, N), (N,), (M, N)))
    w *= K ** -0.5
    out = torch.full((M * N + 256,), float("nan"), device=gpu)
    stream = STREAM(torch.cuda.current_stream().cuda_stream)
    assert run(ptr(x), ptr(w), ptr(b), ptr(r), ptr(out), M, N, K, False, stream)
    assert torch.equal(out[:M * N].view(M, N), pkg.matmul_ex(x, w, b, r).float())
    assert out[M * N:].isnan().all()
    assert not run(ptr(x), ptr(w), None, ptr(r), ptr(out), M, N, K, False, stream)


@pytest.mark.parametrize("m,n", [(1, 8), (3, 520), (186, 768), (257, 1000), (1000, 2048), (65, 4096)])
def test_layer_norm_in_fp32(pkg, gpu, m, n):
    pkg.ops()
    run = internal(pkg, "_ZN4mgpu17layerNormF16ToF32EPKvS1_S1_S1_PffiiP12ihipStream_t", ctypes.c_bool, *[ctypes.c_void_p] * 5,
                   ctypes.c_float, ctypes.c_int, ctypes.c_int, STREAM)
    gen = torch.Generator(device=gpu).manual_seed(n)
    x, r, g, b = (torch.randn(s, device=gpu, generator=gen).half() for s in ((m, n), (m, n), (n,), (n,)))
    out = torch.full((m * n + 256,), float("nan"), device=gpu)
    stream = STREAM(torch.cuda.current_stream().cuda_stream)
    assert run(ptr(x), ptr(r), ptr(g), ptr(b), ptr(out), 1e-5, m, n, stream)
    _, want = pkg.add_residual_layer_norm(x, r, g, b)
    got = out[:m * n].view(m, n)
    assert torch.equal(got, got.half().float())
    # (the compiler rounds the last multiply-add and the fp16 value at once in one kernel and one after another in the other: ties apart)
    assert (got - want.float()).abs().le(want.float().abs() * 2.0 ** -10 + 2.0 ** -24).all() and got.ne(want.float()).double().mean() <= 1e-3
    assert out[m * n:].isnan().all()
    assert not run(ptr(x), ptr(r), ptr(g), ptr(b), ptr(out), 1e-5, m, 4104, stream)


@pytest.mark.parametrize("M,d,ffn,shift", [(5, 72, 40, 0), (77, 768, 3072, 0), (77, 768, 3072, 1), (9, 4104, 64, 0)])
def test_casts_beside_the_layer_norm(pkg, gpu, M, d, ffn, shift):
    """Weights whose sizes are no whole blocks, off the 16-byte grid, and a width that takes the LayerNorm for itself: a layer of
    ones and zeros in its weights, of which the result is known."""
    gen = torch.Generator(device=gpu).manual_seed(d)
    x = torch.randn((1, M, d), device=gpu, generator=gen)

    def place(t):
        flat = torch.zeros(t.numel() + shift, device=gpu)
        flat[shift:] = t.reshape(-1)
        return flat[shift:].view(t.shape)

    eye = torch.zeros((d, 3 * d), device=gpu)
    eye[:, 2 * d:] = torch.eye(d, device=gpu)  # V = LN(x), Q = K = 0: the context is the mean of LN(x) over the sequence
    up, down = torch.randn((d, ffn), device=gpu, generator=gen) / 32, torch.randn((ffn, d), device=gpu, generator=gen) / 32
    bias = [torch.randn(n, device=gpu, generator=gen) for n in (d, ffn, d)]
    got = pkg.decoding_context_layer(x, *map(place, (eye, torch.eye(d, device=gpu), bias[0], up, bias[1], down, bias[2])), heads=d // 24, causal=False)
    h = lambda t: t.half().double()  # noqa: E731
    ln = lambda t: torch.nn.functional.layer_norm(t, (d,), eps=1e-5)  # noqa: E731
    y = h(x) + ln(h(x)).mean(1, keepdim=True) + h(bias[0])
    want = y + torch.relu(ln(y) @ h(up) + h(bias[1])) @ h(down) + h(bias[2])
    # (a handful of fp16 roundings of values up to 8, and of the weights' products)
    assert (got - want).norm() <= 2e-3 * want.norm()
