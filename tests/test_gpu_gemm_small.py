"""The kernels behind mgpuMatmulEx for few and for overhanging tiles - gemm_ksplit (both weight layouts), gemm_mfma with
tiles that overhang the shape, gemm_f32_small - against the oracle, at the edges of their tiles and of the reduction."""
import numpy as np
import pytest

from conftest import to_dev
from test_gpu_gemm_mfma import epilogues, spacing_tol

pytestmark = pytest.mark.gpu


# M, K, N: one row, one 8-k step, K = 8 / 16 / 24 mod 32, rows and columns past a tile by one vector, every tile of
# gemm_ksplit (32 x 32: 77 x 768 x 200; 32 x 64: 100 x 1024 x 1536; 64 x 64: 300 x 640 x 1544), gemm_mfma overhanging
# 128- and 96-column tiles, with steps of 64 and eight wavefronts, in pairs of 32, and of 32
SMALL = [(1, 8, 8), (1, 24, 40), (31, 40, 32), (33, 8 * 33, 72), (77, 768, 200), (5, 3072, 96), (64, 520, 64), (100, 1024, 1536),
         (300, 640, 1544), (300, 648, 1544), (129, 2048, 1032), (600, 1024, 3080), (1000, 768, 776), (2500, 128, 2312), (2500, 160, 2312),
         (700, 96, 808)]


@pytest.mark.parametrize("M,K,N", SMALL)
def test_matmul_ex_f16_any_shape(pkg, gpu, oracle, rng, M, K, N):
    x = rng.standard_normal((M, K)).astype(np.float16)
    w = (rng.standard_normal((K, N)) / np.sqrt(K)).astype(np.float16)
    b, r = rng.standard_normal(N).astype(np.float16), rng.standard_normal((M, N)).astype(np.float16)
    tx, tw, tb, tr = [to_dev(t, gpu) for t in (x, w, b, r)]
    packed = pkg.pack_weight(tw)
    for kw, okw in epilogues(pkg, oracle, tb, b, tr, r):
        ref = oracle.gemm(x, w, **okw)
        for weight, kernel in ((tw, "auto"), (packed, "packed")):
            if kernel == "packed" and (M > 300 or okw.get("act") == 2):
                continue  # (the library's: it rounds before a separate GELU)
            got = pkg.matmul_ex(tx, weight, kernel=kernel, **kw).cpu().numpy().astype(np.float32)
            assert np.all(np.abs(got - ref) <= spacing_tol(ref, 10, 1e-3)), (kernel, sorted(kw), np.abs(got - ref).max())


@pytest.mark.parametrize("M,K,N", [(1, 8, 8), (77, 776, 200), (300, 640, 1544), (1000, 768, 776)])
def test_matmul_ex_bf16_any_shape(pkg, gpu, M, K, N):
    import torch
    g = torch.Generator(device=gpu).manual_seed(M)
    x, w = torch.randn(M, K, device=gpu, generator=g).bfloat16(), (torch.randn(K, N, device=gpu, generator=g) / K ** 0.5).bfloat16()
    b = torch.randn(N, device=gpu, generator=g).bfloat16()
    ref = (x.double() @ w.double() + b.double()).float()
    got = pkg.matmul_ex(x, w, b).float()
    assert torch.all((got - ref).abs() <= 2.0 ** -8 * ref.abs() + 4e-3)
    if M <= 300:
        got = pkg.matmul_ex(x, pkg.pack_weight(w), b, kernel="packed").float()
        assert torch.all((got - ref).abs() <= 2.0 ** -8 * ref.abs() + 4e-3)


@pytest.mark.parametrize("M,K,N", [(1, 1, 1), (96, 32, 64), (33, 7, 65), (32, 64, 32), (100, 77, 300), (513, 9, 31), (40, 500, 130)])
def test_matmul_ex_f32_small_shapes(pkg, gpu, M, K, N):
    import torch
    g = torch.Generator(device=gpu).manual_seed(K)
    x, w, b, r = [torch.randn(*s, device=gpu, generator=g) for s in ((M, K), (K, N), (N,), (M, N))]
    ref = x.double() @ w.double()
    for kw, f in (({}, lambda y: y), ({"bias": b, "act": 1}, lambda y: (y + b).relu()), ({"bias": b, "residual": r}, lambda y: y + b + r),
                  ({"bias": b, "act": 2}, lambda y: torch.nn.functional.gelu(y + b))):
        err = (pkg.matmul_ex(x, w, **kw).double() - f(ref)).abs().max().item()
        assert err <= 2e-7 * K + 2e-6 * K ** 0.5, (sorted(kw), err)


def test_rows_and_columns_outside_the_shape_are_neither_read_nor_written(pkg, gpu):
    """Operands in the middle of larger arrays full of NaN: nothing of it reaches a result, no neighbour is written."""
    import torch
    for M, K, N, dt in ((77, 776, 200, torch.float16), (300, 640, 1544, torch.float16), (1000, 768, 776, torch.float16), (33, 7, 65, torch.float32)):
        def inside(*shape):
            big = torch.full((shape[0] * shape[1] + 4096,), float("nan"), device=gpu, dtype=dt)
            part = big[2048:2048 + shape[0] * shape[1]].view(*shape)
            part.copy_(torch.randn(*shape, device=gpu))
            return big, part
        (_, x), (_, w), (_, r) = inside(M, K), inside(K, N), inside(M, N)
        big, out = inside(M, N)
        lib = pkg.ops()
        fn = lib.mgpuMatmulExF16 if dt == torch.float16 else lib.mgpuMatmulExF32
        fn(x.data_ptr(), w.data_ptr(), None, out.data_ptr(), r.data_ptr(), M, N, K, 0, 0, 1, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        ref = x.double() @ w.double() + r.double()
        assert torch.all((out.double() - ref).abs() <= 2e-3 * ref.abs() + 0.03 if dt == torch.float16 else (out.double() - ref).abs() < 1e-4)
        assert torch.isnan(big[:2048]).all() and torch.isnan(big[2048 + M * N:]).all()


@pytest.mark.parametrize("M,K,N,act,residual", [
    (1000, 250, 768, 0, True),      # 768 tiles, just short of the line without a GELU, K no multiple of a step
    (2301, 33, 2600, 1, False),     # many tiles of a short reduction, cut on both sides
    (6000, 127, 1990, 2, False),    # 11 844 tiles in front of a GELU
    (1136, 400, 1700, 2, False),
    (100, 1021, 1500, 2, False),    # the deepest reduction
])
def test_matmul_ex_f32_up_to_the_library(pkg, gpu, M, K, N, act, residual):
    import torch
    g = torch.Generator(device=gpu).manual_seed(K)
    x, w, b, r = [torch.randn(*s, device=gpu, generator=g) for s in ((M, K), (K, N), (N,), (M, N))]
    ref = x.double() @ w.double() + b
    ref = ref + r if residual else ref.relu() if act == 1 else torch.nn.functional.gelu(ref) if act == 2 else ref
    err = (pkg.matmul_ex(x, w, b, r if residual else None, act=act).double() - ref).abs().max().item()
    assert err <= 2e-7 * K + 2e-6 * K ** 0.5, err  # the bound of the small shapes above


@pytest.mark.parametrize("M,K,N", [(1145, 80, 1472), (1000, 504, 2040), (2048, 168, 1000)])
def test_packed_weight_two_rounds_of_tiles(pkg, gpu, oracle, rng, M, K, N):
    x = rng.standard_normal((M, K)).astype(np.float16)
    w = (rng.standard_normal((K, N)) / np.sqrt(K)).astype(np.float16)
    b, r = rng.standard_normal(N).astype(np.float16), rng.standard_normal((M, N)).astype(np.float16)
    tx, tw, tb, tr = [to_dev(t, gpu) for t in (x, w, b, r)]
    packed = pkg.pack_weight(tw)
    for kw, okw in epilogues(pkg, oracle, tb, b, tr, r):
        ref = oracle.gemm(x, w, **okw)
        got = pkg.matmul_ex(tx, packed, kernel="packed", **kw).cpu().numpy().astype(np.float32)
        assert np.all(np.abs(got - ref) <= spacing_tol(ref, 10, 1e-3)), (sorted(kw), np.abs(got - ref).max())
