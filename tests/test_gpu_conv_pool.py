"""Parity of mgpuConv2d / mgpuPool2d (C ABI, NCHW fp32) with the oracle.

Pooling is exact (max) or one fp32 rounding of the window sum (average).  The
convolution accumulates fp32 products on the matrix cores in an order of its
own (true fp32 products, unlike the reduced-precision ones the reference
allows through CUDNN_TENSOR_OP_MATH_ALLOW_CONVERSION): the bound is
1e-4 (1 + |ref|), checked elementwise."""
import numpy as np
import pytest

from conftest import to_dev

pytestmark = pytest.mark.gpu


def conv_case(pkg, gpu, oracle, rng, N, IC, H, W, OC, K, pad, stride, dilation, relu, add):
    x = rng.standard_normal((N, IC, H, W)).astype(np.float32)
    w = (rng.standard_normal((OC, IC) + K) / np.sqrt(IC * K[0] * K[1])).astype(np.float32)
    b = rng.standard_normal(OC).astype(np.float32)
    ref = oracle.conv2d(x, w, b, None, pad, stride, dilation, False)
    a = rng.standard_normal(ref.shape).astype(np.float32) if add else None
    ref = oracle.conv2d(x, w, b, a, pad, stride, dilation, relu)
    got = pkg.conv2d(to_dev(x, gpu), to_dev(w, gpu), to_dev(b, gpu), to_dev(a, gpu) if add else None,
                     pad, stride, dilation, relu).cpu().numpy()
    assert got.shape == ref.shape
    err = np.abs(got - ref)
    assert np.all(err <= 1e-4 * (1.0 + np.abs(ref))), err.max()
    return err.max()


@pytest.mark.parametrize("N,IC,H,W,OC,K,pad,stride,dilation,relu,add", [
    (2, 3, 9, 11, 4, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), False, False),
    (1, 4, 12, 10, 5, (3, 2), (0, 1, 2, 0), (2, 1), (1, 1), True, True),    # asymmetric padding
    (2, 2, 15, 15, 3, (3, 3), (2, 2, 2, 2), (2, 2), (2, 2), True, False),    # dilation
    (3, 8, 7, 7, 6, (1, 1), (0, 0, 0, 0), (1, 1), (1, 1), False, True),      # pointwise
    (1, 1, 5, 5, 1, (5, 5), (0, 0, 0, 0), (1, 1), (1, 1), False, False),     # one output element
    (2, 3, 64, 64, 16, (7, 7), (3, 3, 3, 3), (2, 2), (1, 1), True, False),   # ResNet stem, scaled down
    (4, 64, 28, 28, 64, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), True, True),   # ResNet basic block conv + shortcut
    (4, 256, 14, 14, 64, (1, 1), (0, 0, 0, 0), (1, 1), (1, 1), True, False), # bottleneck reduce
    (2, 64, 28, 28, 128, (1, 1), (0, 0, 0, 0), (2, 2), (1, 1), False, False),# strided pointwise (downsample)
])
def test_conv2d(pkg, gpu, oracle, rng, N, IC, H, W, OC, K, pad, stride, dilation, relu, add):
    conv_case(pkg, gpu, oracle, rng, N, IC, H, W, OC, K, pad, stride, dilation, relu, add)


@pytest.mark.parametrize("N,IC,H,W,OC,K,pad,stride,dilation,relu,add", [
    (2, 3, 64, 64, 256, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), True, True),       # nine window rows, whole tiles
    (64, 3, 8, 16, 250, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), False, True),      # an image a tile, channels past the end
    (130, 3, 6, 12, 225, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), True, False),     # tiles over several images, the last one cut
    (40, 1, 16, 20, 249, (5, 5), (2, 2, 2, 2), (1, 1), (1, 1), False, False),    # five rows of five
    (40, 1, 16, 20, 249, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), False, False),    # three rows
    (20, 2, 20, 24, 256, (3, 3), (0, 2, 2, 0), (1, 1), (1, 1), False, False),    # both columns left of the pixel
    (20, 3, 40, 26, 256, (3, 3), (1, 0, 1, 0), (2, 1), (1, 1), True, False),     # none, stride down
    (30, 3, 20, 20, 256, (2, 1), (0, 0, 0, 0), (1, 1), (1, 1), False, True),     # six rows of one column
    (30, 1, 24, 20, 256, (3, 1), (2, 0, 2, 0), (1, 1), (2, 3), False, False),    # dilated down (across, one column: nothing to dilate)
    (24, 16, 20, 24, 256, (1, 1), (0, 0, 0, 0), (1, 1), (1, 1), False, False),   # sixteen rows
])
def test_conv2d_of_few_taps_four_pixels_a_lane(pkg, gpu, oracle, rng, N, IC, H, W, OC, K, pad, stride, dilation, relu, add):
    conv_case(pkg, gpu, oracle, rng, N, IC, H, W, OC, K, pad, stride, dilation, relu, add)


@pytest.mark.parametrize("N,IC,H,W,OC,K,pad,stride,dilation,relu,add", [
    # eight wavefronts a tile: 80 and 48 groups of channels (shares that are no whole chunks), 73 (cut shares, a last piece half past
    # the filter's end), 25 (5 x 5), a last channel tile of one, images smaller than a tile
    (5, 160, 7, 7, 33, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), True, True), (2, 96, 9, 31, 32, (3, 3), (0, 2, 1, 0), (2, 1), (1, 2), False, False),
    (5, 146, 50, 51, 32, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), True, True), (3, 50, 11, 13, 40, (5, 5), (2, 2, 2, 2), (1, 1), (1, 1), True, True),
    (1, 256, 1, 1, 33, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), False, True), (1, 256, 3, 5, 17, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), False, True),
    (2, 128, 7, 9, 64, (3, 3), (1, 1, 1, 1), (2, 2), (1, 1), True, False),
    # four: 17, 19 and 33 groups, one and several channel tiles, 64-channel tiles cut, the last pixel tile cut
    (7, 34, 50, 51, 32, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), False, True), (6, 38, 41, 40, 64, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), True, False),
    (4, 66, 41, 66, 64, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), False, True), (4, 18, 30, 91, 32, (5, 5), (2, 2, 2, 2), (1, 1), (1, 1), False, True),
    (9, 32, 50, 61, 32, (5, 5), (2, 2, 2, 2), (1, 1), (1, 1), True, False),
    (3, 70, 61, 60, 96, (3, 3), (2, 2, 2, 2), (1, 1), (2, 2), False, False),
    (7, 38, 41, 40, 48, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), True, False),
    # the same where rows of the filter are no whole lines, or channels few: another kernel
    (1, 256, 3, 5, 1, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), False, True),
    (5, 66, 7, 7, 33, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), True, True), (2, 70, 9, 31, 32, (3, 3), (0, 2, 1, 0), (2, 1), (1, 2), False, False),
    (1, 64, 1, 1, 1, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), False, True), (3, 34, 11, 13, 40, (5, 5), (2, 2, 2, 2), (1, 1), (1, 1), True, True),
    (5, 34, 50, 51, 32, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), False, True), (8, 38, 41, 40, 48, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), True, False),
    # 7 x 7: rows and columns outside on every side, dilation, eight groups and an odd number; eight and four wavefronts
    (2, 18, 5, 6, 33, (7, 7), (3, 3, 3, 3), (1, 1), (1, 1), True, True), (3, 16, 20, 23, 40, (7, 7), (4, 6, 5, 2), (2, 1), (1, 2), False, False),
    (4, 22, 41, 60, 32, (7, 7), (3, 3, 3, 3), (1, 1), (1, 1), False, True), (3, 16, 50, 51, 64, (7, 7), (3, 3, 3, 3), (1, 1), (2, 1), True, False)])
def test_conv2d_with_the_filter_through_lds(pkg, gpu, oracle, rng, N, IC, H, W, OC, K, pad, stride, dilation, relu, add):
    conv_case(pkg, gpu, oracle, rng, N, IC, H, W, OC, K, pad, stride, dilation, relu, add)


@pytest.mark.parametrize("N,IC,H,W,OC,K,pad,stride,dilation,relu,add", [
    (2, 3, 37, 67, 33, (7, 7), (3, 3, 3, 3), (1, 1), (1, 1), True, True),      # rows of two tiles and a bit, a channel tile of one
    (3, 3, 40, 130, 64, (7, 7), (3, 3, 3, 3), (2, 2), (1, 1), True, False),    # the ResNet stem; tiles with nothing outside
    (2, 1, 20, 100, 32, (7, 7), (0, 5, 6, 0), (1, 1), (2, 1), False, True),    # dilated down, padding on two sides
    (70, 1, 9, 22, 40, (7, 7), (3, 2, 3, 4), (3, 1), (1, 1), False, False),    # rows shorter than a tile, several tiles a wavefront
    (2, 3, 33, 96, 520, (5, 5), (2, 2, 2, 2), (1, 1), (1, 1), False, True),    # whole tiles, 17 channel tiles
    (1, 3, 5, 39, 1, (5, 5), (0, 0, 0, 0), (1, 2), (1, 1), True, False),       # one output row: few tiles, not by patches
    (40, 3, 5, 299, 96, (5, 5), (0, 0, 0, 0), (1, 2), (1, 1), True, False),    # one output row an image
    (40, 3, 5, 299, 64, (5, 5), (0, 0, 0, 0), (1, 2), (1, 1), True, True),     # ... of fewer tiles: not by patches
])
def test_conv2d_of_few_channels_by_patches(pkg, gpu, oracle, rng, N, IC, H, W, OC, K, pad, stride, dilation, relu, add):
    conv_case(pkg, gpu, oracle, rng, N, IC, H, W, OC, K, pad, stride, dilation, relu, add)


@pytest.mark.parametrize("C,H,W,K,pad,stride", [
    (3, 8, 8, (2, 2), (0, 0, 0, 0), (2, 2)), (2, 9, 7, (3, 3), (1, 1, 1, 1), (2, 2)),
    (64, 112, 112, (3, 3), (1, 1, 1, 1), (2, 2)),  # ResNet stem pool
    (512, 7, 7, (7, 7), (0, 0, 0, 0), (1, 1)),     # global average pool
    (2, 10, 11, (3, 2), (1, 0, 1, 1), (2, 1)),
])
def test_pool2d(pkg, gpu, oracle, rng, C, H, W, K, pad, stride):
    x = rng.standard_normal((2, C, H, W)).astype(np.float32)
    tx = to_dev(x, gpu)
    assert np.array_equal(pkg.pool2d(tx, K, pad, stride, "max").cpu().numpy(), oracle.pool2d(x, K, pad, stride, "max"))
    avg, ref = pkg.pool2d(tx, K, pad, stride, "avg").cpu().numpy(), oracle.pool2d(x, K, pad, stride, "avg")
    assert np.all(np.abs(avg - ref) <= 1e-6 * (1 + np.abs(ref)))


def test_conv_pool_reject_bad_arguments(pkg, gpu):
    import torch
    x = torch.zeros((1, 2, 8, 8), device=gpu)
    w = torch.zeros((3, 2, 3, 3), device=gpu)
    b = torch.zeros(3, device=gpu)
    lib = pkg.ops()
    out = torch.zeros((1, 3, 8, 8), device=gpu)
    args = lambda OH: (x.data_ptr(), w.data_ptr(), b.data_ptr(), out.data_ptr(), None, 1, 2, 8, 8, 3, 3, 3, OH, 8,
                       1, 1, 1, 1, 1, 1, 1, 1, False, False, None)
    lib.mgpuConv2d(*args(7))
    assert b"output size does not follow" in lib.mgpuOpsTakeLastError()
    lib.mgpuConv2d(*args(8)[:4], None, *args(8)[5:22], True, False, None)
    assert b"hasPostAdd" in lib.mgpuOpsTakeLastError()
    lib.mgpuPool2d(x.data_ptr(), out.data_ptr(), 1, 2, 8, 8, 4, 4, 2, 2, 0, 0, 0, 0, 2, 2, 5, None)
    assert b"method" in lib.mgpuOpsTakeLastError()
    lib.mgpuPool2d(x.data_ptr(), out.data_ptr(), 1, 2, 8, 8, 5, 5, 2, 2, 2, 2, 0, 0, 2, 2, 0, None)
    assert b"padding must be smaller" in lib.mgpuOpsTakeLastError()
    assert lib.mgpuOpsTakeLastError() is None


@pytest.mark.parametrize("N,IC,H,W,OC,K,pad,stride,dilation,relu,add", [
    # few taps (K <= 32): the step counts 5, 8, 14 and 16, one and two accumulators, a last channel tile of one, dilation
    (3, 1, 9, 7, 33, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), True, True), (2, 16, 6, 5, 1, (1, 1), (0, 0, 0, 0), (1, 1), (1, 1), False, False),
    (40, 3, 33, 31, 65, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), True, True), (5, 2, 17, 19, 40, (4, 4), (2, 1, 1, 2), (2, 1), (1, 2), False, False),
    # window kernel: odd channels, 5 x 5 and 7 x 7 rows, images smaller than a tile
    (5, 5, 7, 7, 33, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), True, False), (2, 3, 21, 18, 32, (5, 5), (2, 2, 2, 2), (1, 1), (1, 1), False, True),
    (1, 4, 20, 23, 8, (7, 7), (3, 3, 3, 3), (2, 2), (1, 1), True, False), (9, 37, 3, 3, 64, (1, 1), (0, 0, 0, 0), (1, 1), (1, 1), False, True),
    (6, 8, 60, 61, 96, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), True, False), (10, 36, 60, 61, 32, (1, 1), (0, 0, 0, 0), (1, 1), (1, 1), False, False),
    (8, 3, 90, 90, 24, (5, 5), (2, 2, 2, 2), (1, 1), (1, 1), False, False), (3, 8, 60, 61, 32, (3, 3), (1, 1, 1, 1), (1, 1), (2, 2), False, False),
    # LDS tiles: one, two and four wavefront groups, channels that do not fill the last group
    (8, 9, 50, 51, 64, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), True, True), (8, 50, 40, 40, 48, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), False, False),
    (6, 131, 30, 31, 100, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), True, False), (8, 72, 41, 40, 130, (1, 1), (0, 0, 0, 0), (1, 1), (1, 1), False, True),
    (5, 6, 64, 64, 64, (5, 5), (2, 2, 2, 2), (1, 1), (1, 1), False, False), (6, 4, 90, 90, 64, (7, 7), (3, 3, 3, 3), (1, 1), (1, 1), True, False),
    # the table: windows that are no square of 1, 3, 5 or 7; more than one segment of it
    (2, 12, 20, 22, 40, (1, 7), (0, 3, 0, 3), (1, 1), (1, 1), True, True), (2, 300, 9, 11, 33, (2, 4), (1, 1, 0, 2), (1, 1), (2, 1), False, False),
    # windows and dilations beyond the table's narrow form
    (1, 1, 70, 3, 2, (40, 1), (0, 0, 0, 0), (1, 1), (1, 1), False, False), (1, 2, 4000, 1, 3, (3, 1), (1, 0, 0, 0), (7, 1), (1500, 1), True, False)])
def test_conv2d_every_kernel(pkg, gpu, oracle, rng, N, IC, H, W, OC, K, pad, stride, dilation, relu, add):
    conv_case(pkg, gpu, oracle, rng, N, IC, H, W, OC, K, pad, stride, dilation, relu, add)


def test_conv2d_padding_and_filler_do_not_multiply_garbage(pkg, gpu):
    """Operands the kernels make up (taps outside the image, channels and taps past the end) are zeros on both sides:
    an Inf or NaN in a neighbouring channel, filter row or image never reaches another output."""
    import torch
    for IC, OC, K, HW in ((3, 34, 3, 20), (5, 34, 3, 20), (5, 64, 3, 70), (33, 40, 1, 12), (7, 33, 2, 9)):
        g = torch.Generator(device=gpu).manual_seed(IC)
        x, w = torch.randn(2, IC, HW, HW, device=gpu, generator=g), torch.randn(OC, IC, K, K, device=gpu, generator=g)
        b = torch.zeros(OC, device=gpu)
        p = K // 2
        clean = pkg.conv2d(x, w, b, pad=(p,) * 4)
        x[1], w[1] = float("nan"), float("inf")
        dirty = pkg.conv2d(x, w, b, pad=(p,) * 4)
        keep = [o for o in range(OC) if o != 1]
        assert torch.equal(clean[0, keep], dirty[0, keep]), (IC, OC, K)


@pytest.mark.parametrize("N,H,W,K", [
    (1, 20001, 20003, (1, 1)),  # the table's wide form (an image beyond 2 GiB): pixels and taps past the end in one tile
    # more pixels than one grid dimension holds threads for: 2^29 and some; the wide form again, the table in 32 bits
    (1, 23184, 23175, (1, 1)), (3, 11009, 16400, (2, 17)),
])
def test_conv2d_of_large_images(pkg, gpu, N, H, W, K):
    """Whole numbers, every sum below 2^24: exact in any order."""
    import torch
    g = torch.Generator(device=gpu).manual_seed(H)
    x = torch.empty((N, 1, H, W), device=gpu).random_(0, 1000, generator=g)
    w = torch.empty((1, 1) + K, device=gpu).random_(-7, 8, generator=g)
    y = pkg.conv2d(x, w, torch.full((1,), 5.0, device=gpu))
    for n in range(N):
        want = torch.full_like(y[n, 0], 5.0)
        for i in range(K[0]):
            for j in range(K[1]):
                want += w[0, 0, i, j] * x[n, 0, i:i + y.shape[2], j:j + y.shape[3]]
        assert torch.equal(y[n, 0], want), n


@pytest.mark.gpu
@pytest.mark.parametrize("N,H,W,OC,add", [
    (27, 219, 40, 256, False),   # 231 MiB of rows that are no whole lines: plain stores
    (16, 256, 256, 64, False),   # 256 MiB of whole ones: non-temporal
    (14, 200, 200, 64, False),   # 137 MiB: written through
    (27, 219, 40, 250, True),    # beside an addend: non-temporal, channels past the end
])
def test_conv2d_of_few_taps_and_large_outputs(pkg, gpu, N, H, W, OC, add):
    """Each way of storing; 1 x 1 from two channels, so that a reference is two products and sums in float64."""
    import torch
    g = torch.Generator(device=gpu).manual_seed(N + OC)
    r = lambda *s: torch.randn(s, generator=g, device=gpu)
    x, w, b = r(N, 2, H, W), r(OC, 2, 1, 1), r(OC)
    post = r(N, OC, H, W) if add else None
    count = N * OC * H * W
    out = torch.full((count + 64,), 7.0, device=gpu)  # 32 elements before and behind
    pkg.ops().mgpuConv2d(x.data_ptr(), w.data_ptr(), b.data_ptr(), out[32:].data_ptr(), post.data_ptr() if add else None, N, 2, H, W, OC, 1, 1,
                         H, W, 0, 0, 0, 0, 1, 1, 1, 1, add, False, torch.cuda.current_stream().cuda_stream)
    assert (out[:32] == 7).all() and (out[-32:] == 7).all()
    got = out[32:-32].view(N, OC, H, W)
    for n in range(N):
        a, c = (w[:, i, :, :].double() * x[n, i].double() for i in (0, 1))
        ref, size = a + c + b.double()[:, None, None], a.abs() + c.abs() + b.abs().double()[:, None, None]
        if add:
            ref, size = ref + post[n].double(), size + post[n].abs().double()
        assert ((got[n].double() - ref).abs() <= 4 * 2.0**-24 * size).all()  # a rounding each of at most four partial sums
