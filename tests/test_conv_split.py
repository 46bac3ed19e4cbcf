"""3 x 3 convolution in three bf16 numbers (csrc/kernels/conv_split.hip): that its tiles' input rows fit their place in LDS, which
convolutions it takes, and its results against the oracle and against 64 bits, on operands of every size."""
import ctypes
import random

import numpy as np
import pytest

from conftest import to_dev
from test_index_bounds import internal


class Plan(ctypes.Structure):
    _fields_ = [("tile", ctypes.c_int), ("strips", ctypes.c_int), ("us", ctypes.c_double)]


TILES = [(64, 256), (64, 448), (128, 256), (128, 448), (256, 448)]  # pixels, staged pixels at most


def plan_of(pkg, *args, limit=1e9):
    return internal(pkg, "_ZN4mgpu13convSplitPlanEiiiiiiiiiid", Plan, *[ctypes.c_int] * 10, ctypes.c_double)(*args, 256, limit)


def most_staged(pixels, N, OH, OW, S, D, strips):
    """Input pixels that a tile's windows lie in at most, as the kernel stages them: whole rows from the first to the last."""
    width = -(-OW // strips)
    rows, pitch, total = (OH - 1) * S[0] + 2 * D[0] + 1, (width - 1) * S[1] + 2 * D[1] + 1, N * strips * OH * width

    def first_row(q):
        return q // (OH * width) * rows + q % (OH * width) // width * S[0]
    return max(first_row(min(p + pixels, total) - 1) + 2 * D[0] + 1 - first_row(p) for p in range(0, total, pixels)) * pitch


def test_staged_rows_fit(pkg):
    rng = random.Random(5)
    size = lambda low, high: int(round(low * (high / low) ** rng.random()))  # noqa: E731
    seen = set()
    for _ in range(3000):
        N, OH, OW, IC, OC = size(1, 40), size(1, 70), size(1, 400), rng.choice([32, 48, 256]), rng.choice([8, 96, 512])
        S, D = (rng.randint(1, 3), rng.randint(1, 3)), (rng.randint(1, 3), rng.randint(1, 2))
        plan = plan_of(pkg, N, IC, OC, OH, OW, *S, *D)
        if plan.strips == 0: continue
        seen.add(plan.tile)
        pixels, cap = TILES[plan.tile]
        assert most_staged(pixels, N, OH, OW, S, D, plan.strips) <= cap, (N, OH, OW, S, D, plan.tile, plan.strips)
    assert seen == set(range(5))


@pytest.mark.parametrize("N,IC,OC,HW,split", [
    (4, 64, 64, 28, False),    # one tile of 32 x 32 a CU
    (32, 64, 64, 56, True),
    (7, 128, 128, 10, False),
    (13, 128, 128, 30, True),
    (1, 256, 256, 24, False),
    (5, 256, 256, 18, True),
])
def test_who_takes_it(pkg, N, IC, OC, HW, split):
    time = internal(pkg, "_ZN4mgpu14convWindowTimeEllllll", ctypes.c_double, *[ctypes.c_int64] * 6)(1, N * HW * HW, IC, OC, HW, 256)
    assert (plan_of(pkg, N, IC, OC, HW, HW, 1, 1, 1, 1, limit=0.97 * time).strips > 0) is split


def split_conv(pkg, tile, strips, x, w, b, add, pad, stride, dilation, relu):
    import torch
    N, IC, H, W = x.shape
    OC = w.shape[0]
    OH, OW = ((s + pad[i] + pad[i + 2] - 2 * dilation[i] - 1) // stride[i] + 1 for i, s in enumerate((H, W)))
    strips = next((s for s in range(strips, OW + 1) if most_staged(TILES[tile][0], N, OH, OW, stride, dilation, s) <= TILES[tile][1]), 0)
    if not strips: pytest.skip("no strips of it fit this tile")
    count = N * OC * OH * OW
    out = torch.full((count + 64,), 7.0, device=x.device)  # 32 elements before and behind
    launch = internal(pkg, "_ZN4mgpu9convSplitERKNS_13ConvSplitPlanEPKfS4_S4_PfS4_lllllllllllllbP12ihipStream_t", ctypes.c_bool, ctypes.POINTER(Plan),
                      *[ctypes.c_void_p] * 5, *[ctypes.c_int64] * 13, ctypes.c_bool, ctypes.c_void_p)
    pkg.ops()
    assert launch(ctypes.byref(Plan(tile, strips, 0.0)), x.data_ptr(), w.data_ptr(), b.data_ptr(), out[32:].data_ptr(), add.data_ptr() if add is not None else None,
                  N, IC, H, W, OC, OH, OW, pad[0], pad[1], *stride, *dilation, relu, torch.cuda.current_stream().cuda_stream)
    assert (out[:32] == 7).all() and (out[-32:] == 7).all()
    return out[32:-32].view(N, OC, OH, OW)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", range(5))
@pytest.mark.parametrize("N,IC,H,W,OC,pad,stride,dilation,relu,add,strips", [
    (1, 32, 1, 1, 1, (1, 1, 1, 1), (1, 1), (1, 1), False, False, 1),      # one output, two steps
    (3, 48, 9, 11, 33, (1, 1, 1, 1), (1, 1), (1, 1), True, True, 1),      # an odd number of steps, a channel tile of one, several images a tile
    (2, 64, 16, 17, 40, (0, 2, 1, 0), (1, 1), (1, 1), False, True, 2),    # a last strip that is narrower, asymmetric padding
    (2, 16, 13, 12, 64, (2, 1, 0, 3), (2, 1), (1, 1), True, False, 1),    # one step
    (5, 32, 7, 6, 32, (2, 2, 2, 2), (1, 1), (2, 2), False, False, 1),     # dilation
    (4, 80, 8, 16, 72, (1, 1, 1, 1), (1, 1), (1, 1), False, False, 2),    # whole tiles
])
def test_against_the_oracle(pkg, gpu, oracle, rng, tile, N, IC, H, W, OC, pad, stride, dilation, relu, add, strips):
    x, w = rng.standard_normal((N, IC, H, W)).astype(np.float32), (rng.standard_normal((OC, IC, 3, 3)) / np.sqrt(9 * IC)).astype(np.float32)
    b = rng.standard_normal(OC).astype(np.float32)
    shape = oracle.conv2d(x, w, b, None, pad, stride, dilation, False).shape
    a = rng.standard_normal(shape).astype(np.float32) if add else None
    ref = oracle.conv2d(x, w, b, a, pad, stride, dilation, relu)
    got = split_conv(pkg, tile, strips, to_dev(x, gpu), to_dev(w, gpu), to_dev(b, gpu), to_dev(a, gpu) if add else None, pad, stride, dilation,
                     relu).cpu().numpy()
    # both sides are a sum of K products of fp32 accuracy: 2^-24 of the sum of their sizes (here about 1) times some sqrt(K)
    assert np.all(np.abs(got - ref) <= 1e-5 * (1 + np.abs(ref))), np.abs(got - ref).max()


KINDS = ["normal", "tiny", "huge", "dark half", "outlier", "growing", "growing filter", "zero channels", "zero filter channels", "dead filters", "zeros",
         "inf", "inf filter", "nan"]
# Values that are small beside others of the same window, by channel, by pixel and by image, which the filter brings up again or has alone.
UNEVEN = ["channels 1e-4", "channels 1e-6", "channels 1e-9", "selected 1e-6", "selected 1e-12", "selected beside an outlier", "last channels", "dim image",
          "near the smallest"]


def uneven(kind, x, w):
    r = float(kind.split()[-1]) if "1e-" in kind else 1e-7
    if kind.startswith("channels"): x[:, 1::2] *= r; w[:, ::2] *= r  # noqa: E702
    if kind.startswith("selected"): x[:, 1::2] *= r; w[:, ::2] = 0  # noqa: E702
    if kind == "selected beside an outlier": x[:, 1, 3, 3] = 1.0
    if kind == "last channels": x[:, -1] *= r; w[:, :-1] *= r  # noqa: E702
    if kind == "dim image": x[1, 1::2] *= r; w[:, ::2] *= r  # noqa: E702
    if kind == "near the smallest": x *= 1e-36; w *= 1e8  # noqa: E702


def operands(kind, N, IC, H, W, OC, device):
    import torch
    gen = torch.Generator(device=device).manual_seed(len(kind))
    r = lambda *s: torch.randn(s, device=device, generator=gen)  # noqa: E731
    x, w, c = r(N, IC, H, W), r(OC, IC, 3, 3), min(IC - 1, 16)
    if kind == "tiny": x, w = x * 1e-12, w * 1e-9
    if kind == "huge": x, w = x * 1e14, w * 1e9
    if kind == "dark half": x[:, :, :, :W // 2 + 1] *= 1e-9
    if kind == "outlier": x[1, IC // 2, 3, 3] = 1e7
    if kind == "growing": x[:, c:] *= 1e4
    if kind == "growing filter": w[:, c:] *= 1e4
    if kind == "zero channels": x[:, :c] = 0
    if kind == "zero filter channels": w[:, :c], w[1] = 0, 1e-12 * w[1]
    if kind == "dead filters": w[::3] *= 1e-20
    if kind == "zeros": x.zero_()
    if kind == "inf": x[0, c - 1, 4, 4] = float("inf")
    if kind == "inf filter": w[3, c, 1, 1] = float("-inf")
    if kind == "nan": x[1, c - 1, 5, 6], w[2, c - 1, 0, 0] = float("nan"), float("nan")
    if kind in UNEVEN: uneven(kind, x, w)
    return x, w


def check(got, x, w, kind):
    """Against 64 bits, elementwise to the size of the products summed up: infinities and NaNs go the fp32 way."""
    import torch
    H, W = x.shape[2:]
    conv = lambda x, w: sum(torch.nn.functional.pad(x, (1, 1, 1, 1))[:, None, :, i:i + H, j:j + W].mul(w[None, :, :, i, j, None, None]).sum(2)  # noqa: E731
                            for i in range(3) for j in range(3))
    ref, size, got = conv(x.double(), w.double()), conv(x.double().abs(), w.double().abs()), got.double()
    finite = torch.isfinite(ref)
    assert torch.equal(torch.isnan(got), torch.isnan(ref))
    assert torch.equal(got[~finite & ~torch.isnan(ref)], ref[~finite & ~torch.isnan(ref)])
    # 2^-24 a product and rounding: some hundreds of them, whose errors are far from all of one sign
    assert (got - ref).abs()[finite].le(2.0 ** -20 * size[finite]).all(), kind


@pytest.mark.gpu
@pytest.mark.parametrize("kind", KINDS + UNEVEN)
def test_operands_of_every_size(pkg, gpu, kind):
    import torch
    x, w = operands(kind, 2, 64, 14, 16, 40, gpu)
    for tile in (0, 4):
        check(split_conv(pkg, tile, 1, x, w, torch.zeros(40, device=gpu), None, (1, 1, 1, 1), (1, 1), (1, 1), False), x, w, kind)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [0, 2, 4])
def test_an_image_for_itself(pkg, gpu, tile):
    """The bits of an image's result, whatever the images are that share its tiles."""
    import torch
    x, w = operands("normal", 3, 48, 7, 9, 40, gpu)
    b = torch.randn(40, device=gpu)
    alone = split_conv(pkg, tile, 1, x[1:2].contiguous(), w, b, None, (1, 1, 1, 1), (1, 1), (1, 1), False)
    for value in (1.0, 1e-8, 1e8, float("inf"), float("nan")):
        x[0], x[2] = x[0] * 1e4, value
        assert torch.equal(split_conv(pkg, tile, 1, x, w, b, None, (1, 1, 1, 1), (1, 1), (1, 1), False)[1:2], alone), value


@pytest.mark.gpu
@pytest.mark.parametrize("kind", KINDS + UNEVEN)
@pytest.mark.parametrize("IC", [2, 3])
def test_operands_of_every_size_in_a_stem(pkg, gpu, kind, IC):
    """The kernel of few taps and four pixels a lane, on the same terms (512 tiles of 128 pixels x 32 channels)."""
    import torch
    x, w = operands(kind, 2, IC, 64, 64, 250, gpu)
    check(pkg.conv2d(x, w, torch.zeros(250, device=gpu), pad=(1, 1, 1, 1)), x, w, kind)


@pytest.mark.gpu
def test_a_stem_of_nothing_beside_large_values(pkg, gpu):
    """Where the other products overflow, a filter of zeros and a window of zeros still give the bias."""
    import torch
    x, w = operands("normal", 2, 3, 64, 64, 250, gpu)
    b = torch.randn(250, device=gpu)
    x, w = x * 1e25, w * 1e25
    x[:, :, 8:16, 8:16], w[77] = 0, 0
    got = pkg.conv2d(x, w, b, pad=(1, 1, 1, 1))
    assert torch.equal(got[:, 77], b[77].expand(2, 64, 64)) and torch.equal(got[:, :, 9:15, 9:15], b[:, None, None].expand(2, 250, 6, 6))


@pytest.mark.gpu
def test_an_image_of_a_stem_for_itself(pkg, gpu):
    import torch
    x, w = operands("normal", 3, 3, 61, 60, 250, gpu)  # 128 pixels of a tile lie in two images
    b = torch.randn(250, device=gpu)
    alone = pkg.conv2d(x, w, b, pad=(1, 1, 1, 1))[1]
    for value in (1e-8, 1e8, float("inf")):
        x[0], x[2] = value, value
        assert torch.equal(pkg.conv2d(x, w, b, pad=(1, 1, 1, 1))[1], alone), value
