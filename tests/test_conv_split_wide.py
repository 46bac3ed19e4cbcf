"""5 x 5 and 7 x 7 convolution in three bf16 numbers (csrc/kernels/conv_split.hip): that its tiles' input rows fit their place in LDS, which convolutions
it takes, and its results against the oracle and against 64 bits, on operands of every size."""
import ctypes
import random

import numpy as np
import pytest

from conftest import to_dev
from test_conv_split import KINDS, UNEVEN, Plan, uneven
from test_index_bounds import internal

TILES = {5: (64, 512), 6: (128, 512), 7: (64, 960), 8: (128, 960)}  # pixels, staged pixels at most
TILES_OF = {5: (5, 6), 7: (7, 8)}


def plan_of(pkg, win, *args, limit=1e9):
    return internal(pkg, f"_ZN4mgpu14convSplitPlan{win}Eiiiiiiiiiid", Plan, *[ctypes.c_int] * 10, ctypes.c_double)(*args, 256, limit)


def most_staged(win, pixels, N, OH, OW, S, D, strips):
    """Input pixels that a tile's windows lie in at most, as the kernel stages them: whole rows from the first to the last."""
    width = -(-OW // strips)
    rows, pitch, total = (OH - 1) * S[0] + (win - 1) * D[0] + 1, (width - 1) * S[1] + (win - 1) * D[1] + 1, N * strips * OH * width

    def first_row(q):
        return q // (OH * width) * rows + q % (OH * width) // width * S[0]
    return max(first_row(min(p + pixels, total) - 1) + (win - 1) * D[0] + 1 - first_row(p) for p in range(0, total, pixels)) * pitch


@pytest.mark.parametrize("win", [5, 7])
def test_staged_rows_fit(pkg, win):
    rng = random.Random(win)
    size = lambda low, high: int(round(low * (high / low) ** rng.random()))  # noqa: E731
    seen = set()
    for _ in range(3000):
        N, OH, OW, IC, OC = size(1, 40), size(1, 70), size(1, 400), rng.choice([16, 24, 256]), rng.choice([8, 96, 512])
        S, D = (rng.randint(1, 2), rng.randint(1, 2)), (rng.randint(1, 2), rng.randint(1, 2) if win == 5 else 1)
        plan = plan_of(pkg, win, N, IC, OC, OH, OW, *S, *D)
        if plan.strips == 0: continue
        seen.add(plan.tile)
        pixels, cap = TILES[plan.tile]
        assert most_staged(win, pixels, N, OH, OW, S, D, plan.strips) <= cap, (N, OH, OW, S, D, plan.tile, plan.strips)
    assert seen == set(TILES_OF[win])


def split_conv(pkg, tile, strips, x, w, b, add, pad, stride, dilation, relu):
    import torch
    N, IC, H, W = x.shape
    OC, win = w.shape[0], w.shape[2]
    OH, OW = ((s + pad[i] + pad[i + 2] - (win - 1) * dilation[i] - 1) // stride[i] + 1 for i, s in enumerate((H, W)))
    strips = next((s for s in range(strips, OW + 1) if most_staged(win, TILES[tile][0], N, OH, OW, stride, dilation, s) <= TILES[tile][1]), 0)
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
@pytest.mark.parametrize("win", [5, 7])
@pytest.mark.parametrize("tile", [0, 1, None])  # None: through the package, which takes the larger ones here (the last shape)
@pytest.mark.parametrize("N,IC,H,W,OC,pad,stride,dilation,relu,add,strips", [
    (1, 16, 1, 1, 1, (2, 2, 2, 2), (1, 1), (1, 1), False, False, 1),      # one output, two (7 x 7: four) steps
    (3, 24, 9, 11, 33, (2, 2, 2, 2), (1, 1), (1, 1), True, True, 1),      # an odd number of steps, a channel tile of one, several images a tile
    (2, 32, 16, 17, 40, (0, 3, 2, 1), (1, 1), (1, 1), False, True, 2),    # a last strip that is narrower, asymmetric padding
    (2, 4, 13, 12, 64, (2, 1, 4, 3), (2, 1), (1, 1), True, False, 1),     # one step of 7 x 7
    (2, 8, 13, 12, 64, (2, 1, 4, 3), (2, 1), (1, 1), True, False, 1),     # one step
    (5, 16, 7, 6, 32, (4, 4, 4, 4), (1, 1), (2, 2), False, False, 1),     # dilation
    (4, 40, 8, 16, 72, (2, 2, 2, 2), (1, 1), (1, 1), False, False, 2),    # whole tiles
    (9, 32, 50, 56, 32, (2, 2, 2, 2), (1, 1), (1, 1), True, True, 1),
])
def test_against_the_oracle(pkg, gpu, oracle, rng, win, tile, N, IC, H, W, OC, pad, stride, dilation, relu, add, strips):
    if IC % (8 if win == 5 else 4) or (win == 7 and dilation[1] > 1): pytest.skip("not for this kernel")
    pad = tuple(p + (win - 5) // 2 * d for p, d in zip(pad, dilation * 2))
    x, w = rng.standard_normal((N, IC, H, W)).astype(np.float32), (rng.standard_normal((OC, IC, win, win)) / (win * np.sqrt(IC))).astype(np.float32)
    b = rng.standard_normal(OC).astype(np.float32)
    shape = oracle.conv2d(x, w, b, None, pad, stride, dilation, False).shape
    a = rng.standard_normal(shape).astype(np.float32) if add else None
    ref = oracle.conv2d(x, w, b, a, pad, stride, dilation, relu)
    args = to_dev(x, gpu), to_dev(w, gpu), to_dev(b, gpu), to_dev(a, gpu) if add else None
    if tile is None: got = pkg.conv2d(*args, pad=pad, stride=stride, dilation=dilation, relu=relu).cpu().numpy()
    else: got = split_conv(pkg, TILES_OF[win][tile], strips, *args, pad, stride, dilation, relu).cpu().numpy()
    # both sides are a sum of K products of fp32 accuracy: 2^-24 of the sum of their sizes (here about 1) times some sqrt(K)
    assert np.all(np.abs(got - ref) <= 1e-5 * (1 + np.abs(ref))), np.abs(got - ref).max()


def operands(kind, N, IC, H, W, OC, win, device):
    import torch
    gen = torch.Generator(device=device).manual_seed(len(kind))
    r = lambda *s: torch.randn(s, device=device, generator=gen)  # noqa: E731
    x, w, c = r(N, IC, H, W), r(OC, IC, win, win), 8 if win == 5 else 4
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
    if kind == "inf": x[0, c - 1, 4, 4] = float("inf")  # (the last position of a window among them, beside the fillers)
    if kind == "inf filter": w[3, c, -1, -1] = float("-inf")
    if kind == "nan": x[1, c - 1, 5, 6], w[2, c - 1, -1, -1] = float("nan"), float("nan")
    if kind in UNEVEN: uneven(kind, x, w)
    return x, w


@pytest.mark.gpu
@pytest.mark.parametrize("win", [5, 7])
@pytest.mark.parametrize("kind", KINDS + UNEVEN)
def test_operands_of_every_size(pkg, gpu, kind, win):
    """Against 64 bits, elementwise to the size of the products summed up: infinities and NaNs go the fp32 way."""
    import torch
    x, w = operands(kind, 2, 32, 14, 16, 40, win, gpu)
    (H, W), p = x.shape[2:], win // 2
    conv = lambda x, w: sum(torch.nn.functional.pad(x, (p, p, p, p))[:, None, :, i:i + H, j:j + W].mul(w[None, :, :, i, j, None, None]).sum(2)  # noqa: E731
                            for i in range(win) for j in range(win))
    ref, size = conv(x.double(), w.double()), conv(x.double().abs(), w.double().abs())
    finite = torch.isfinite(ref)
    for tile in TILES_OF[win]:
        got = split_conv(pkg, tile, 1, x, w, torch.zeros(40, device=gpu), None, (p, p, p, p), (1, 1), (1, 1), False).double()
        assert torch.equal(torch.isnan(got), torch.isnan(ref))
        assert torch.equal(got[~finite & ~torch.isnan(ref)], ref[~finite & ~torch.isnan(ref)])
        # The fp32 way has two chains of K / 4 additions, each of which rounds by up to 2^-24 of the running sum (which an outlier makes as large as
        # the whole), 0.58 of that in the root mean square: five standard deviations.
        assert (got - ref).abs()[finite].le(3 * (x[0, :, 0, 0].numel() * win * win / 4) ** 0.5 * 2.0 ** -24 * size[finite]).all(), kind


@pytest.mark.parametrize("win,N,IC,OC,H,W,split", [
    (5, 1, 128, 128, 17, 17, False),   # few tiles: conv_small and the staged filter
    (5, 9, 32, 32, 50, 56, True),
    (5, 7, 128, 128, 21, 28, True),
    (5, 16, 16, 8, 90, 101, False),    # two steps only
    (7, 2, 128, 128, 32, 32, False),   # one round of the other kernels
    (7, 9, 32, 32, 50, 56, True),
    (7, 7, 64, 64, 43, 35, True),
])
def test_who_takes_it(pkg, win, N, IC, OC, H, W, split):
    others = 3.0 + -(-(-(-N * H * W // 32) * -(-OC // 32)) // 256) * (0.13 if win == 5 else 0.27) * IC
    assert (plan_of(pkg, win, N, IC, OC, H, W, 1, 1, 1, 1, limit=others).strips > 0) is split


def test_seven_by_seven_is_not_dilated(pkg):
    assert plan_of(pkg, 7, 9, 32, 32, 50, 56, 1, 1, 2, 1).strips > 0
    assert plan_of(pkg, 7, 9, 32, 32, 50, 56, 1, 1, 1, 2).strips == 0
