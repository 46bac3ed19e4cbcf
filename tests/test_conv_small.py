"""Convolution on tiles of 16 pixels (csrc/kernels/conv_small.hip): the rule (no GPU: it is asked, for 256 compute units) and the kernel
where its tiles, shares and windows end."""
import ctypes

import numpy as np
import pytest

from conftest import to_dev
from test_index_bounds import internal


class Plan(ctypes.Structure):
    _fields_ = [("oc_side", ctypes.c_int), ("us", ctypes.c_double)]


@pytest.mark.parametrize("win,pixels,IC,OC,side", [
    (3, 16 * 16, 64, 256, 16),       # a tile of 16 x 16 a CU
    (3, 16 * 16 + 1, 64, 256, 32),   # a tile more: halves in one round
    (3, 16 * 16, 64, 257, 32),
    (3, 32 * 16, 64, 256, 32),
    (3, 32 * 16 + 1, 128, 256, 32),  # two rounds of halves
    (3, 64 * 16, 128, 256, 32),
    (3, 64 * 16 + 1, 128, 256, 0),   # a third: the tiles of 32 x 32 fill the chip as well
    (5, 300, 64, 256, 32),
    (7, 300, 64, 256, 16),           # no halves of it
    (7, 300, 62, 256, 0),
])
def test_tile(pkg, win, pixels, IC, OC, side):
    plan = internal(pkg, "_ZN4mgpu13convSmallPlanEillll", Plan, ctypes.c_int, *[ctypes.c_int64] * 4)(win, pixels, IC, OC, 256)
    assert plan.oc_side == side


@pytest.mark.parametrize("win,pixels,IC,OC,few", [
    (3, 200 * 32, 64, 32, True),     # 200 tiles, eight wavefronts each
    (3, 400 * 32, 128, 32, True),
    (3, 400 * 32 + 1, 128, 64, False),
    (5, 256 * 32, 32, 32, True),
    (5, 257 * 32, 32, 32, False),    # four wavefronts a tile
    (7, 256 * 32, 16, 32, True),
])
def test_few_tiles(pkg, win, pixels, IC, OC, few):
    time = internal(pkg, "_ZN4mgpu16convFewTilesTimeEillllll", ctypes.c_double, ctypes.c_int, *[ctypes.c_int64] * 6)
    assert (time(win, 1, pixels, IC, OC, 32, 256) > 0) is few


SHAPES = [  # N, IC, H, W, OC, pad (top, left, bottom, right), stride, dilation
    (1, 4, 7, 7, 8, (0, 0, 0, 0), (1, 1), (1, 1)),        # one channel group: seven shares without one; fewer channels than a tile
    (3, 36, 5, 6, 17, (1, 1, 1, 1), (1, 1), (1, 1)),      # nine groups on eight wavefronts, a channel beyond a tile, images end in a tile
    (11, 64, 2, 1, 48, (3, 2, 3, 2), (1, 1), (1, 1)),     # images smaller than the window, many in a tile
    (2, 100, 13, 9, 31, (2, 0, 1, 3), (2, 1), (1, 1)),
    (2, 32, 17, 15, 40, (3, 3, 3, 3), (1, 2), (2, 1)),
    (1, 128, 16, 16, 33, (1, 2, 2, 1), (1, 1), (1, 2)),   # whole tiles of pixels
]


def small_conv(pkg, side, x, w, b, add, pad, stride, dilation, relu):
    import torch
    (N, IC, H, W), (OC, _, win, _) = x.shape, w.shape
    OH, OW = ((s + pad[i] + pad[i + 2] - (win - 1) * dilation[i] - 1) // stride[i] + 1 for i, s in enumerate((H, W)))
    pkg.ops()
    launch = internal(pkg, "_ZN4mgpu9convSmallEiiPKfS1_S1_PfS1_lllllllllllllbP12ihipStream_t", ctypes.c_bool, ctypes.c_int, ctypes.c_int,
                      *[ctypes.c_void_p] * 5, *[ctypes.c_int64] * 13, ctypes.c_bool, ctypes.c_void_p)
    count = N * OC * OH * OW
    out = torch.full((count + 64,), 7.0, device=x.device)  # 32 elements before and behind
    assert launch(win, side, x.data_ptr(), w.data_ptr(), b.data_ptr(), out[32:].data_ptr(), add.data_ptr() if add is not None else None, N, IC, H, W, OC,
                  OH, OW, pad[0], pad[1], *stride, *dilation, relu, torch.cuda.current_stream().cuda_stream)
    assert torch.all(out[:32] == 7) and torch.all(out[32 + count:] == 7)
    return out[32:32 + count].view(N, OC, OH, OW)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("win,side", [(3, 16), (3, 32), (5, 16), (5, 32), (7, 16)])
def test_edges(pkg, gpu, oracle, shape, win, side):
    N, IC, H, W, OC, pad, stride, dilation = shape
    OH, OW = ((s + pad[i] + pad[i + 2] - (win - 1) * dilation[i] - 1) // stride[i] + 1 for i, s in enumerate((H, W)))
    if OH < 1 or OW < 1: pytest.skip("no such window in it")
    rng = np.random.Generator(np.random.PCG64(IC + win))
    x, w = rng.standard_normal((N, IC, H, W)).astype(np.float32), (rng.standard_normal((OC, IC, win, win)) * (IC * win * win) ** -0.5).astype(np.float32)
    b, a = rng.standard_normal(OC).astype(np.float32), rng.standard_normal((N, OC, OH, OW)).astype(np.float32)
    tx, tw, tb, ta = (to_dev(t, gpu) for t in (x, w, b, a))
    for add, relu in ((None, False), (a, True)):
        got = small_conv(pkg, side, tx, tw, tb, ta if add is not None else None, pad, stride, dilation, relu).cpu().numpy()
        ref = oracle.conv2d(x, w, b, add, pad, stride, dilation, relu)
        # both sides are a sum of K products of fp32 accuracy: 2^-24 of the sum of their sizes (here about 1) times some sqrt(K)
        assert np.all(np.abs(got - ref) <= 1e-5 * (1 + np.abs(ref))), np.abs(got - ref).max()


@pytest.mark.gpu
@pytest.mark.parametrize("win,side", [(3, 16), (3, 32), (5, 16), (5, 32), (7, 16)])
def test_infinities_and_nan(pkg, gpu, win, side):
    import torch
    gen = torch.Generator(device=gpu).manual_seed(win)
    x, w = (torch.randint(1, 4, s, device=gpu, generator=gen).float() for s in ((2, 36, 9, 11), (33, 36, win, win)))  # (sums are whole numbers below 2^24)
    x[0, 3, 1, 1], x[0, 35, 8, 10], x[1, 17, 4, 4], w[5, 0, 0, 0], w[32, 30, win - 1, win - 1] = (float(v) for v in ("inf", "nan", "-inf", "inf", "-inf"))
    p = win // 2
    got = small_conv(pkg, side, x, w, torch.zeros(33, device=gpu), None, (p, p, p, p), (1, 1), (1, 1), False)
    ref = torch.nn.functional.conv2d(x.double().cpu(), w.double().cpu(), padding=p).float().to(gpu)
    # (outside the image a tap is 0, which an infinite filter value makes a NaN in either)
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got[~ref.isnan()], ref[~ref.isnan()])
    assert ref.isnan().any() and ref.isinf().any() and ref.isfinite().any()
