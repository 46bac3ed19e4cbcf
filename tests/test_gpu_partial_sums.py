"""Layers whose products before a LayerNorm (or before the fp32 result) are split over blocks and added up by the next
kernel (csrc/kernels/partial_sums.hip): few tokens in 32-row tiles, some more in ragged 128-row tiles, three and four parts,
rows of one, two and four vectors per lane."""
import numpy as np
import pytest

from conftest import to_dev

pytestmark = pytest.mark.gpu


def close(got, ref):
    # fp16 intermediates of seven kernels, outputs of unit variance: the layers' bound in the other tests
    err = np.abs(got - ref)
    assert np.isfinite(got).all() and np.all(err <= 2e-2 + 2e-2 * np.abs(ref)), err.max()


@pytest.mark.parametrize("B,S,d,ffn,lens", [
    (1, 77, 768, 3072, None),         # 32 x 32 tiles, three parts
    (1, 1, 512, 4096, None),          # one token, one vector per lane
    (9, 152, 768, 3072, None),        # 128-row tiles cut at row 1368, three parts
    (2, 30, 1032, 4104, [30, 11]),    # widths that are no multiple of a tile, four vectors per lane, K no multiple of 32
])
def test_bert_layer(pkg, gpu, oracle, rng, B, S, d, ffn, lens):
    H = {768: 12, 512: 8, 1032: 43}[d]
    f = lambda *s: (0.03 * rng.standard_normal(s)).astype(np.float16)
    x = rng.standard_normal((B, S, d)).astype(np.float16)
    W = [f(d, 3 * d), f(3 * d), f(d, d), f(d), 1 + f(d), f(d), f(d, ffn), f(ffn), f(ffn, d), f(d), 1 + f(d), f(d)]
    dev = [to_dev(w, gpu) for w in W]
    tl = to_dev(np.asarray(lens, np.int32), gpu) if lens else None
    got = pkg.bert_encoder_layer(to_dev(x, gpu), *dev, heads=H, seqlens=tl).float().cpu().numpy()
    rows = min(B, 2)  # sequences are independent of each other
    pick = list(range(rows - 1)) + [B - 1]  # the last one among them
    close(got[pick], oracle.bert_layer_f16(x[pick], *W, heads=H, seqlens=[lens[i] for i in pick] if lens else None))


@pytest.mark.parametrize("B,S,d,ffn,norm_first", [
    (1, 30, 768, 3072, True),    # the fp32 result straight from the sums
    (1, 30, 768, 3072, False),
    (3, 20, 1024, 4096, False),
    (1, 5, 2048, 2048, True),    # both products split, the rounded sum kept as the next residual
])
def test_decoding_layer(pkg, gpu, oracle, rng, B, S, d, ffn, norm_first):
    f = lambda *s: (0.03 * rng.standard_normal(s)).astype(np.float32)
    x = rng.standard_normal((B, S, d)).astype(np.float32)
    W = [f(d, 3 * d), f(d, d), f(d), f(d, ffn), f(ffn), f(ffn, d), f(d)]
    got = pkg.decoding_context_layer(to_dev(x, gpu), *[to_dev(w, gpu) for w in W], heads=d // 64, norm_first=norm_first).cpu().numpy()
    close(got[-1:], oracle.decoding_context_layer(x[-1:], *W, heads=d // 64, norm_first=norm_first))
