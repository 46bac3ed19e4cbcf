"""The tensor functions take the native call where they can and ctypes otherwise (a stream named, an operand off the
ordinary case): both ways give the same bits, and what the native call declines is still checked and reported."""
import pytest

pytestmark = pytest.mark.gpu


def _calls(pkg, torch, dev, dtype):
    r = lambda *s, t=dtype: torch.randn(s, device=dev).to(t)  # noqa: E731
    f, h = torch.float32, torch.float16
    qkv, lens = r(2, 40, 3, 2, 64), torch.tensor([40, 17], dtype=torch.int32, device=dev)
    cu = torch.tensor([0, 13, 40], dtype=torch.int32, device=dev)
    x, g, b = r(33, 72), r(72), r(72)
    w, bias, res = r(72, 40), r(40), r(33, 40)
    img, filt, ob = r(2, 3, 9, 11, t=f), r(5, 3, 3, 3, t=f), r(5, t=f)
    d = 128
    bert = [r(*s, t=h) * 0.05 for s in ((d, 3 * d), (3 * d,), (d, d), (d,), (d,), (d,), (d, 2 * d), (2 * d,), (2 * d, d), (d,), (d,), (d,))]
    dec = [r(*s, t=f) * 0.05 for s in ((d, 3 * d), (d, d), (d,), (d, 2 * d), (2 * d,), (2 * d, d), (d,))]
    act, act32 = r(2, 16, d, t=h), r(2, 16, d, t=f)
    return [lambda **k: pkg.add(img, img, **k), lambda **k: pkg.layer_norm(x, g, b, **k),
            lambda **k: pkg.add_residual_layer_norm(x, x, g, b, **k), lambda **k: pkg.cast_layer_norm(x.float(), g.half(), b.half(), **k),
            lambda **k: pkg.fused_mha(qkv, lens, causal=True, **k), lambda **k: pkg.fused_mha_cu_seqlens(qkv.reshape(80, 3, 2, 64)[:40], cu, 27, **k),
            lambda **k: pkg.cast_f32_to_f16(img, **k), lambda **k: pkg.cast_f16_to_f32(act, **k), lambda **k: pkg.cast_f32_to_bf16(img, **k),
            lambda **k: pkg.cast_bf16_to_f32(img.to(torch.bfloat16), **k), lambda **k: pkg.qkv_bias_transpose(qkv.clone(), r(3, 2, 64) * 0, **k),
            lambda **k: pkg.matmul_ex(x, w, bias, res, **k), lambda **k: pkg.matmul_ex(x, pkg.pack_weight(w), bias, act=1, kernel="packed", **k),
            lambda **k: pkg.conv2d(img, filt, ob, pad=(1, 0, 2, 1), stride=(2, 1), relu=True, **k), lambda **k: pkg.pool2d(img, (3, 2), (1, 0, 1, 0), (2, 2), "avg", **k),
            lambda **k: pkg.bert_encoder_layer(act, *bert, heads=2, seqlens=torch.tensor([16, 9], dtype=torch.int32, device=dev), **k),
            lambda **k: pkg.decoding_context_layer(act32, *dec, heads=2, norm_first=False, **k)]


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
def test_native_and_ctypes_calls_agree(pkg, gpu, dtype):
    import torch
    for i, call in enumerate(_calls(pkg, torch, gpu, getattr(torch, dtype))):
        native, plain = call(), call(stream=torch.cuda.current_stream())
        for p, q in zip(native if isinstance(native, tuple) else (native,), plain if isinstance(plain, tuple) else (plain,)):
            assert p.shape == q.shape and p.dtype == q.dtype and torch.equal(p, q), i


def test_declined_operands_are_reported_as_before(pkg, gpu):
    import torch
    a = torch.randn(6, 8, device=gpu)
    with pytest.raises(pkg.MgpuError):
        pkg.add(a, a.cpu())
    with pytest.raises(pkg.MgpuError):
        pkg.add(a.t(), a.t())
    with pytest.raises(AssertionError):
        pkg.add(a, a[:3])
    with pytest.raises(pkg.MgpuError):  # the library's own rejection, through the native call
        pkg.fused_mha(torch.zeros(1, 4, 3, 1, 12, dtype=torch.float16, device=gpu))
    out = torch.empty_like(a)
    assert pkg.add(a, a, out) is out and torch.equal(out, a + a)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):  # the native call enqueues on the caller's current stream
        b = pkg.add(a, a)
    side.synchronize()
    assert torch.equal(b, a + a)
