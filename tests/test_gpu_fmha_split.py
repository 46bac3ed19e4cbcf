"""The attention kernel whose wavefronts split the keys (csrc/kernels/fmha_split.hip), at the sizes where its tiles of 32
keys, its query groups and its merge can go wrong, against the oracle.  Bounds as in test_gpu_fmha.py: one rounding of
the output type on values below 1, relative above."""
import numpy as np
import pytest

from conftest import to_dev

pytestmark = pytest.mark.gpu

TOL = {"f16": 2e-3, "bf16": 8e-3}


def groups(D, B, S, H, causal, cus):
    """The launcher's rule: query groups of 32 a block, 0 for the 128-query kernel."""
    g = 64 if D <= 64 else 128 if D <= 128 else 256
    from1 = 65 if g == 256 or causal else 129 if g == 128 else 193
    from2 = (65 if causal else 321) if g == 64 else 257 if g == 128 and not causal else 193
    if B * H * -(-S // 32) <= cus:
        return int(S >= from1)
    blocks2 = B * H * -(-S // 64)
    if blocks2 <= cus:
        return 2 if S >= from2 else 0
    return 2 if causal and S >= 2048 and blocks2 <= 2 * cus else 0


@pytest.mark.parametrize("D,B,S,H,lens,causal,dtype,expected", [
    (64, 1, 193, 2, None, False, "f16", 1),            # the shortest unmasked; seven tiles, a wavefront without one
    (64, 2, 257, 14, [257, 129], False, "bf16", 1),    # nine tiles, as many blocks as still fit one round
    (64, 1, 321, 2, None, False, "f16", 1),            # eleven tiles over eight wavefronts
    (64, 2, 500, 4, [500, 1], False, "bf16", 1),       # a sequence of one key: seven wavefronts without a tile
    (64, 3, 1100, 2, [1100, 0, 545], False, "f16", 1), # an empty sequence, more tiles than the rings hold
    (64, 1, 65, 3, None, True, "f16", 1),
    (64, 1, 300, 4, [170], True, "bf16", 1),
    (64, 2, 384, 16, [384, 200], False, "f16", 2),     # two groups of four key shares
    (64, 5, 100, 16, [100, 99, 1, 64, 65], True, "f16", 2),
    (64, 1, 2048, 9, None, True, "f16", 2),            # the second round of a long causal launch
    (40, 1, 333, 3, [290], False, "f16", 1),           # a head size padded into the geometry
    (128, 1, 129, 2, None, False, "f16", 1),           # one tile in flight per wavefront
    (128, 1, 515, 2, [260], True, "bf16", 1),
    (128, 4, 257, 12, [257, 256, 30, 100], False, "f16", 2),
    (80, 2, 193, 30, [193, 40], True, "f16", 2),
    (256, 1, 65, 2, None, False, "f16", 1),
    (256, 2, 300, 3, [300, 131], True, "f16", 1),
    (256, 3, 195, 16, [195, 194, 33], False, "bf16", 2),
    (144, 1, 210, 2, None, True, "f16", 1),
])
def test_split_keys(pkg, gpu, oracle, D, B, S, H, lens, causal, dtype, expected):
    import torch
    assert groups(D, B, S, H, causal, torch.cuda.get_device_properties(gpu).multi_processor_count) == expected
    rng = np.random.Generator(np.random.PCG64(D * 10000 + S))
    tq = torch.from_numpy(rng.standard_normal((B, S, 3, H, D)).astype(np.float32)).to(gpu)
    tq = tq.to(torch.float16 if dtype == "f16" else torch.bfloat16)
    bits = tq.view(torch.int16).cpu().numpy().view(np.uint16)
    ref = oracle.fmha(bits if dtype == "bf16" else bits.view(np.float16), lens, causal=causal, bf16=dtype == "bf16")

    def check(got, want):
        bound = TOL[dtype] * np.maximum(1.0, np.abs(want))
        assert np.isfinite(got).all() and (np.abs(got - want) <= bound).all()

    if lens is not None:  # keys beyond a sequence may hold anything
        for b, n in enumerate(lens):
            tq[b, n:, 1:] = float("nan")
    tl = to_dev(np.asarray(lens, np.int32), gpu) if lens is not None else None
    check(pkg.fused_mha(tq, tl, causal=causal).float().cpu().numpy(), ref)
    # the same sequences packed back to back, a guard row behind them
    rows = lens if lens is not None else [S] * B
    cu = np.concatenate([[0], np.cumsum(rows)]).astype(np.int32)
    packed = torch.cat([tq[b, :n] for b, n in enumerate(rows)]).contiguous()
    out = torch.full((int(cu[-1]) + 1, H * D), 7.0, dtype=tq.dtype, device=gpu)
    pkg.fused_mha_cu_seqlens(packed, to_dev(cu, gpu), S, causal=causal, out=out[:int(cu[-1])])
    got = out.float().cpu().numpy()
    assert np.all(got[-1] == 7.0)
    for b, n in enumerate(rows):
        check(got[cu[b]:cu[b + 1]], ref[b, :n])


@pytest.mark.parametrize("D", [64, 128, 256])
def test_split_keys_with_references_far_apart(pkg, gpu, oracle, D):
    """Logits from -60 D^-1/2 8 to +60 D^-1/2 8 along the keys: every wavefront of a block ends with another reference
    maximum, most of them with sums that vanish in the merge."""
    rng = np.random.Generator(np.random.PCG64(D))
    B, S, H = 1, 420, 2
    qkv = (rng.standard_normal((B, S, 3, H, D)) * 0.5).astype(np.float16)
    for ramp in (np.linspace(-60, 60, S), np.linspace(60, -60, S), np.full(S, -60.0)):
        qkv[:, :, 0, :, :] = 0
        qkv[:, :, 0, :, 0] = 8.0
        qkv[:, :, 1, :, 0] = ramp.astype(np.float16)[None, :, None]
        for causal in (False, True):
            got = pkg.fused_mha(to_dev(qkv, gpu), causal=causal).float().cpu().numpy()
            ref = oracle.fmha(qkv, causal=causal)
            assert np.isfinite(got).all() and (np.abs(got - ref) <= TOL["f16"] * np.maximum(1.0, np.abs(ref))).all()


def two_sets(D, B, S, H, causal, cus):
    """The launcher's rule for two sets of wavefronts over the same 128 queries, each with every other tile of keys."""
    if groups(D, B, S, H, causal, cus):
        return False
    nqb = -(-S // 128)
    if causal:
        return S >= 512 and 2 * B * H * nqb <= cus * (4 if nqb >= 12 else 3 if nqb >= 8 else 2)
    return S >= (768 if D > 128 else 512) and B * H * nqb <= cus


@pytest.mark.parametrize("D,B,S,H,lens,causal,dtype", [
    (64, 2, 520, 15, None, False, "f16"),           # nine tiles of 64 keys: the second set has one fewer, the last tile is cut
    (64, 2, 577, 15, [577, 64], False, "bf16"),     # one tile: nothing for the second set
    (40, 2, 640, 16, [640, 65], False, "f16"),      # ten whole tiles; two, the second of one key
    (128, 3, 640, 10, [640, 0, 129], False, "f16"), # an empty sequence
    (80, 2, 600, 14, [600, 1], True, "bf16"),
    (64, 2, 1100, 16, None, True, "f16"),           # more than a round, longest blocks first
    (64, 1, 1540, 20, None, True, "bf16"),
    (256, 2, 800, 11, [800, 33], False, "f16"),     # tiles of 32
    (144, 2, 520, 15, None, True, "f16"),
])
def test_two_sets(pkg, gpu, oracle, D, B, S, H, lens, causal, dtype):
    import torch
    assert two_sets(D, B, S, H, causal, torch.cuda.get_device_properties(gpu).multi_processor_count)
    test_split_keys(pkg, gpu, oracle, D, B, S, H, lens, causal, dtype, 0)


@pytest.mark.parametrize("D", [64, 128, 256])
def test_two_sets_with_references_far_apart(pkg, gpu, oracle, D):
    """Logits that differ by 960 D^-1/2 between the sets' tiles, along the keys and alternating with them."""
    rng = np.random.Generator(np.random.PCG64(D))
    B, S, H = 2, 790, 11
    tile = np.arange(S) // (32 if D == 256 else 64) % 2
    qkv = (rng.standard_normal((B, S, 3, H, D)) * 0.5).astype(np.float16)
    for ramp in (np.linspace(-60, 60, S), np.linspace(60, -60, S), 120.0 * tile - 60, 60 - 120.0 * tile, np.full(S, -60.0)):
        qkv[:, :, 0, :, :] = 0
        qkv[:, :, 0, :, 0] = 8.0
        qkv[:, :, 1, :, 0] = ramp.astype(np.float16)[None, :, None]
        for causal in (False, True):
            got = pkg.fused_mha(to_dev(qkv, gpu), causal=causal).float().cpu().numpy()
            ref = oracle.fmha(qkv, causal=causal)
            assert np.isfinite(got).all() and (np.abs(got - ref) <= TOL["f16"] * np.maximum(1.0, np.abs(ref))).all()
