"""Head sizes on either side of the lines between the attention kernels' instances, which leave out the matrix steps that hold nothing
but filler: every kernel, both masks."""
import numpy as np
import pytest

from conftest import to_dev
from test_gpu_fmha import TOL_BF16, TOL_F16, excess

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [16, 24, 32, 40, 48, 56, 72, 80, 88, 96, 104, 136, 152, 160, 168])
@pytest.mark.parametrize("B,S,H,lens", [
    (33, 70, 8, None),          # blocks of 128 queries, a tile and a bit of keys
    (20, 64, 16, None),         # one tile
    (1, 230, 3, [201]),         # few queries: the wavefronts split the keys
    (1, 520, 25, None),         # two groups of queries a block
    (3, 600, 14, [600, 1, 77]), # two sets of wavefronts
])
def test_head_sizes_around_the_instances(pkg, gpu, oracle, D, B, S, H, lens):
    import torch
    rng = np.random.Generator(np.random.PCG64(D * 1000 + S))
    bf16 = D % 16 == 8
    qkv = torch.from_numpy(rng.standard_normal((B, S, 3, H, D)).astype(np.float32)).to(gpu).to(torch.bfloat16 if bf16 else torch.float16)
    # (unit variance throughout, as the tolerances ask for: with values twice as large in bf16 an output near 0 is the difference of
    # terms up to 8, each off by the 2^-9 of its rounded weight: 0.016, twice the bound)
    tl = to_dev(np.asarray(lens, np.int32), gpu) if lens is not None else None
    pick = rng.choice(B, min(B, 2), replace=False)  # (sequences are independent of each other; and so are heads)
    heads = rng.choice(H, min(H, 2), replace=False)
    part = qkv[torch.as_tensor(pick, device=gpu)][:, :, :, torch.as_tensor(heads, device=gpu)].contiguous()
    bits = part.view(torch.int16).cpu().numpy().view(np.uint16)
    for causal in (False, True):
        out = torch.full((B * S + 1, H * D), 7.0, dtype=qkv.dtype, device=gpu)  # a guard row behind the output
        pkg.fused_mha(qkv, tl, causal=causal, out=out[:B * S].view(B, S, H * D))
        got = out.float().cpu().numpy()
        assert np.all(got[B * S] == 7.0)
        ref = oracle.fmha(bits if bf16 else bits.view(np.float16), None if lens is None else [lens[b] for b in pick], causal=causal, bf16=bf16)
        mine = got[:B * S].reshape(B, S, H, D)[pick][:, :, heads].reshape(len(pick), S, -1)
        assert excess(mine, ref, TOL_BF16 if bf16 else TOL_F16) <= 1.0, (causal, heads)
