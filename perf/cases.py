"""The work that programs have this library do, as cases that can be timed: one call (or the few calls of one block of a
model) through the package's public functions, on operands that are already on the GPU.

The listed cases are the benchmark configurations, the End2End models and the plans of this repository, from the smallest
call to the largest; draw() gives more of the same kinds over the whole range of sizes, types and options."""
import importlib
import math

import torch

pkg = importlib.import_module("multi-device-model-compiler_amd")

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
ACTS = {"none": pkg.ACT_NONE, "relu": pkg.ACT_RELU, "gelu": pkg.ACT_GELU}


def listed():
    return [
        # The smallest model of the End2End set: MatMul + Add + Relu on [3, 32, 32] rows.  All latency: a few KB of operands.
        dict(name="linear_f32_96x64x32", op="linear", dtype="f32", M=96, N=64, K=32, act="relu", residual=False, packed=False),
        # The elementwise add every residual graph holds, at the benchmark's (3, 640, 640).
        dict(name="add_3x640x640", op="add", n=3 * 640 * 640),
        # LayerNorm of a BERT-base activation in fp32: (32, 128, 768).
        dict(name="layer_norm_f32_4096x768", op="layer_norm", dtype="f32", m=4096, n=768, residual=False),
        # Residual add + LayerNorm between two blocks: a ragged number of tokens and a width that is no whole number of
        # 16-byte vectors.
        dict(name="add_layer_norm_f16_2051x770", op="layer_norm", dtype="f16", m=2051, n=770, residual=True),
        # Attention of a BERT-base encoder over short, full sequences.
        dict(name="attention_f16_b32_s128", op="attention", dtype="f16", B=32, S=128, H=12, D=64, causal=False, lengths="full"),
        # Attention over a padded batch: 256 to 512 valid keys a sequence.
        dict(name="attention_f16_b8_s512_padded", op="attention", dtype="f16", B=8, S=512, H=16, D=64, causal=False, lengths="padded"),
        # Causal prefill with 128-wide heads, in bf16.
        dict(name="attention_bf16_b4_s2048_causal", op="attention", dtype="bf16", B=4, S=2048, H=32, D=128, causal=True, lengths="full"),
        # A BERT-base encoder layer that serves one request of 77 tokens: seven small kernels in a row.
        dict(name="bert_layer_b1_s77", op="bert_layer", B=1, S=77, d=768, heads=12, ffn=3072, lengths="full"),
        # The same layer on the benchmark's batch.
        dict(name="bert_layer_b32_s128", op="bert_layer", B=32, S=128, d=768, heads=12, ffn=3072, lengths="full"),
        # The context (prefill) layer of a decoder, fp32 activations and weights: pre-LN, causal, ReLU.
        dict(name="decoding_layer_b8_s512", op="decoding_layer", B=8, S=512, d=2048, heads=16, ffn=2048, causal=True, act="relu", norm_first=True),
        # The End2End convolution: a network's stem, three channels in, most of the traffic in the output.
        dict(name="conv_16x3x256x256", op="conv", N=16, IC=3, H=256, W=256, OC=64, K=3, stride=1, relu=False, post_add=False),
        # The residual block of plans/resnet_block.plan: conv + ReLU, conv + shortcut + ReLU, 2 x 2 max pool.
        dict(name="resnet_block_4x64x28x28", op="resnet_block", N=4, C=64, H=28, W=28),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["linear", "add", "layer_norm", "attention", "attention", "bert_layer", "decoding_layer", "conv", "resnet_block"])
    while True:
        c = _DRAW[kind](rng)
        w = work(c)
        # no dearer than the decoding layer above (fp32 products run at a sixteenth of the 16-bit rate)
        dear = 16 if c["op"] in ("conv", "resnet_block") or c.get("dtype") == "f32" and c["op"] == "linear" else 1
        if w["flops"] * dear <= 140e9 and w["bytes"] <= 600e6:
            return c


def _draw_linear(rng):
    # any number of tokens; widths of 16-bit layers are multiples of 8, fp32 ones arbitrary
    dtype = rng.choice(["f16", "f16", "bf16", "f32"])
    unit = 1 if dtype == "f32" and rng.random() < 0.5 else 8
    size = lambda low, high: max(unit, _log(rng, low, high) // unit * unit)  # noqa: E731
    act = rng.choice(["none", "relu", "gelu"])
    return dict(op="linear", dtype=dtype, M=_log(rng, 1, 8192), N=size(32, 6144), K=size(32, 4096), act=act,
                residual=act == "none" and rng.random() < 0.5, packed=dtype != "f32" and rng.random() < 0.3)


def _draw_add(rng):
    return dict(op="add", n=_log(rng, 200, 1 << 25))


def _draw_layer_norm(rng):
    n = _log(rng, 64, 8192)
    return dict(op="layer_norm", dtype=rng.choice(["f32", "f16", "bf16"]), m=_log(rng, 16, 16384),
                n=n if rng.random() < 0.3 else n // 8 * 8, residual=rng.random() < 0.5)


def _draw_attention(rng):
    return dict(op="attention", dtype=rng.choice(["f16", "bf16"]), B=_log(rng, 1, 32), S=_log(rng, 16, 4096), H=rng.choice([4, 8, 12, 16, 32]),
                D=rng.choice([32, 40, 64, 64, 64, 80, 128, 128, 128, 256]), causal=rng.random() < 0.5,
                lengths=rng.choice(["full", "padded", "packed"]))


def _draw_bert_layer(rng):
    heads = rng.choice([4, 8, 12, 16])
    return dict(op="bert_layer", B=_log(rng, 1, 32), S=_log(rng, 5, 512), d=64 * heads, heads=heads, ffn=256 * heads,
                lengths=rng.choice(["full", "padded"]))


def _draw_decoding_layer(rng):
    d = rng.choice([512, 768, 1024, 2048])
    return dict(op="decoding_layer", B=_log(rng, 1, 16), S=_log(rng, 16, 1024), d=d, heads=d // rng.choice([64, 128, 256]),
                ffn=d * rng.choice([1, 2, 4]), causal=rng.random() < 0.7, act=rng.choice(["relu", "gelu"]), norm_first=rng.random() < 0.7)


def _draw_conv(rng):
    K = rng.choice([1, 3, 3, 3, 5, 7])
    return dict(op="conv", N=_log(rng, 1, 32), IC=rng.choice([1, 3, 16, 32, 64, 128, 256]), H=_log(rng, 7, 256), W=_log(rng, 7, 256),
                OC=rng.choice([8, 16, 32, 64, 96, 128, 256, 512]), K=K, stride=rng.choice([1, 1, 2]), relu=rng.random() < 0.5,
                post_add=rng.random() < 0.3)


def _draw_resnet_block(rng):
    return dict(op="resnet_block", N=_log(rng, 1, 32), C=rng.choice([16, 32, 64, 128, 256]), H=_log(rng, 7, 56), W=_log(rng, 7, 56))


_DRAW = {"linear": _draw_linear, "add": _draw_add, "layer_norm": _draw_layer_norm, "attention": _draw_attention, "bert_layer": _draw_bert_layer,
         "decoding_layer": _draw_decoding_layer, "conv": _draw_conv, "resnet_block": _draw_resnet_block}


def _lengths(c):
    """Valid tokens of each sequence: all S, or spread evenly over S/2 .. S (the seed only deals them out)."""
    B, S = c["B"], c["S"]
    if c["lengths"] == "full":
        return [S] * B
    low = max(1, S // 2)
    return [low + (S - low) * (i + 1) // B for i in range(B)]


def _conv_out(size, K, stride):
    return (size + 2 * (K // 2) - K) // stride + 1


def prepare(c, seed):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(seed)

    def normal(*shape, std=1.0, mean=0.0, dtype=torch.float32):
        return torch.empty(shape, device=dev).normal_(mean, std, generator=gen).to(dtype)

    op, t = c["op"], DTYPES.get(c.get("dtype"), torch.float16)
    s = {"op": op, "case": c}
    if op == "add":
        s["args"] = [torch.empty(c["n"], device=dev).uniform_(-1, 1, generator=gen) for _ in range(2)]
    elif op == "layer_norm":
        rows = [normal(c["m"], c["n"], dtype=t) for _ in range(2 if c["residual"] else 1)]
        s["args"] = rows + [normal(c["n"], mean=1.0, std=0.02, dtype=t), normal(c["n"], std=0.02, dtype=t)]
    elif op == "linear":
        w = normal(c["K"], c["N"], std=c["K"] ** -0.5, dtype=t)
        s["x"], s["w"] = normal(c["M"], c["K"], dtype=t), pkg.pack_weight(w) if c["packed"] else w
        s["bias"], s["residual"] = normal(c["N"], dtype=t), normal(c["M"], c["N"], dtype=t) if c["residual"] else None
    elif op in ("attention", "bert_layer"):
        lens = torch.tensor(_lengths(c), dtype=torch.int32)[torch.randperm(c["B"], generator=torch.Generator().manual_seed(seed))]
        s["lens"] = lens.to(dev) if c["lengths"] == "padded" else None
        if op == "attention" and c["lengths"] == "packed":
            s["cu"] = torch.cat([torch.zeros(1, dtype=torch.int32), lens.cumsum(0, dtype=torch.int32)]).to(dev)
            s["qkv"] = normal(int(lens.sum()), 3, c["H"], c["D"], dtype=t)
        elif op == "attention":
            s["qkv"] = normal(c["B"], c["S"], 3, c["H"], c["D"], dtype=t)
        else:
            d, f = c["d"], c["ffn"]
            s["x"] = normal(c["B"], c["S"], d, dtype=t)
            s["weights"] = [normal(*shape, std=0.02, mean=mean, dtype=t) for shape, mean in
                            (((d, 3 * d), 0), ((3 * d,), 0), ((d, d), 0), ((d,), 0), ((d,), 1), ((d,), 0), ((d, f), 0), ((f,), 0),
                             ((f, d), 0), ((d,), 0), ((d,), 1), ((d,), 0))]
    elif op == "decoding_layer":
        d, f = c["d"], c["ffn"]
        s["x"] = normal(c["B"], c["S"], d)
        s["weights"] = [normal(*shape, std=0.02) for shape in ((d, 3 * d), (d, d), (d,), (d, f), (f,), (f, d), (d,))]
    elif op == "conv":
        s["x"] = normal(c["N"], c["IC"], c["H"], c["W"])
        s["w"], s["b"] = normal(c["OC"], c["IC"], c["K"], c["K"], std=(c["IC"] * c["K"] ** 2) ** -0.5), normal(c["OC"])
        oh, ow = _conv_out(c["H"], c["K"], c["stride"]), _conv_out(c["W"], c["K"], c["stride"])
        s["post"] = normal(c["N"], c["OC"], oh, ow) if c["post_add"] else None
    elif op == "resnet_block":
        C = c["C"]
        s["x"] = normal(c["N"], C, c["H"], c["W"])
        s["w"], s["b"] = [normal(C, C, 3, 3, std=(9 * C) ** -0.5) for _ in range(2)], [normal(C, std=0.1) for _ in range(2)]
    return s


def run(s):
    op, c = s["op"], s["case"]
    if op == "add":
        return pkg.add(*s["args"])
    if op == "layer_norm":
        return (pkg.add_residual_layer_norm if c["residual"] else pkg.layer_norm)(*s["args"])
    if op == "linear":
        return pkg.matmul_ex(s["x"], s["w"], s["bias"], s["residual"], act=ACTS[c["act"]], kernel="packed" if c["packed"] else "auto")
    if op == "attention":
        if c["lengths"] == "packed":
            return pkg.fused_mha_cu_seqlens(s["qkv"], s["cu"], c["S"], causal=c["causal"])
        return pkg.fused_mha(s["qkv"], s["lens"], causal=c["causal"])
    if op == "bert_layer":
        return pkg.bert_encoder_layer(s["x"], *s["weights"], heads=c["heads"], seqlens=s["lens"])
    if op == "decoding_layer":
        return pkg.decoding_context_layer(s["x"], *s["weights"], heads=c["heads"], causal=c["causal"], relu=c["act"] == "relu",
                                          norm_first=c["norm_first"])
    if op == "conv":
        p = c["K"] // 2
        return pkg.conv2d(s["x"], s["w"], s["b"], s["post"], pad=(p, p, p, p), stride=(c["stride"],) * 2, relu=c["relu"])
    h = pkg.conv2d(s["x"], s["w"][0], s["b"][0], pad=(1, 1, 1, 1), relu=True)
    r = pkg.conv2d(h, s["w"][1], s["b"][1], s["x"], pad=(1, 1, 1, 1), relu=True)
    return r, pkg.pool2d(r, (2, 2), stride=(2, 2))


def _attention_flops(lens, queries, width, causal):
    """Both products over the pairs of one query and one admissible key (half of them under the causal mask)."""
    return 4 * width * sum(n * q if not causal else n * (n + 1) / 2 + n * (q - n) for n, q in zip(lens, queries))


def work(c):
    op, size = c["op"], 4 if c.get("dtype") == "f32" else 2
    if op == "add":
        return {"bytes": 12 * c["n"], "flops": c["n"]}
    if op == "layer_norm":
        return {"bytes": size * (c["m"] * c["n"] * (4 if c["residual"] else 2) + 2 * c["n"]), "flops": 8 * c["m"] * c["n"]}
    if op == "linear":
        M, N, K = c["M"], c["N"], c["K"]
        return {"bytes": size * (M * K + K * N + N + M * N * (2 if c["residual"] else 1)), "flops": 2 * M * N * K}
    if op == "attention":
        lens, width = _lengths(c), c["H"] * c["D"]
        queries = lens if c["lengths"] == "packed" else [c["S"]] * c["B"]
        return {"bytes": 2 * width * sum(2 * q + 2 * n for n, q in zip(lens, queries)), "flops": _attention_flops(lens, queries, width, c["causal"])}
    if op in ("bert_layer", "decoding_layer"):
        d, f, M = c["d"], c["ffn"], c["B"] * c["S"]
        size = 2 if op == "bert_layer" else 4
        lens = _lengths(c) if op == "bert_layer" else [c["S"]] * c["B"]
        weights = 4 * d * d + 2 * d * f
        return {"bytes": size * (2 * M * d + weights + 2 * d + f), "flops": 2 * M * weights + _attention_flops(lens, [c["S"]] * c["B"], d, c.get("causal", False))}
    if op == "conv":
        oh, ow = _conv_out(c["H"], c["K"], c["stride"]), _conv_out(c["W"], c["K"], c["stride"])
        y, k = c["N"] * c["OC"] * oh * ow, c["IC"] * c["K"] ** 2
        return {"bytes": 4 * (c["N"] * c["IC"] * c["H"] * c["W"] + c["OC"] * (k + 1) + y * (2 if c["post_add"] else 1)), "flops": 2 * y * k}
    y, k = c["N"] * c["C"] * c["H"] * c["W"], 9 * c["C"]
    return {"bytes": 4 * (2 * y + y // 4 + 2 * c["C"] * (k + 1)), "flops": 4 * y * k}


def tolerance(c):
    """What another correct implementation at the same precision shows: one rounding of the stored type for single
    operations, the roundings of the stored intermediates for the layers."""
    op, dtype = c["op"], c.get("dtype")
    if op == "add":
        return "exact"
    if op in ("conv", "resnet_block") or dtype == "f32":
        return {"rel": 1e-5}
    if op in ("bert_layer", "decoding_layer"):
        return {"rel": 4e-3}
    return {"rel": 6e-3 if dtype == "bf16" else 1e-3}
