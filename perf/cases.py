"""The work a user of this package has it do, as cases that can be prepared, run and compared.

Every case goes through the package's public entry points the way a program that runs a diffusion transformer does:
modules and composite operators for the linears, the operator pair for programs that bring their own modules, attention,
the adaLN and text-encoder projections, and a whole forward pass of the FLUX.1-shaped transformer.
"""

import math

import torch

from nunchaku_rocm_amd import ops
from nunchaku_rocm_amd.flux_shaped import FluxShapedConfig, FluxShapedTransformer, flux_ids, rope_table
from nunchaku_rocm_amd.linear import AWQW4A16Linear, SVDQW4A4Linear

DEVICE = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    return [
        # one adaLN modulation projection of one image: the smallest call a model makes, one vector against a 4-bit weight
        {"name": "modulation", "kind": "modulation", "dtype": "bf16", "rows": 1, "k": 3072, "n": 18432},
        # the text stream's output projection: 512 prompt tokens, a fraction of the chip
        {"name": "linear-text", "kind": "linear", "dtype": "bf16", "tokens": 512, "k": 3072, "n": 3072, "rank": 32},
        # quantizer and GEMM called as operators on the packed (M, K/2) matrix, as the reference's own modules call them
        {"name": "operators", "kind": "operators", "dtype": "fp16", "tokens": 1536, "k": 3072, "n": 3072, "rank": 32},
        # joint QKV projection with LayerNorm + modulate in front and Q/K RMSNorm + RoPE behind it, 1024 x 1024 pixels
        {"name": "qkv-image", "kind": "qkv", "dtype": "bf16", "tokens": 4608, "k": 3072, "heads": 24, "rank": 32},
        # the same for a small image of odd size in fp16, with a LoRA attached (its rank adds to the low-rank branch's)
        {"name": "qkv-ragged", "kind": "qkv", "dtype": "fp16", "tokens": 1201, "k": 3072, "heads": 24, "rank": 64},
        # feed-forward of the image stream (GELU and requantization between the two GEMMs)
        {"name": "mlp-image", "kind": "mlp", "dtype": "bf16", "tokens": 4608, "k": 3072, "hidden": 12288, "rank": 32},
        # feed-forward of the text stream for a prompt of odd length
        {"name": "mlp-text", "kind": "mlp", "dtype": "bf16", "tokens": 333, "k": 3072, "hidden": 12288, "rank": 32},
        # gated feed-forward (SwiGLU and requantization between the two GEMMs)
        {"name": "swiglu", "kind": "swiglu", "dtype": "fp16", "tokens": 2048, "k": 3072, "hidden": 8192, "rank": 32},
        # joint attention of one block at 1024 x 1024 pixels on the strided views of the QKV projection
        {"name": "attention-joint", "kind": "attention", "dtype": "bf16", "batch": 1, "heads": 24, "q": 4608, "kv": 4608, "d": 128},
        # cross attention of a UNet to 77 prompt tokens, two images (or the two halves of guidance) at once
        {"name": "attention-cross", "kind": "attention", "dtype": "fp16", "batch": 2, "heads": 10, "q": 4096, "kv": 77, "d": 64},
        # one linear of a 4-bit text encoder over 512 prompt tokens
        {"name": "encoder-linear", "kind": "encoder", "dtype": "bf16", "tokens": 512, "k": 4096, "n": 10240, "group": 128},
        # a forward pass of the transformer at 1024 x 1024 pixels: embedders, modulations, one dual-stream and two
        # single-stream blocks (the model's own ratio), output layer
        {"name": "transformer", "kind": "transformer", "dtype": "bf16", "grid_h": 64, "grid_w": 64, "text": 512, "double": 1, "single": 2},
    ]


def _tokens(rng, lo, hi):
    """Token counts spread over their logarithm: multiples of 64 (latent grids, padded prompts) and odd ones."""
    t = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, t // 64 * 64) if t >= 128 and rng.random() < 0.4 else t


def draw(rng):
    kind = rng.choice(("modulation", "linear", "operators", "qkv", "qkv", "mlp", "mlp", "swiglu", "attention", "attention", "encoder", "transformer"))
    c = {"kind": kind, "dtype": rng.choice(("bf16", "bf16", "fp16"))}
    width = rng.choice((1536, 1920, 2048, 3072, 3072, 3072, 3584))
    rank = rng.choice((32, 32, 32, 48, 64, 128))
    if kind == "modulation":
        c.update(rows=rng.choice((1, 1, 2, 3, 4, 6, 8)), k=width, n=width * rng.choice((2, 3, 6)))
    elif kind in ("linear", "operators"):
        c.update(tokens=_tokens(rng, 64, 8704), k=width, n=width * rng.choice((1, 1, 3)), rank=rank)
    elif kind == "qkv":
        c.update(tokens=_tokens(rng, 64, 8704), k=width, heads=width // 128, rank=rank)
    elif kind == "mlp":
        c.update(tokens=_tokens(rng, 64, 8704), k=width, hidden=4 * width, rank=rank)
    elif kind == "swiglu":
        c.update(tokens=_tokens(rng, 64, 8704), k=width, hidden=rng.choice((2 * width, 8192)), rank=rank)
    elif kind == "attention":
        d, q = rng.choice((128, 128, 64)), _tokens(rng, 64, 8704)
        kv = q if rng.random() < 0.7 else rng.choice((77, 154, 256, 512))
        c.update(batch=rng.choice((1, 1, 2)), heads=rng.choice((8, 10, 16, 20, 24)), q=q, kv=kv, d=d)
    elif kind == "encoder":
        c.update(tokens=rng.choice((77, 128, 256, 333, 512)) * rng.choice((1, 1, 2)), k=4096, n=rng.choice((4096, 10240)), group=rng.choice((64, 128)))
    else:
        c.update(grid_h=rng.randint(16, 64), grid_w=rng.randint(16, 64), text=rng.choice((77, 128, 256, 333, 512)), double=1, single=rng.choice((1, 2)))
    return c


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _normal(g, *shape, scale=1.0, dtype):
    return (torch.randn(*shape, device=DEVICE, generator=g) * scale).to(dtype)


def _uniform(g, *shape, lo, hi, dtype):
    return (torch.rand(*shape, device=DEVICE, generator=g) * (hi - lo) + lo).to(dtype)


def _activations(g, rows, k, dtype):
    """Hidden states as the benchmark draws them: N(0, 1) with 1 % of the channels twenty times as large."""
    x = torch.randn(rows, k, device=DEVICE, generator=g)
    x[:, torch.randperm(k, device=DEVICE, generator=g)[: max(1, k // 100)]] *= 20.0
    return x.to(dtype)[None]


def _svdq(g, k, n, rank, dtype, unsigned=False):
    lin = SVDQW4A4Linear(k, n, rank=rank, act_unsigned=unsigned, torch_dtype=dtype, device=DEVICE)
    with torch.no_grad():
        lin.qweight.copy_(torch.randint(0, 256, lin.qweight.shape, device=DEVICE, generator=g, dtype=torch.uint8).view(torch.int8))
        lin.wscales.copy_(_uniform(g, k // 64, n, lo=0.005, hi=0.02, dtype=dtype))
        lin.smooth_factor.copy_(_uniform(g, k, lo=0.5, hi=4.0, dtype=dtype))
        lin.proj_down.copy_(_normal(g, k, rank, scale=0.02, dtype=dtype))
        lin.proj_up.copy_(_normal(g, n, rank, scale=0.02, dtype=dtype))
        lin.bias.copy_(_normal(g, n, scale=0.01, dtype=dtype))
    return lin.requires_grad_(False)


def _awq(g, k, n, group, dtype):
    lin = AWQW4A16Linear(k, n, group_size=group, torch_dtype=dtype, device=DEVICE)
    with torch.no_grad():
        lin.qweight.copy_(torch.randint(-(2**31), 2**31 - 1, lin.qweight.shape, device=DEVICE, generator=g))
        scales = _uniform(g, k // group, n, lo=0.005, hi=0.02, dtype=dtype)
        lin.wscales.copy_(scales)
        lin.wzeros.copy_(-torch.randint(0, 16, scales.shape, device=DEVICE, generator=g) * scales.float())
        lin.bias.copy_(_normal(g, n, scale=0.01, dtype=dtype))
    return lin.requires_grad_(False)


def _norm_weight(g, dtype):
    norm = torch.nn.RMSNorm(128, eps=1e-6, device=DEVICE, dtype=dtype)
    norm.weight.data.copy_(_uniform(g, 128, lo=0.5, hi=1.5, dtype=dtype))
    return norm.requires_grad_(False)


def prepare(case, seed):
    """A model's weights with their working copies made (by a pass over a few other rows, as a program's earlier steps have
    done), and the inputs of the next call."""
    g, dtype, kind = _generator(seed), DTYPES[case["dtype"]], case["kind"]
    s = {"kind": kind}
    if kind == "modulation":
        s["lin"] = _awq(g, case["k"], case["n"], 64, dtype)
        s["x"] = torch.nn.functional.silu(_normal(g, case["rows"], case["k"], dtype=dtype))
    elif kind == "linear":
        s["lin"] = _svdq(g, case["k"], case["n"], case["rank"], dtype)
        s["x"] = _activations(g, case["tokens"], case["k"], dtype)
        s["lin"](s["x"][:, :1] * 0.5)
    elif kind == "operators":
        k, n, rank, tokens = case["k"], case["n"], case["rank"], case["tokens"]
        padded = -(-tokens // 256) * 256
        s["lin"] = _svdq(g, k, n, rank, dtype)
        s["x"] = _activations(g, tokens, k, dtype)[0]
        # buffers the program keeps; rows past the tokens are never written
        s["codes"] = torch.zeros(padded, k // 2, dtype=torch.uint8, device=DEVICE)
        s["scales"] = torch.zeros(k // 64, padded, dtype=dtype, device=DEVICE)
        s["lora"] = torch.zeros(padded, rank, dtype=torch.float32, device=DEVICE)
        s["out"] = torch.zeros(tokens, n, dtype=dtype, device=DEVICE)
        _operators(s)
        s["x"] = _activations(g, tokens, k, dtype)[0]
    elif kind == "qkv":
        k, tokens = case["k"], case["tokens"]
        s["lin"] = _svdq(g, k, 3 * case["heads"] * 128, case["rank"], dtype)
        s["norm_q"], s["norm_k"] = _norm_weight(g, dtype), _norm_weight(g, dtype)
        s["mod"] = (1 + _normal(g, k, scale=0.3, dtype=dtype), _normal(g, k, scale=0.2, dtype=dtype))
        s["rot"] = rope_table(flux_ids(0, 1, tokens, device=DEVICE), (16, 56, 56), 10000.0)
        s["x"] = _activations(g, tokens, k, dtype)
        ops.fused_qkv_norm_rottary(s["x"] * 0.5, s["lin"], s["norm_q"], s["norm_k"], s["rot"], norm=s["mod"])
    elif kind == "mlp":
        k, hidden = case["k"], case["hidden"]
        s["fc1"] = _svdq(g, k, hidden, case["rank"], dtype)
        s["fc2"] = _svdq(g, hidden, k, case["rank"], dtype, unsigned=True)
        s["mod"] = (1 + _normal(g, k, scale=0.3, dtype=dtype), _normal(g, k, scale=0.2, dtype=dtype))
        s["x"] = _activations(g, case["tokens"], k, dtype)
        ops.fused_gelu_mlp(s["x"][:, :1] * 0.5, s["fc1"], s["fc2"], norm=s["mod"])
    elif kind == "swiglu":
        k, hidden = case["k"], case["hidden"]
        s["fc1"] = _svdq(g, k, 2 * hidden, case["rank"], dtype)
        s["fc2"] = _svdq(g, hidden, k, case["rank"], dtype)
        ops.interleave_swiglu_linear_(s["fc1"])
        s["x"] = _activations(g, case["tokens"], k, dtype)
        ops.fused_swiglu_mlp(s["x"][:, :1] * 0.5, s["fc1"], s["fc2"])
    elif kind == "attention":
        B, H, D, q, kv = case["batch"], case["heads"], case["d"], case["q"], case["kv"]
        if q == kv:  # self attention: views of one fused projection
            parts = _normal(g, B, q, 3 * H * D, dtype=dtype).chunk(3, dim=-1)
        else:
            parts = (_normal(g, B, q, H * D, dtype=dtype), *_normal(g, B, kv, 2 * H * D, dtype=dtype).chunk(2, dim=-1))
        s["qkv"] = [t.view(B, -1, H, D).transpose(1, 2) for t in parts]
    elif kind == "encoder":
        s["lin"] = _awq(g, case["k"], case["n"], case["group"], dtype)
        s["x"] = _normal(g, 1, case["tokens"], case["k"], dtype=dtype)
        s["group"] = case["group"]
    else:
        cfg = FluxShapedConfig(n_double=case["double"], n_single=case["single"])
        h, w, text = case["grid_h"], case["grid_w"], case["text"]
        s["model"] = FluxShapedTransformer(cfg, device=DEVICE, dtype=dtype, seed=seed)
        s["rot"] = rope_table(flux_ids(text, h, w, device=DEVICE), cfg.axes_dim, cfg.theta)
        s["text"] = _normal(g, 1, text, cfg.text_dim, dtype=dtype)
        s["pooled"] = _normal(g, 1, cfg.pooled_dim, dtype=dtype)
        s["time"] = torch.rand(1, device=DEVICE, generator=g)
        s["latents"] = _normal(g, 1, h * w, cfg.in_channels, dtype=dtype)
        with torch.no_grad():  # the step before this one
            s["model"](s["latents"] * 0.5, s["text"], s["pooled"], s["time"], s["rot"])
    return s


def _operators(s):
    lin = s["lin"]
    codes, scales, lora = ops.svdq_quantize_w4a4_act_fuse_lora_cuda(
        s["x"], output=s["codes"], oscales=s["scales"], lora_down=lin.proj_down, lora_act_out=s["lora"], smooth=lin.smooth_factor
    )
    ops.svdq_gemm_w4a4_cuda(act=codes, wgt=lin.qweight, out=s["out"], ascales=scales, wscales=lin.wscales, lora_act_in=lora,
                            lora_up=lin.proj_up, bias=lin.bias)  # fmt: skip
    return codes, scales, lora, s["out"]


@torch.no_grad()
def run(s):
    kind = s["kind"]
    if kind in ("modulation", "linear"):
        return s["lin"](s["x"])
    if kind == "operators":
        return _operators(s)
    if kind == "qkv":
        return ops.fused_qkv_norm_rottary(s["x"], s["lin"], s["norm_q"], s["norm_k"], s["rot"], norm=s["mod"])
    if kind == "mlp":
        return ops.fused_gelu_mlp(s["x"], s["fc1"], s["fc2"], norm=s["mod"])
    if kind == "swiglu":
        return ops.fused_swiglu_mlp(s["x"], s["fc1"], s["fc2"])
    if kind == "attention":
        return ops.scaled_dot_product_attention(*s["qkv"])
    if kind == "encoder":
        lin = s["lin"]
        return ops.awq_gemm_w4a16(s["x"], lin.qweight, lin.wscales, lin.wzeros, group_size=s["group"])
    return s["model"](s["latents"], s["text"], s["pooled"], s["time"], s["rot"])


def _linear_work(m, k, n, rank):
    """Packed weight with its scales and bias, low-rank factors, smoothing; 16-bit input and output."""
    weights = n * k / 2 + 2 * n * k / 64 + 2 * n + 2 * rank * (k + n) + 2 * k
    return weights, 2.0 * m * n * k + 2.0 * m * rank * (k + n)


def work(case):
    kind = case["kind"]
    if kind == "modulation":
        m, k, n = case["rows"], case["k"], case["n"]
        return {"bytes": n * k / 2 + 4 * n * k / 64 + 2 * n + 2 * m * (k + n), "flops": 2.0 * m * n * k}
    if kind == "encoder":
        m, k, n = case["tokens"], case["k"], case["n"]
        return {"bytes": n * k / 2 + 4 * n * k / case["group"] + 2 * m * (k + n), "flops": 2.0 * m * n * k}
    if kind == "attention":
        B, H, D, q, kv = case["batch"], case["heads"], case["d"], case["q"], case["kv"]
        return {"bytes": 2.0 * B * H * D * (2 * q + 2 * kv), "flops": 4.0 * B * H * D * q * kv}
    if kind == "transformer":
        C, m, text = 3072, case["grid_h"] * case["grid_w"] + case["text"], case["text"]
        image, total_b, total_f = m - text, 0.0, 4.0 * 128 * 24 * m * m * (case["double"] + case["single"])
        for count, rows in ((case["double"], image), (case["double"], text), (case["single"], m)):
            for k, n in ((C, 3 * C), (C, C), (C, 4 * C), (4 * C, C)):
                b, f = _linear_work(rows, k, n, 32)
                total_b, total_f = total_b + count * b, total_f + count * f
        modulations = C * C * (2 * 6 * case["double"] + 3 * case["single"])
        # modulations, embedders, output layer; the latents come in and the velocity goes out
        total_b += modulations * (0.5 + 4 / 64) + 2 * (C * C * 4 + C * (256 + 768 + 4096 + 128)) + 2 * (2 * image * 64 + text * 4096)
        return {"bytes": total_b, "flops": total_f + 2.0 * (modulations + 4 * C * C) + 2.0 * C * (image * 128 + text * 4096)}
    m, k, rank = case["tokens"], case["k"], case["rank"]
    if kind in ("linear", "operators", "qkv"):
        n = 3 * case["heads"] * 128 if kind == "qkv" else case["n"]
        b, f = _linear_work(m, k, n, rank)
        if kind == "operators":  # the codes, scales and low-rank state are results too
            b += m * k / 2 + 2 * m * k / 64 + 4 * m * rank
        if kind == "qkv":  # rotary table
            b += 4 * m * 128
        return {"bytes": b + 2 * m * (k + n), "flops": f}
    hidden = case["hidden"]
    b1, f1 = _linear_work(m, k, hidden * (2 if kind == "swiglu" else 1), rank)
    b2, f2 = _linear_work(m, hidden, k, rank)
    return {"bytes": b1 + b2 + 4 * m * k, "flops": f1 + f2}


# Largest relative error, (bf16, fp16): about four times what the path differed by from itself with its sums made another
# way (the GEMM's other main loop, whose offset terms round differently; attention and the 4-bit projections against 32-
# and 64-bit arithmetic).  Between two GEMMs a last-bit difference can move an int4 code by one step, and a transformer
# hands such steps on from layer to layer (1.6e-2 seen with another attention kernel).
_REL = {
    "modulation": (8e-3, 1.2e-3),  # 2.2e-3 / 3.1e-4: the product is rounded before the bias is added
    "encoder": (7e-3, 8e-4),  # 1.7e-3 / 2.1e-4
    "linear": (1e-3, 2e-4),  # 8.4e-5 / 1.6e-5, and the 16-bit rounding of the low-rank state on top
    "operators": (1e-3, 2e-4),
    "qkv": (1e-3, 2e-4),  # 7.7e-5 / 1.6e-5, likewise
    "mlp": (1.5e-3, 3.5e-4),  # 3.6e-4 / 8.6e-5
    "swiglu": (4.5e-3, 1.2e-3),  # 1.1e-3 / 3.0e-4
    "attention": (1e-2, 1.5e-3),  # 2.9e-3 / 3.6e-4: the probabilities are 16-bit operands
    "transformer": (3e-2, 3e-2),
}


def tolerance(case):
    return {"rel": _REL[case["kind"]][case["dtype"] == "fp16"]}
