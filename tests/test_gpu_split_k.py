"""The GEMM for few rows (K split over the wavefronts of 32 x 128 workgroups) against the kernel with 128 x 128 tiles and in
exact arithmetic, at the edges of its rows, columns and K, and on both sides of the lines where it takes over."""

import pytest
import torch

from oracle import svdq_oracle as O

pytestmark = pytest.mark.gpu


def _both(call):
    """``call()`` by the tile kernel and, twice, as the rule chooses."""
    from nunchaku_rocm_amd.ops import gemm as gemm_mod

    gemm_mod.set_fp8_loop_variant(1)
    try:
        tiles = call()
    finally:
        gemm_mod.set_fp8_loop_variant(-1)
    return tiles, call(), call()


def _module(dev, K, N, R, dtype, unsigned=False):
    from nunchaku_rocm_amd.linear import SVDQW4A4Linear

    lin = O.make_svdq_linear(K, N, R=R, seed=K + N, dtype=dtype)
    mod = SVDQW4A4Linear(K, N, rank=R, act_unsigned=unsigned, torch_dtype=dtype, device=dev).requires_grad_(False)
    for name in ("qweight", "wscales", "smooth_factor", "proj_down", "proj_up", "bias"):
        getattr(mod, name).data.copy_(lin[name])
    return mod


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(
    "M,K,N,R",
    [
        (1, 64, 8, 16),  # one group: most wavefronts have no stage
        (31, 192, 136, 16),  # odd number of groups, a column block past N
        (33, 512, 128, 32),  # half the wavefronts without a stage
        (100, 1088, 264, 48),  # nine stages over eight wavefronts
        (333, 1536, 1544, 64),  # 8 wavefronts, one column block of eight rows
        (333, 1216, 4096, 32),  # 352 workgroups: 4 wavefronts, an odd number of groups
        (512, 3072, 4096, 32),  # the last launch that is split: 512 workgroups
    ],
)
def test_split_against_tiles(dev, M, K, N, R, dtype):
    print(f"case M={M} K={K} N={N} R={R} {dtype}", flush=True)
    mod = _module(dev, K, N, R, dtype)
    x = O.make_activations(M, K, seed=M, dtype=dtype).to(dev)[None]
    canary = torch.full((M + 8, N), 7.0, dtype=dtype, device=dev)
    with torch.no_grad():
        tiles, a, b = _both(lambda: mod(x, output=canary[:M]).clone())
    assert torch.equal(a, b)  # the same bits every time
    assert (canary[M:] == 7.0).all()
    # fp32 sums of the K / 64 group terms in another order, then one rounding to the 16-bit type on either side
    absum = (K // 64) * 2.0**-24 * _abs_terms(mod, x)
    bound = tiles.float().abs() * (2.0**-7 if dtype == torch.bfloat16 else 2.0**-10) + 2 * absum + 1e-6
    assert ((a.float() - tiles.float()).abs() <= bound).all()


def _abs_terms(mod, x):
    """Sum of the absolute group terms of every output, for the bound on reordered fp32 sums."""
    q, s, la = mod.quantize(x[0])
    M, K = x.shape[1], x.shape[2]
    act = O.unpack_int4(q[:M].cpu(), True).float().abs().view(M, K // 64, 64) * s.cpu()[:, :M].t().float()[:, :, None]
    wgt = O.unpack_int4(mod.qweight.cpu(), True).float().abs().view(-1, K // 64, 64) * mod.wscales.cpu().t().float()[:, :, None]
    lora = la[:M].cpu().abs() @ mod.proj_up.float().cpu().abs().t()
    return (act.reshape(M, K) @ wgt.reshape(-1, K).t() + lora + mod.bias.float().cpu().abs()).to(x.device)[None]


@pytest.mark.parametrize("blocked", [0, 1, 2, 3])
@pytest.mark.parametrize("M,N,K", [(40, 136, 512), (333, 4104, 1024)])
def test_unsigned_hand_over_forms_at_unit_scales(dev, M, N, K, blocked):
    """Every form of unsigned activations through the split: integers below 2^24, exact in any order."""
    from nunchaku_rocm_amd import ops
    from nunchaku_rocm_amd.layout import block_activations, block_activations_f6, block_scales

    print(f"case M={M} N={N} K={K} blocked={blocked}", flush=True)
    rows = -(-M // 32) * 32
    g = torch.Generator().manual_seed(M + blocked)
    act = torch.randint(0, 256, (rows, K // 2), dtype=torch.uint8, generator=g)
    wgt = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, generator=g).view(torch.int8)
    one = lambda n: torch.ones(K // 64, n, dtype=torch.float16, device=dev)  # noqa: E731
    ref = O.unpack_int4(act[:M], False).double() @ O.unpack_int4(wgt, True).double().t()
    sent = {0: lambda: act, 1: lambda: block_activations(act), 2: lambda: block_activations_f6(act, True), 3: lambda: block_activations_f6(act, True)}[blocked]()
    scales = block_scales(one(rows)) if blocked == 3 else one(rows)
    out = torch.empty(M, N, dtype=torch.float16, device=dev)
    param = torch.nn.Parameter(wgt.to(dev), requires_grad=False)
    ops.svdq_gemm_w4a4_cuda(act=sent.to(dev), wgt=param, out=out, ascales=scales, wscales=one(N), act_unsigned=True, act_blocked=blocked)
    assert torch.equal(out.cpu(), ref.to(torch.float16))


@pytest.mark.parametrize("dtype,rel", [(torch.bfloat16, 1.5e-3), (torch.float16, 3.5e-4)])
@pytest.mark.parametrize("tokens,K,hidden", [(1, 512, 512), (130, 1024, 4096), (333, 1536, 2048)])
def test_requantizing_epilogues(dev, tokens, K, hidden, dtype, rel):
    """GELU and SwiGLU feed-forwards; a last-bit difference may move a code by one step: the bound on the result is the one
    for two correct orders of the sums (measured between the tile kernel's two main loops, times four)."""
    from nunchaku_rocm_amd import ops

    print(f"case tokens={tokens} K={K} hidden={hidden} {dtype}", flush=True)
    x = O.make_activations(tokens, K, seed=tokens, dtype=dtype).to(dev)[None]
    gelu = _module(dev, K, hidden, 32, dtype), _module(dev, hidden, K, 32, dtype, unsigned=True)
    glu = _module(dev, K, 2 * hidden, 32, dtype), _module(dev, hidden, K, 32, dtype)
    ops.interleave_swiglu_linear_(glu[0])
    for fn, (fc1, fc2), bar in ((ops.fused_gelu_mlp, gelu, rel), (ops.fused_swiglu_mlp, glu, 3 * rel)):
        with torch.no_grad():
            tiles, a, b = _both(lambda: fn(x, fc1, fc2))
        assert torch.equal(a, b)
        assert ((a.double() - tiles.double()).norm() / tiles.double().norm()).item() <= bar


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tokens,heads", [(7, 1), (257, 3), (300, 12)])
def test_qk_norm_rope(dev, tokens, heads, dtype):
    from nunchaku_rocm_amd import ops
    from nunchaku_rocm_amd.flux_shaped import flux_ids, rope_table

    print(f"case tokens={tokens} heads={heads} {dtype}", flush=True)
    mod = _module(dev, 512, 3 * heads * 128, 32, dtype)
    norm = torch.nn.RMSNorm(128, eps=1e-6, device=dev, dtype=dtype).requires_grad_(False)
    rot = rope_table(flux_ids(0, 1, tokens, device=dev), (16, 56, 56), 10000.0)
    x = O.make_activations(tokens, 512, seed=tokens, dtype=dtype).to(dev)[None]
    with torch.no_grad():
        tiles, a, b = _both(lambda: ops.fused_qkv_norm_rottary(x, mod, norm, norm, rot))
    assert torch.equal(a, b)
    # each side within one rounding of values that differ in the order of eight group terms
    assert ((a.float() - tiles.float()).abs() <= tiles.float().abs() * (2.0**-7 if dtype == torch.bfloat16 else 2.0**-10) + 1e-4).all()
