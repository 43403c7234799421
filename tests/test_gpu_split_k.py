"""The GEMM for few rows (K split over the wavefronts of 32 x 128 workgroups) against the kernel with 128 x 128 tiles and in
exact arithmetic, at the edges of its rows, columns and K, and on both sides of the lines where it takes over."""

import pytest
import torch

from oracle import svdq_oracle as O



@pytest.fixture
def splits(monkeypatch):
    """Over how many wavefronts each GEMM launched so far split K (0: the tile kernel)."""
    from nunchaku_rocm_amd import _lib

    lib, seen = _lib.load(), []

    class Watched:
        def __getattr__(self, name):
            return getattr(lib, name)

        def svdq_gemm_w4a4(self, args, stream):
            seen.append(lib.svdq_gemm_w4a4_split_wavefronts(args, 0))
            return lib.svdq_gemm_w4a4(args, stream)

    watched = Watched()
    monkeypatch.setattr(_lib, "load", lambda: watched)
    return seen


def _both(call, splits, expected):
    """``call()`` by the tile kernel and, twice, as the rule chooses: its GEMMs split over the ``expected`` wavefronts."""
    from nunchaku_rocm_amd.ops import gemm as gemm_mod

    gemm_mod.set_fp8_loop_variant(1)
    try:
        tiles = call()
    finally:
        gemm_mod.set_fp8_loop_variant(-1)
    assert splits == [0] * len(expected)
    splits.clear()
    results = tiles, call(), call()
    assert splits == 2 * list(expected)
    return results


@pytest.mark.parametrize("epilogue,quant,first,at_2048", [(0, False, 1216, 4), (1, False, 1344, 0), (2, True, 1600, 0), (3, True, 1216, 4)])
def test_lines_of_the_rule(epilogue, quant, first, at_2048):
    """Where the split begins and ends, in rows, columns, K and rank, on 256 CUs; forms that it does not take.  ``first``: the
    shortest K of a launch with more workgroups than CUs and a rank below 64."""
    from nunchaku_rocm_amd import _lib

    def wavefronts(rows, n, k, rank=32, **more):
        m = -(-rows // 256) * 256
        args = dict(wgt_planes=16, M=rows if quant else m, actual_m=rows, N=n, K=k, epilogue=epilogue, act_blocked=2, R=rank, R2=rank)
        return _lib.load().svdq_gemm_w4a4_split_wavefronts(_lib.GemmArgs(**{**args, **more}), 256)

    assert wavefronts(32, 8, 256) == 0 and wavefronts(32, 8, 320) == 8
    assert wavefronts(256, 4096, 320) == 8 and wavefronts(256, 4096, 12288) == 8  # 256 workgroups
    assert wavefronts(288, 4096, first - 64) == 0 and wavefronts(288, 4096, first) == 4  # 288
    assert wavefronts(512, 4096, 2048) == at_2048 and wavefronts(512, 4096, 2112) == 4  # 512
    assert wavefronts(32, 8, 64, 48) == 0 and wavefronts(32, 8, 64, 64) == 8
    assert wavefronts(288, 4096, 256, 64) == 0 and wavefronts(288, 4096, 320, 64) == 4 and wavefronts(288, 4096, 1024, 112) == 0
    assert wavefronts(288, 4096, 64, 128) == 4 and wavefronts(512, 4096, 1024, 128) == 4
    assert wavefronts(288, 4096, 320, 64, R2=16) == (0 if quant else 4)
    assert wavefronts(544, 4096, 3072) == 0 and wavefronts(544, 4096, 3072, 256) == 0  # 544
    assert wavefronts(32, 8, 1024, wgt_planes=None) == 0
    assert wavefronts(32, 8, 1024, act_blocked=1) == 0 and wavefronts(32, 8, 1024, act_blocked=0) == 0
    assert wavefronts(32, 8, 1024, act_blocked=1, act_unsigned=1) == 8 and wavefronts(32, 8, 1024, act_blocked=0, act_unsigned=1) == 8


def _module(dev, K, N, R, dtype, unsigned=False):
    from nunchaku_rocm_amd.linear import SVDQW4A4Linear

    lin = O.make_svdq_linear(K, N, R=R, seed=K + N, dtype=dtype)
    mod = SVDQW4A4Linear(K, N, rank=R, act_unsigned=unsigned, torch_dtype=dtype, device=dev).requires_grad_(False)
    for name in ("qweight", "wscales", "smooth_factor", "proj_down", "proj_up", "bias"):
        getattr(mod, name).data.copy_(lin[name])
    return mod


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(
    "M,K,N,R,wavefronts",
    [
        (1, 64, 8, 16, 0),  # one group: left to the tiles
        (31, 192, 136, 16, 0),
        (40, 64, 136, 64, 8),  # one group, half a stage: seven wavefronts have none
        (333, 128, 4104, 128, 4),  # one stage: three have none
        (1, 320, 8, 16, 8),  # three stages, the last one half: five wavefronts have none
        (31, 448, 136, 16, 8),  # odd number of groups, a column block past N
        (33, 512, 128, 32, 8),  # half the wavefronts without a stage
        (100, 1088, 264, 48, 8),  # nine stages over eight wavefronts
        (333, 1536, 1544, 64, 8),  # one column block of eight rows
        (333, 1216, 4096, 32, 4),  # 352 workgroups, an odd number of groups
        (333, 1408, 4104, 128, 4),  # 363 workgroups, eleven stages over four wavefronts
        (512, 3072, 4096, 32, 4),  # the last launch that is split: 512 workgroups
        (513, 3072, 4096, 32, 0),  # 544
    ],
)
def test_split_against_tiles(dev, splits, M, K, N, R, wavefronts, dtype):
    print(f"case M={M} K={K} N={N} R={R} {dtype}", flush=True)
    mod = _module(dev, K, N, R, dtype)
    x = O.make_activations(M, K, seed=M, dtype=dtype).to(dev)[None]
    canary = torch.full((M + 8, N), 7.0, dtype=dtype, device=dev)
    with torch.no_grad():
        tiles, a, b = _both(lambda: mod(x, output=canary[:M]).clone(), splits, [wavefronts])
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


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["matrix", "lane order", "fp6", "fp6 and scales", "signed fp6", "signed fp6 and scales"])
@pytest.mark.parametrize("M,N,K,wavefronts", [(40, 136, 512, 8), (333, 4104, 1536, 4)])
def test_hand_over_forms_at_unit_scales(dev, splits, M, N, K, wavefronts, form):
    """Every form of activations that the split takes: integers below 2^24, exact in any order."""
    from nunchaku_rocm_amd import ops
    from nunchaku_rocm_amd.layout import block_activations, block_activations_f6, block_scales

    print(f"case M={M} N={N} K={K} {form}", flush=True)
    unsigned = "signed" not in form
    rows = -(-M // 32) * 32
    g = torch.Generator().manual_seed(M)
    act = torch.randint(0, 256, (rows, K // 2), dtype=torch.uint8, generator=g)
    wgt = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, generator=g).view(torch.int8)
    one = lambda n: torch.ones(K // 64, n, dtype=torch.float16, device=dev)  # noqa: E731
    ref = O.unpack_int4(act[:M], not unsigned).double() @ O.unpack_int4(wgt, True).double().t()
    sent, blocked = {"matrix": (lambda: act, 0), "lane order": (lambda: block_activations(act), 1)}.get(
        form, (lambda: block_activations_f6(act, unsigned), 3 if "scales" in form else 2)
    )
    scales = block_scales(one(rows)) if blocked == 3 else one(rows)
    out = torch.empty(M, N, dtype=torch.float16, device=dev)
    param = torch.nn.Parameter(wgt.to(dev), requires_grad=False)
    ops.svdq_gemm_w4a4_cuda(act=sent().to(dev), wgt=param, out=out, ascales=scales, wscales=one(N), act_unsigned=unsigned, act_blocked=blocked)
    assert splits == [wavefronts]
    assert torch.equal(out.cpu(), ref.to(torch.float16))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,rel", [(torch.bfloat16, 1.5e-3), (torch.float16, 3.5e-4)])
@pytest.mark.parametrize(
    "tokens,K,hidden,gelu_split,glu_split",  # of the two GEMMs: the first has its rows padded to 256 and, for SwiGLU, twice the columns
    [
        (1, 512, 512, [8, 8], [8, 8]),
        (130, 1024, 4096, [8, 8], [0, 8]),
        (333, 1536, 2048, [8, 8], [4, 8]),
        (600, 1600, 2048, [4, 8], [0, 8]),
    ],
)
def test_requantizing_epilogues(dev, splits, tokens, K, hidden, gelu_split, glu_split, dtype, rel):
    """GELU and SwiGLU feed-forwards; a last-bit difference may move a code by one step: the bound on the result is the one
    for two correct orders of the sums (measured between the tile kernel's two main loops, times four)."""
    from nunchaku_rocm_amd import ops

    print(f"case tokens={tokens} K={K} hidden={hidden} {dtype}", flush=True)
    x = O.make_activations(tokens, K, seed=tokens, dtype=dtype).to(dev)[None]
    gelu = _module(dev, K, hidden, 32, dtype), _module(dev, hidden, K, 32, dtype, unsigned=True)
    glu = _module(dev, K, 2 * hidden, 32, dtype), _module(dev, hidden, K, 32, dtype)
    ops.interleave_swiglu_linear_(glu[0])
    for fn, (fc1, fc2), bar, expected in ((ops.fused_gelu_mlp, gelu, rel, gelu_split), (ops.fused_swiglu_mlp, glu, 3 * rel, glu_split)):
        splits.clear()
        with torch.no_grad():
            tiles, a, b = _both(lambda: fn(x, fc1, fc2), splits, expected)
        assert torch.equal(a, b)
        assert ((a.double() - tiles.double()).norm() / tiles.double().norm()).item() <= bar


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tokens,heads,K,wavefronts", [(7, 1, 512, 8), (257, 3, 512, 8), (300, 12, 512, 0), (300, 12, 1536, 4)])
def test_qk_norm_rope(dev, splits, tokens, heads, K, wavefronts, dtype):
    from nunchaku_rocm_amd import ops
    from nunchaku_rocm_amd.flux_shaped import flux_ids, rope_table

    print(f"case tokens={tokens} heads={heads} K={K} {dtype}", flush=True)
    mod = _module(dev, K, 3 * heads * 128, 32, dtype)
    norm = torch.nn.RMSNorm(128, eps=1e-6, device=dev, dtype=dtype).requires_grad_(False)
    rot = rope_table(flux_ids(0, 1, tokens, device=dev), (16, 56, 56), 10000.0)
    x = O.make_activations(tokens, K, seed=tokens, dtype=dtype).to(dev)[None]
    with torch.no_grad():
        tiles, a, b = _both(lambda: ops.fused_qkv_norm_rottary(x, mod, norm, norm, rot), splits, [wavefronts])
    assert torch.equal(a, b)
    # each side within one rounding of values that differ in the order of the K / 64 group terms
    assert ((a.float() - tiles.float()).abs() <= tiles.float().abs() * (2.0**-7 if dtype == torch.bfloat16 else 2.0**-10) + 1e-4).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,N", [(65, 1280, 16640), (65, 1280, 16384), (33, 1344, 18440), (160, 3072, 8192)])
def test_rows_of_a_workgroup(dev, splits, M, K, N, dtype):
    """Workgroups of 64 rows up to one per CU (256 at 65 x 16384 on 256 CUs), beyond that (260) of 32; a last workgroup of one row,
    a second row block without rows and a column half past N."""
    print(f"case M={M} K={K} N={N} {dtype}", flush=True)
    mod = _module(dev, K, N, 32, dtype)
    x = O.make_activations(M, K, seed=M, dtype=dtype).to(dev)[None]
    canary = torch.full((M + 8, N), 7.0, dtype=dtype, device=dev)
    with torch.no_grad():
        tiles, a, b = _both(lambda: mod(x, output=canary[:M]).clone(), splits, [4])
    assert torch.equal(a, b) and (canary[M:] == 7.0).all()
    # as in test_split_against_tiles
    bound = tiles.float().abs() * (2.0**-7 if dtype == torch.bfloat16 else 2.0**-10) + 2 * (K // 64) * 2.0**-24 * _abs_terms(mod, x) + 1e-6
    assert ((a.float() - tiles.float()).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(40, 136, 512), (333, 4104, 1536), (65, 16640, 1536)])
def test_hand_over_forms_give_the_same_bits(dev, splits, M, N, K):
    """Unsigned activations with ordinary scales: the same sums in the same order in every form."""
    from nunchaku_rocm_amd import ops
    from nunchaku_rocm_amd.layout import block_activations, block_activations_f6, block_scales

    print(f"case M={M} N={N} K={K}", flush=True)
    rows = -(-M // 32) * 32
    g = torch.Generator().manual_seed(M)
    act = torch.randint(0, 256, (rows, K // 2), dtype=torch.uint8, generator=g)
    asc = (torch.rand(K // 64, rows, generator=g) * 0.1 + 0.01).to(torch.bfloat16)
    wgt = torch.nn.Parameter(torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, generator=g).view(torch.int8).to(dev), requires_grad=False)
    wsc = (torch.rand(K // 64, N, generator=g) * 0.02 + 0.005).to(torch.bfloat16).to(dev)
    f6 = block_activations_f6(act, True)
    results = []
    for sent, scales, blocked in ((act, asc, 0), (block_activations(act), asc, 1), (f6, asc, 2), (f6, block_scales(asc), 3)):
        out = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
        ops.svdq_gemm_w4a4_cuda(act=sent.to(dev), wgt=wgt, out=out, ascales=scales.to(dev), wscales=wsc, act_unsigned=True, act_blocked=blocked)
        results.append(out.cpu())
    assert len(set(splits)) == 1 and splits[0] in (4, 8)
    assert all(torch.equal(r, results[0]) for r in results[1:])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("form", ["fp6 and scales", "fp6", "nibbles"])
@pytest.mark.parametrize("M,K", [(65, 1536), (90, 2560), (96, 4608)])
def test_rows_of_a_workgroup_leave_the_sums_alone(dev, splits, M, K, form, dtype):
    """16640 columns are 260 workgroups of 64 rows, more than 256 CUs, and run as 32-row ones; the first 16384 alone are 256 and do not: the same
    bits in either."""
    from nunchaku_rocm_amd import ops
    from nunchaku_rocm_amd.layout import block_activations_f6, block_scales

    print(f"case M={M} K={K} {form} {dtype}", flush=True)
    g = torch.Generator().manual_seed(M + K)
    act = torch.randint(0, 256, (96, K // 2), dtype=torch.uint8, generator=g)
    asc = (torch.rand(K // 64, 96, generator=g) * 0.1 + 0.01).to(dtype)
    wgt = torch.randint(0, 256, (16640, K // 2), dtype=torch.uint8, generator=g).view(torch.int8)
    wsc = (torch.rand(K // 64, 16640, generator=g) * 0.02 + 0.005).to(dtype)
    nibbles, blocked = form == "nibbles", {"fp6 and scales": 3, "fp6": 2, "nibbles": 0}[form]
    sent, scales = (act if nibbles else block_activations_f6(act, False)).to(dev), (block_scales(asc) if blocked == 3 else asc).to(dev)
    out = []
    for n in (16640, 16384):
        out.append(torch.empty(M, n, dtype=dtype, device=dev))
        param = torch.nn.Parameter(wgt[:n].contiguous().to(dev), requires_grad=False)
        ops.svdq_gemm_w4a4_cuda(act=sent, wgt=param, out=out[-1], ascales=scales, wscales=wsc[:, :n].contiguous().to(dev), act_unsigned=nibbles, act_blocked=blocked)
    assert splits == [4, 4]
    assert torch.equal(out[0][:, :16384], out[1])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,rel", [(torch.bfloat16, 1.5e-3), (torch.float16, 3.5e-4)])
@pytest.mark.parametrize("K", [320, 512])
def test_epilogues_of_32_row_workgroups(dev, splits, K, dtype, rel):
    """Four wavefronts along K of 64-rank launches with 260 and 273 workgroups: K up to 896 stays with 32 rows to a workgroup (some wavefronts have one
    stage, at K = 320 one has none).  Bounds as in test_requantizing_epilogues and test_qk_norm_rope."""
    from nunchaku_rocm_amd import ops
    from nunchaku_rocm_amd.flux_shaped import flux_ids, rope_table

    print(f"case K={K} {dtype}", flush=True)
    x = O.make_activations(400, K, seed=K, dtype=dtype).to(dev)[None]
    glu = _module(dev, K, 2560, 64, dtype), _module(dev, 1280, K, 64, dtype)
    ops.interleave_swiglu_linear_(glu[0])
    for fn, fc1, fc2, bar in (
        (ops.fused_gelu_mlp, _module(dev, K, 2560, 64, dtype), _module(dev, 2560, K, 64, dtype, unsigned=True), rel),
        (ops.fused_swiglu_mlp, *glu, 3 * rel),
    ):
        splits.clear()
        with torch.no_grad():
            tiles, a, b = _both(lambda: fn(x, fc1, fc2), splits, [4, 8])
        assert torch.equal(a, b)
        assert ((a.double() - tiles.double()).norm() / tiles.double().norm()).item() <= bar
    mod = _module(dev, K, 3 * 7 * 128, 64, dtype)
    norm = torch.nn.RMSNorm(128, eps=1e-6, device=dev, dtype=dtype).requires_grad_(False)
    rot = rope_table(flux_ids(0, 1, 400, device=dev), (16, 56, 56), 10000.0)
    splits.clear()
    with torch.no_grad():
        tiles, a, b = _both(lambda: ops.fused_qkv_norm_rottary(x, mod, norm, norm, rot), splits, [4])
    assert torch.equal(a, b)
    assert ((a.float() - tiles.float()).abs() <= tiles.float().abs() * (2.0**-7 if dtype == torch.bfloat16 else 2.0**-10) + 1e-4).all()
