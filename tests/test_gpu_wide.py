"""The GEMM with 256 x 128 tiles against the kernel with 128 x 128 tiles (which the oracle tests cover), bit for bit, at the edges
of its rows, columns, K and ranks, and at launches that mix whole tiles with halves."""

import pytest
import torch

from oracle import svdq_oracle as O

pytestmark = pytest.mark.gpu


def _outputs(rows, k, n, rank, epilogue, dtype, dev, build):
    """Everything one launch writes, buffers' untouched rows included."""
    from nunchaku_rocm_amd import ops
    from nunchaku_rocm_amd.ops import gemm as G

    lin = {name: t.to(dev) for name, t in O.make_svdq_linear(k, n, R=max(rank, 16), seed=k + n, dtype=dtype).items()}
    g = torch.Generator(device=dev).manual_seed(rows)
    x = torch.randn(rows, k, generator=g, device=dev).to(dtype)
    down, up = (lin["proj_down"][:, :rank].contiguous(), lin["proj_up"][:, :rank].contiguous()) if rank else (None, None)
    M = -(-rows // 256) * 256  # rows past the tokens stay zero: the requantizing epilogues read them too
    q, s = torch.zeros(M, k * 3 // 4, dtype=torch.uint8, device=dev), torch.zeros(k // 64, M, dtype=dtype, device=dev)
    la = torch.zeros(M, rank, dtype=torch.float32, device=dev)
    ops.svdq_quantize_w4a4_act_fuse_lora_cuda(x, output=q, oscales=s, lora_down=down, lora_act_out=la if rank else None,
                                              smooth=lin["smooth_factor"], out_blocked=3)  # fmt: skip
    kw = dict(act=q, wgt=lin["qweight"], ascales=s, wscales=lin["wscales"], lora_act_in=la if rank else None, lora_up=up, bias=lin["bias"],
              act_blocked=3)  # fmt: skip
    if epilogue in ("plain", "qkv"):
        kw["out"] = torch.full((rows, n), 3.0, dtype=dtype, device=dev)
        if epilogue == "qkv":
            kw.update(norm_q=torch.rand(128, generator=g, device=dev).to(dtype), norm_k=torch.rand(128, generator=g, device=dev).to(dtype),
                      rotary_emb=torch.randn(rows, 128, generator=g, device=dev))  # fmt: skip
        names = ("out",)
    else:
        nq = n // 2 if epilogue == "swiglu" else n
        blocked = 3 if nq % 512 == 0 else 2
        kw.update(qout=torch.full((M, nq * 3 // 4), 7, dtype=torch.uint8, device=dev), oscales=torch.full((nq // 64, M), 3.0, dtype=dtype, device=dev),
                  lora_down=torch.randn(nq, 48, generator=g, device=dev).to(dtype), lora_act_out=torch.empty(M, 48, device=dev),
                  smooth_factor=torch.rand(nq, generator=g, device=dev).to(dtype) + 0.5, fuse_swiglu=epilogue == "swiglu",
                  qout_blocked=blocked)  # fmt: skip
        names = ("qout", "oscales", "lora_act_out")
    old, G.USE_WEIGHT_PLANES = G.USE_WEIGHT_PLANES, "all"
    G.set_fp8_loop_variant(build)
    try:
        ops.svdq_gemm_w4a4_cuda(**kw)
        torch.cuda.synchronize()
    finally:
        G.set_fp8_loop_variant(-1)
        G.USE_WEIGHT_PLANES = old
    return [kw[name].view(torch.uint8).cpu() for name in names]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(
    "rows,k,n,rank,epilogue",
    [
        (1, 512, 8, 0, "plain"), (33, 512, 136, 32, "plain"), (128, 1024, 128, 48, "plain"), (129, 512, 264, 16, "plain"),
        (256, 3584, 384, 32, "plain"), (257, 512, 392, 32, "plain"), (385, 512, 128, 160, "plain"),
        (300, 512, 384, 32, "qkv"), (513, 1024, 768, 64, "qkv"),
        (16, 512, 128, 32, "gelu"), (333, 512, 512, 16, "gelu"), (400, 1024, 256, 64, "swiglu"), (129, 512, 1024, 32, "swiglu"),
        # 36 of these tiles to an XCD of 32 CUs: four as halves; 54: all whole; 10: all halves; 33 or 34, and a last row of tiles
        # with 65 rows: halves that have none
        (1024, 512, 9216, 32, "plain"), (1500, 512, 9216, 0, "plain"), (256, 512, 10240, 16, "gelu"), (833, 512, 8576, 32, "plain"),
        # what the rule gives to the three kernels: long and short K for the epilogue, one 256-row tile less than CUs
        (1100, 1024, 8192, 32, "plain"), (1024, 1024, 8064, 32, "plain"), (1100, 2048, 9216, 64, "qkv"), (1100, 1024, 9216, 64, "qkv"),
        (1100, 3584, 8192, 16, "gelu"), (1100, 1024, 8192, 32, "gelu"), (1100, 1536, 8192, 16, "swiglu"), (1100, 1024, 8192, 32, "swiglu"),
    ],
)  # fmt: skip
def test_wide_tiles_agree_bit_for_bit(dev, rows, k, n, rank, epilogue, dtype):
    print(f"case {rows} x {n}, K={k} R={rank} {epilogue} {dtype}", flush=True)
    want = _outputs(rows, k, n, rank, epilogue, dtype, dev, 1)
    for build in (0, -1):  # these tiles, and what the rules choose (where K is not split: bits agree)
        if build == -1 and rows < 833:
            continue
        for a, b in zip(_outputs(rows, k, n, rank, epilogue, dtype, dev, build), want):
            assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(
    "rows,k,n,rank,epilogue,unsigned",
    [
        (1, 1024, 128, 16, "plain", False), (33, 6144, 136, 0, "plain", False), (33, 6144, 136, 32, "plain", True), (257, 6144, 264, 48, "plain", False),
        (289, 2048, 4096, 32, "plain", False), (65, 1024, 384, 32, "qkv", False), (40, 6144, 128, 32, "gelu", False), (300, 6144, 256, 16, "swiglu", False),
        (2100, 2048, 4096, 32, "plain", False), (2100, 2048, 4096, 32, "plain", True),
    ],
)  # fmt: skip
def test_nibbles_relaid_out_agree_with_fp6_codes(dev, rows, k, n, rank, epilogue, unsigned, dtype):
    """Launches that turn the (M, K / 2) matrix, or its bytes in lane order, into fp6 codes first: the bits of the launch that was
    handed the codes.  (Unsigned activations of few rows are not re-laid-out; their bits agree all the same.)"""
    from nunchaku_rocm_amd import _lib, ops
    from nunchaku_rocm_amd.layout import block_activations, block_activations_f6, block_scales
    from nunchaku_rocm_amd.ops import gemm as G

    print(f"case {rows} x {n}, K={k} R={rank} {epilogue} unsigned={unsigned} {dtype}", flush=True)
    g = torch.Generator(device=dev).manual_seed(rows + k)
    lin = {name: t.to(dev) for name, t in O.make_svdq_linear(k, n, R=max(rank, 16), seed=k + n, dtype=dtype).items()}
    M = -(-rows // 32) * 32
    act = torch.randint(0, 256, (M, k // 2), generator=g, device=dev, dtype=torch.int16).to(torch.uint8)
    asc = (torch.rand(k // 64, M, generator=g, device=dev) * 0.1 + 0.01).to(dtype)
    kw = dict(wgt=lin["qweight"], wscales=lin["wscales"], lora_act_in=torch.randn(M, rank, generator=g, device=dev) if rank else None,
              lora_up=lin["proj_up"][:, :rank].contiguous() if rank else None, bias=lin["bias"], act_unsigned=unsigned)  # fmt: skip
    nq = n // 2 if epilogue == "swiglu" else n
    if epilogue == "qkv":
        kw.update(norm_q=torch.rand(128, generator=g, device=dev).to(dtype), norm_k=torch.rand(128, generator=g, device=dev).to(dtype),
                  rotary_emb=torch.randn(rows, 128, generator=g, device=dev))  # fmt: skip
    elif epilogue != "plain":
        kw.update(lora_down=torch.randn(nq, 16, generator=g, device=dev).to(dtype), fuse_swiglu=epilogue == "swiglu")
    wanted, real = [], G._act_scratch
    old, G.USE_WEIGHT_PLANES = G.USE_WEIGHT_PLANES, "all"
    G._act_scratch = lambda args, device: wanted.append(t := real(args, device)) or t
    try:
        results = []
        for a, s, mode in ((act, asc, 0), (block_activations(act.cpu()).to(dev), asc, 1), (block_activations_f6(act.cpu(), unsigned).to(dev), block_scales(asc.cpu()).to(dev), 3)):
            out = dict(out=torch.zeros(rows, n, dtype=dtype, device=dev)) if epilogue in ("plain", "qkv") else dict(
                qout=torch.zeros(M, nq * 3 // 4, dtype=torch.uint8, device=dev), oscales=torch.zeros(nq // 64, M, dtype=dtype, device=dev),
                lora_act_out=torch.zeros(M, 16, device=dev), qout_blocked=2)  # fmt: skip
            for _ in range(2):  # the second call is the native one
                ops.svdq_gemm_w4a4_cuda(act=a, ascales=s, act_blocked=mode, **kw, **out)
                torch.cuda.synchronize()
            results.append([t.view(torch.uint8).cpu() for t in out.values() if torch.is_tensor(t)])
    finally:
        G.USE_WEIGHT_PLANES, G._act_scratch = old, real
    few_unsigned = unsigned and _lib.load().svdq_gemm_w4a4_split_wavefronts(_lib.GemmArgs(wgt_planes=16, M=M, actual_m=rows, N=n, K=k, act_unsigned=1, R=rank), 0)
    assert len(wanted) == 4 and all((t is None) == bool(few_unsigned) for t in wanted)
    for other in results[1:]:
        assert all(torch.equal(x, y) for x, y in zip(results[0], other))
