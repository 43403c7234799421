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
    ],
)  # fmt: skip
def test_wide_tiles_agree_bit_for_bit(dev, rows, k, n, rank, epilogue, dtype):
    print(f"case {rows} x {n}, K={k} R={rank} {epilogue} {dtype}", flush=True)
    want = _outputs(rows, k, n, rank, epilogue, dtype, dev, 1)
    for build in (0, -1):  # these tiles, and what the rules choose (where K is not split: bits agree)
        if build == -1 and rows < 1024:
            continue
        for a, b in zip(_outputs(rows, k, n, rank, epilogue, dtype, dev, build), want):
            assert torch.equal(a, b)
