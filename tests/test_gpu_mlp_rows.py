"""The fused MLPs compute whole blocks of 32 rows of their buffers and no more: the rows of the 256-row padding change nothing."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 32, 33, 255, 257, 333])
@pytest.mark.parametrize("kind", ["gelu", "swiglu"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_fused_mlp_on_blocks_of_32_rows(dev, rows, kind, dtype):
    """Against the same launches on buffers padded to 256 rows.  Where both take the same kernel the bits are the same; where fewer
    rows bring in the one that splits K, sums differ in their last bits and some int4 code by a step: of the 512 codes behind an output one
    in a hundred then moves it by 1 / 7 of a typical product, sqrt(5) / 7 / sqrt(512) = 1.4 %, of which the mean over rows is far less."""
    from nunchaku_rocm_amd import ops
    from nunchaku_rocm_amd.linear import SVDQW4A4Linear

    torch.manual_seed(rows)

    def linear(k, n, unsigned=False):
        lin = SVDQW4A4Linear(k, n, rank=32, bias=True, precision="int4", act_unsigned=unsigned, torch_dtype=dtype, device=dev)
        with torch.no_grad():
            lin.qweight.copy_(torch.randint(-128, 128, lin.qweight.shape, dtype=torch.int8))
            lin.wscales.copy_((torch.rand(lin.wscales.shape) * 0.02 + 0.005).to(dtype))
            for p in (lin.proj_up, lin.proj_down, lin.bias):
                p.copy_((torch.randn(p.shape) * 0.05).to(dtype))
            lin.smooth_factor.copy_((torch.rand(lin.smooth_factor.shape) + 0.5).to(dtype))
        return lin

    k, h = 1024, 512
    fc1, fc2 = linear(k, h if kind == "gelu" else 2 * h), linear(h, k, unsigned=kind == "gelu")
    x = torch.randn(rows, k).to(dtype).to(dev)
    with torch.no_grad():
        y = (ops.fused_gelu_mlp if kind == "gelu" else ops.fused_swiglu_mlp)(x.view(1, rows, k), fc1, fc2).view(rows, k)
        a, b = fc1.takes_blocked(rows), fc2.takes_blocked(rows)
        q, s, la = fc1.quantize(x, blocked=a)
        qo = torch.zeros(q.shape[0], h * (3 if b >= 2 else 2) // 4, dtype=torch.uint8, device=dev)
        so, lo = torch.zeros(h // 64, q.shape[0], dtype=dtype, device=dev), torch.zeros(q.shape[0], 32, device=dev)
        ops.svdq_gemm_w4a4_cuda(act=q, wgt=fc1.qweight, qout=qo, ascales=s, wscales=fc1.wscales, oscales=so, lora_act_in=la, lora_up=fc1.proj_up,
                                lora_down=fc2.proj_down, lora_act_out=lo, bias=fc1.bias, smooth_factor=fc2.smooth_factor,
                                act_unsigned=fc1.act_unsigned, fuse_swiglu=kind == "swiglu", act_blocked=a, qout_blocked=b)  # fmt: skip
        ref = fc2.forward_quant(qo, so, lo, torch.empty(rows, k, dtype=dtype, device=dev), act_blocked=b)
    rel = ((y.float() - ref.float()).norm() / ref.float().norm()).item()
    print(f"{kind} {rows} rows {dtype}: rel {rel:.1e}", flush=True)
    assert torch.isfinite(ref).all() and rel <= 1.4e-2
