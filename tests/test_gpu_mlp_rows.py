"""The fused MLPs compute whole blocks of 32 rows of their buffers and no more: the rows of the 256-row padding change nothing."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,h", [(1, 512), (32, 512), (33, 512), (255, 512), (257, 512), (333, 512), (33, 5120)])  # the last: fc1 splits K for 64 rows, not for 256
@pytest.mark.parametrize("kind", ["gelu", "swiglu"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_fused_mlp_on_blocks_of_32_rows(dev, rows, h, kind, dtype):
    """Against the same launches on buffers padded to 256 rows.  Where both split K alike the bits are the same; where fewer
    rows bring in the kernel that splits K, sums differ in their last bits and some int4 code by a step: of the (512 and more) codes behind an output one
    in a hundred then moves it by 1 / 7 of a typical product, sqrt(5) / 7 / sqrt(512) = 1.4 %, of which the mean over rows is far less.
    No row has more than 25 such codes (five on average): sqrt(25) / 7 / sqrt(512) = 3.2 %."""
    from nunchaku_rocm_amd import _lib, ops
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

    k = 1024
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

    def splits(pad):  # over how many wavefronts the two launches split K with buffers of `pad` rows
        common = dict(wgt_planes=16, M=pad, R=32, act_blocked=2, ascales_blocked=1, dtype=_lib.dtype_code(dtype))
        epilogue = _lib.EPI_GELU_QUANT if kind == "gelu" else _lib.EPI_SWIGLU_QUANT
        both = (_lib.GemmArgs(N=fc1.out_features, K=k, R2=32, actual_m=pad, epilogue=epilogue, **common), _lib.GemmArgs(N=k, K=h, actual_m=rows, **common))
        return [_lib.load().svdq_gemm_w4a4_split_wavefronts(args, 0) for args in both]

    same = splits(-(-rows // 32) * 32) == splits(q.shape[0])
    diff, ref = y.float() - ref.float(), ref.float()
    rel, row = (diff.norm() / ref.norm()).item(), (diff.norm(dim=1) / ref.norm(dim=1)).max().item()
    print(f"{kind} {rows} rows, hidden {h}, {dtype}: rel {rel:.1e}, worst row {row:.1e}{', same bits' if same else ''}", flush=True)
    assert torch.isfinite(ref).all() and same == (h == 512) and rel <= (0.0 if same else 1.4e-2) and row <= (0.0 if same else 3.2e-2)
