"""LoRA-up rows of any 32-bit stride: 32 of them that reach past 4 GB give the bits of the same rows in one piece."""

import pytest
import torch

from oracle import svdq_oracle as O

pytestmark = pytest.mark.gpu

LD = (1 << 26) + 8  # 31 rows of 2 bytes each: more than 32 bits of offset


@pytest.fixture(scope="module")
def far(dev):
    yield torch.empty(136 * LD, dtype=torch.int16, device=dev)  # 18 GB, of which the tests touch a few KB
    torch.cuda.empty_cache()


# the int8 loop, nibbles and fp6 codes in both builds of the fp8 loop (0 with codes and scales: 256-row tiles), K split over wavefronts
@pytest.mark.parametrize("planes,blocked,build", [("none", 0, -1), ("all", 0, 0), ("all", 0, 1), ("all", 2, 0), ("all", 3, 1), ("all", 3, 0), ("all", 3, -1)])
@pytest.mark.parametrize("n,rank,epilogue", [(136, 16, "plain"), (136, 48, "plain"), (128, 32, "gelu")])
def test_rows_beyond_32_bit_offsets(dev, far, planes, blocked, build, n, rank, epilogue, monkeypatch):
    from nunchaku_rocm_amd import ops
    from nunchaku_rocm_amd.ops import gemm as G

    print(f"case {planes} {blocked} {build} {n} {rank} {epilogue}", flush=True)
    M, k, dtype = 160, 512, torch.bfloat16
    lin = {name: t.to(dev) for name, t in O.make_svdq_linear(k, n, R=rank, seed=rank, dtype=dtype).items()}
    x = torch.randn(M, k, device=dev).to(dtype)
    q, s, la = ops.svdq_quantize_w4a4_act_fuse_lora_cuda(x, lora_down=lin["proj_down"], smooth=lin["smooth_factor"], pad_size=32, out_blocked=blocked)
    rows = far.view(dtype).as_strided((n, rank), (LD, 1))
    rows.copy_(lin["proj_up"])
    monkeypatch.setattr(G, "USE_WEIGHT_PLANES", planes)
    G.set_fp8_loop_variant(build)
    outs = []
    try:
        for up in (rows, lin["proj_up"]):
            kw = dict(act=q, wgt=lin["qweight"], ascales=s, wscales=lin["wscales"], lora_act_in=la, lora_up=up, bias=lin["bias"], act_blocked=blocked)
            if epilogue == "plain":
                kw["out"] = torch.zeros(M, n, dtype=dtype, device=dev)
            else:
                kw.update(qout=torch.zeros(M, n // 2, dtype=torch.uint8, device=dev), oscales=torch.zeros(n // 64, M, dtype=dtype, device=dev))
            for _ in range(3):  # the first makes the working copy of the weight, the last finds it complete: Python's checks and the native ones
                ops.svdq_gemm_w4a4_cuda(**kw)
                torch.cuda.synchronize()
                outs.append([kw[name].view(torch.uint8).clone() for name in ("out", "qout", "oscales") if name in kw])
    finally:
        G.set_fp8_loop_variant(-1)
    for out in outs:
        assert all(torch.equal(a, b) for a, b in zip(out, outs[-1])) and out[0].any()
