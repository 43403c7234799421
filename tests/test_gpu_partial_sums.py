"""The requantizing epilogues' LoRA-down result is the sum of the column tiles' partial products in tile order, bit for bit."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# tiles: fewer than a batch of loads, whole batches, batches and a rest of eights, of eights and ones, of ones
@pytest.mark.parametrize("n", [128, 896, 4096, 12288, 6144, 5376, 4352])
@pytest.mark.parametrize("rows,rank", [(16, 16), (48, 32), (272, 48), (2048, 32), (2064, 32)])  # up to, and beyond, a workgroup of 256 columns to a CU
@pytest.mark.parametrize("epilogue", ["gelu", "swiglu"])
def test_sum_in_tile_order(dev, monkeypatch, n, rows, rank, epilogue):
    from nunchaku_rocm_amd import _lib, ops
    from nunchaku_rocm_amd.ops import gemm as G

    print(f"case {rows} x {n} R2={rank} {epilogue}", flush=True)
    k, nq = 128, n // 2 if epilogue == "swiglu" else n
    g = torch.Generator(device=dev).manual_seed(n + rows)
    byte = lambda *s: torch.randint(0, 256, s, generator=g, device=dev, dtype=torch.int16).to(torch.uint8)  # noqa: E731
    val = lambda *s: (torch.rand(*s, generator=g, device=dev) * 0.02 + 0.01).to(torch.bfloat16)  # noqa: E731
    result = torch.full((rows, rank), float("nan"), device=dev)
    kw = dict(act=byte(rows, k // 2), wgt=byte(n, k // 2), ascales=val(k // 64, rows), wscales=val(k // 64, n), fuse_swiglu=epilogue == "swiglu",
              qout=byte(rows, nq // 2), oscales=val(nq // 64, rows), lora_down=torch.randn(nq, rank, generator=g, device=dev).to(torch.bfloat16),
              lora_act_out=result)  # fmt: skip
    native, kept = _lib.host(), []

    class Host:  # the launch's scratch memory is what the native code returns
        def __getattr__(self, name):
            return getattr(native, name)

        def gemm(self, *a):
            kept.append(native.gemm(*a))
            return kept[-1]

    monkeypatch.setattr(_lib, "host", lambda: Host())
    monkeypatch.setattr(G, "USE_WEIGHT_PLANES", "all")
    for _ in range(3):  # the first makes the copies of the weights, the second finds them complete
        ops.svdq_gemm_w4a4_cuda(**kw)
        torch.cuda.synchronize()
    want = torch.zeros(rows, rank, device=dev)
    for part in kept[-1].view(-(-n // 128), rows, rank):
        want = want + part
    assert want.abs().max() > 0 and torch.equal(result, want)
