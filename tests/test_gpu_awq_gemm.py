"""The AWQ GEMM that decodes its weight inside the kernel (``svdq_awq_gemm_w4a16``) at the edges of its tiles."""

import pytest
import torch

from oracle import svdq_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(
    "m,n,k,group_size,tile",
    [
        (1, 4, 64, 64, (32, 128)),  # less than one tile either way, half a stage of k
        (3, 96, 256, 32, (32, 128)),  # a scale group per half of a lane's group
        (33, 100, 192, 64, (32, 128)),  # one row past a block, channels that fill no slice, an odd number of groups of 64
        (65, 132, 448, 64, (32, 128)),  # three stages and a half
        (130, 260, 1344, 96, (32, 128)),  # ten stages and a half, group 96
        (2048, 128, 128, 128, (32, 128)),  # the most rows
        (300, 4100, 640, 128, (64, 128)),  # remainders of rows and channels
        (257, 8196, 64, 64, (128, 128)),  # one row and four channels past the last whole tile, half a stage
        (333, 10244, 448, 32, (128, 128)),  # three stages and a half
        (666, 4096, 896, 128, (128, 128)),
        (500, 8200, 896, 64, (128, 256)),
        (510, 10244, 768, 128, (128, 256)),
    ],
)
def test_awq_gemm_kernel_against_the_decoded_weight(m, n, k, group_size, tile, dtype, monkeypatch):
    from nunchaku_rocm_amd import _lib, ops
    from nunchaku_rocm_amd.ops import gemv

    print(f"case m={m} n={n} k={k} group_size={group_size} {dtype}", flush=True)
    assert divmod(_lib.load().svdq_awq_gemm_tile(m, n, 0), 1 << 16) == tile
    monkeypatch.setattr(gemv, "awq_dequantize", None)  # the library product's first step
    dev = torch.device("cuda", 0)
    g = torch.Generator().manual_seed(m + n)
    q = torch.randint(0, 16, (n, k), generator=g, dtype=torch.int32)
    s = (torch.rand(k // group_size, n, generator=g) * 0.015 + 0.005).to(dtype)
    z = (-torch.randint(0, 16, s.shape, generator=g).float() * s.float()).to(dtype)
    x = torch.randn(m, k, generator=g).to(dtype)
    packed = O.awq_pack(q)
    w = O.awq_dequantize(packed, s, z, group_size).float()
    out = ops.awq_gemm_w4a16(x.to(dev), packed.view(torch.int32).to(dev), s.to(dev), z.to(dev), group_size=group_size).cpu()
    ref = (x.double() @ w.double().t()).float()
    # one rounding to the 16-bit type, and k fp32 additions of exact products in any order
    bound = ref.abs() * (2.0**-8 if dtype == torch.bfloat16 else 2.0**-11) + k * 2.0**-24 * (x.float().abs() @ w.abs().t()) + 1e-6
    assert out.shape == (m, n) and out.dtype == dtype
    assert ((out.float() - ref).abs() <= bound).all()
