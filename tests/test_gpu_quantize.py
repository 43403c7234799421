"""GPU parity of the activation quantizer against the CPU oracle: int4 codes and 16-bit scales bit-exact, LoRA-down
within fp32 accumulation-order noise, pad rows untouched, deterministic."""

import pytest
import torch

from oracle import svdq_oracle as O
from parity_bars import assert_requantized_like_the_reference

pytestmark = pytest.mark.gpu


def _run(x, lin, dev, R, smooth=True, unsigned=False, shift=0.0, pad=0):
    from nunchaku_rocm_amd.ops.quantize import quantize_w4a4_act_fuse_lora

    M, K = x.shape
    ld = lin["proj_down"][:, :R].contiguous() if R else None
    sm = lin["smooth_factor"] if smooth else None
    out = torch.full((M + pad, K // 2), 0xEE, dtype=torch.uint8, device=dev)
    osc = torch.full((K // 64, M + pad), 7.0, dtype=x.dtype, device=dev)
    la = torch.full((M + pad, max(R, 1)), 7.0, dtype=torch.float32, device=dev)[:, :R] if R else None
    quantize_w4a4_act_fuse_lora(
        x.to(dev), out, osc, ld.to(dev) if R else None, la, sm.to(dev) if smooth else None,
        shift_value=shift, unsigned=unsigned,
    )  # fmt: skip
    torch.cuda.synchronize()
    ref = O.quantize_act(x, ld, sm, unsigned=unsigned, shift=shift)
    return (out.cpu(), osc.cpu(), la.cpu() if R else None), ref


@pytest.mark.parametrize("M,K,R", [(1, 128, 16), (16, 256, 32), (130, 384, 48), (257, 3072, 32), (64, 512, 0), (33, 1024, 288),
                                   (40, 640, 64), (18, 3072, 96), (50, 512, 160)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_codes_and_scales_bit_exact(dev, M, K, R, dtype):
    print(f"case M={M} K={K} R={R} {dtype}", flush=True)
    x = O.make_activations(M, K, seed=M + K, dtype=dtype)
    lin = O.make_svdq_linear(K, 64, R=max(R, 16), seed=K, dtype=dtype)
    (out, osc, la), (rp, rs, rl, _) = _run(x, lin, dev, R, pad=5)
    assert torch.equal(out[:M], rp)
    assert torch.equal(osc[:, :M].view(torch.int16), rs.view(torch.int16))
    assert (out[M:] == 0xEE).all() and (osc[:, M:] == 7.0).all()  # pad rows never written
    if R:
        ref64 = x.double() @ lin["proj_down"][:, :R].double()
        assert (la[:M].double() - ref64).abs().max() <= 2e-5 * ref64.abs().max()
        assert (la[M:] == 7.0).all()


@pytest.mark.parametrize("M", [2064, 4112, 4640, 8208])
def test_every_grid_layout_bit_exact(dev, M):
    """The launcher picks 16- or 32-row workgroups and, where CUs would idle, a further workgroup row that only
    quantizes while the others only project (see quantize_grid_y): 2064 rows = 16-row workgroups doing both, 4112 =
    32-row doing both on a 256-CU part, 4640 = 32-row just past the split's limit, 8208 = 16-row again; the small
    shapes of the other tests and M = 4608 take the split layouts."""
    print(f"case M={M}", flush=True)
    K, R = 128, 32
    x = O.make_activations(M, K, seed=M, dtype=torch.bfloat16)
    lin = O.make_svdq_linear(K, 64, R=R, seed=K)
    (out, osc, la), (rp, rs, rl, _) = _run(x, lin, dev, R)
    assert torch.equal(out[:M], rp)
    assert torch.equal(osc[:, :M].view(torch.int16), rs.view(torch.int16))
    ref64 = x.double() @ lin["proj_down"][:, :R].double()
    assert (la[:M].double() - ref64).abs().max() <= 2e-5 * ref64.abs().max()


@pytest.mark.parametrize("M,K", [(512, 3072), (1024, 3072), (96, 320), (48, 704), (2048, 192)])
def test_quantize_only_rows_share_the_groups(dev, M, K):
    """Where CUs are left over the launcher adds up to three workgroup rows that only quantize, each a slice of the
    groups (quantize_grid_y): group counts that do and do not divide by the number of slices, fewer groups than
    wavefronts in a slice, and the largest row count that still takes three slices on a 256-CU part."""
    print(f"case M={M} K={K}", flush=True)
    R = 32
    x = O.make_activations(M, K, seed=M + K, dtype=torch.bfloat16)
    lin = O.make_svdq_linear(K, 64, R=R, seed=K)
    (out, osc, la), (rp, rs, rl, _) = _run(x, lin, dev, R)
    assert torch.equal(out[:M], rp)
    assert torch.equal(osc[:, :M].view(torch.int16), rs.view(torch.int16))
    ref64 = x.double() @ lin["proj_down"][:, :R].double()
    assert (la[:M].double() - ref64).abs().max() <= 2e-5 * ref64.abs().max()


@pytest.mark.parametrize("smooth", [True, False])
def test_unsigned_with_shift_bit_exact(dev, smooth):
    M, K = 96, 512
    g = torch.Generator().manual_seed(3)
    x = (torch.nn.functional.gelu(torch.randn(M, K, generator=g) * 2, approximate="tanh")).to(torch.bfloat16)
    lin = O.make_svdq_linear(K, 64, seed=4)
    (out, osc, la), (rp, rs, rl, _) = _run(x, lin, dev, 32, smooth=smooth, unsigned=True, shift=0.171875)
    assert torch.equal(out, rp)
    assert torch.equal(osc.view(torch.int16), rs.view(torch.int16))


def test_zero_groups_and_ties(dev):
    x = torch.zeros(16, 128, dtype=torch.bfloat16)
    x[1, :64] = torch.arange(64).float().sub(32).mul(0.5).clamp(-7, 7).to(torch.bfloat16)  # exact .5 ties at scale 1
    x[2, 64:] = -3.0
    lin = O.make_svdq_linear(128, 64, seed=5)
    (out, osc, _), (rp, rs, _, _) = _run(x, lin, dev, 0, smooth=False)
    assert torch.equal(out, rp) and torch.equal(osc.view(torch.int16), rs.view(torch.int16))
    (out, osc, _), (rp, rs, _, _) = _run(x, lin, dev, 0, smooth=False, unsigned=True)
    assert torch.equal(out, rp) and torch.equal(osc.view(torch.int16), rs.view(torch.int16))


def test_kernel_multiplies_by_the_reciprocal(dev):
    """Inputs on which ``x * (1 / scale)`` and ``x / scale`` give different codes; the expected codes come from exact
    rational arithmetic (tests/golden/rcp_order_vectors.py)."""
    from nunchaku_rocm_amd import ops
    from test_oracle_pins import _rcp_order_input

    xb, want = _rcp_order_input()
    xp = torch.zeros(16, 64, dtype=torch.bfloat16)
    xp[: xb.shape[0]] = xb
    q, _, _ = ops.svdq_quantize_w4a4_act_fuse_lora_cuda(xp.to(dev))
    codes = O.unpack_int4(q.cpu(), True)
    for i, w in enumerate(want):
        assert int(codes[i, 1 + i]) == w and int(codes[i, 0]) == 7


def test_full_size_qkv_input_bit_exact_and_deterministic(dev):
    """The benchmark configuration: M=4608, K=3072, R=32, outlier channels, smooth U(0.5, 4)."""
    M, K = 4608, 3072
    x = O.make_activations(M, K, seed=1)
    lin = O.make_svdq_linear(K, 64, seed=0)
    (out, osc, la), (rp, rs, rl, _) = _run(x, lin, dev, 32)
    assert torch.equal(out, rp)
    assert torch.equal(osc.view(torch.int16), rs.view(torch.int16))
    assert (la - rl).abs().max() <= 2e-5 * rl.abs().max()
    (out2, osc2, la2), _ = _run(x, lin, dev, 32)
    assert torch.equal(out, out2) and torch.equal(osc.view(torch.int16), osc2.view(torch.int16)) and torch.equal(la, la2)


def test_operator_pads_rows_like_the_reference(dev):
    from nunchaku_rocm_amd import ops

    M, K = 300, 256
    x = O.make_activations(M, K, seed=9).to(dev)
    lin = O.make_svdq_linear(K, 64, seed=9)
    out, osc, la = ops.svdq_quantize_w4a4_act_fuse_lora_cuda(x, lora_down=lin["proj_down"].to(dev), smooth=lin["smooth_factor"].to(dev))
    assert out.shape == (512, K // 2) and osc.shape == (K // 64, 512) and la.shape == (512, 32) and la.dtype == torch.float32
    rp, rs, rl, _ = O.quantize_act(x.cpu(), lin["proj_down"], lin["smooth_factor"])
    assert torch.equal(out[:M].cpu(), rp) and torch.equal(osc[:, :M].cpu().view(torch.int16), rs.view(torch.int16))


def test_fuse_glu_close_to_oracle(dev):
    from nunchaku_rocm_amd.ops.quantize import quantize_w4a4_act_fuse_lora

    M, K = 32, 512
    g = torch.Generator().manual_seed(6)
    x = torch.randn(M, 2 * K, generator=g).to(torch.bfloat16)
    out, osc, _ = quantize_w4a4_act_fuse_lora(x.to(dev), fuse_glu=True)
    rp, rs, _, rc = O.quantize_act(x, fuse_glu=True)
    codes = O.unpack_int4(out.cpu(), True)
    d = (codes - rc).abs()
    assert d.max() <= 1 and ((d > 0).float().mean() < 1e-5 or (d > 0).sum() <= 1)  # exp() differs between libraries
    assert ((osc.cpu().float() - rs.float()).abs() <= rs.float().abs() * 2**-7 + 1e-9).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,R,batches", [(48, 256, 32, 1), (130, 384, 48, 1), (64, 512, 16, 2), (4608, 3072, 32, 1), (96, 1024, 0, 3),
                                           (64, 512, 128, 2)])
def test_norm_modulate_prologue(dev, M, K, R, batches, dtype):
    """LayerNorm + scale + shift applied inside the quantizer: codes, scales and the LoRA-down product are those of
    the oracle's quantizer fed with the oracle's layernorm_modulate output.  exp-free arithmetic, but the row
    statistics are summed in another order than on the CPU: a 16-bit rounding may flip, so codes may differ by one
    step on a small fraction of entries (the contract of the fused GELU epilogue,
    tests/triton/test_native_epilogues.py:246-253)."""
    from nunchaku_rocm_amd import ops

    print(f"case M={M} K={K} R={R} batches={batches} {dtype}", flush=True)
    g = torch.Generator().manual_seed(M + K)
    x = (torch.randn(M, K, generator=g) * 1.7 + 0.3).to(dtype)
    scale = (1 + 0.3 * torch.randn(batches, K, generator=g)).to(dtype)
    shift = (0.2 * torch.randn(batches, K, generator=g)).to(dtype)
    lin = O.make_svdq_linear(K, 64, R=max(R, 16), seed=K, dtype=dtype)
    ld = lin["proj_down"][:, :R].contiguous() if R else None
    q, s, la = ops.svdq_quantize_w4a4_act_fuse_lora_cuda(x.to(dev), lora_down=None if ld is None else ld.to(dev),
                                                          smooth=lin["smooth_factor"].to(dev), norm=(scale.to(dev), shift.to(dev)))  # fmt: skip
    torch.cuda.synchronize()
    xm = O.layernorm_modulate(x, scale, shift)
    rq, rs, rl, rc = O.quantize_act(xm, ld, lin["smooth_factor"])
    # a group maximum that flipped by one 16-bit step moves the stored scale by up to two of its own steps
    assert_requantized_like_the_reference(O.unpack_int4(q[:M].cpu(), True), rc, s[:, :M].cpu(), rs.to(dtype), dtype, scale_steps=2.01)
    if R:
        assert (la[:M].cpu() - rl).abs().max() <= 1e-2 * rl.abs().max()
    # statistics computed once and passed in give the same bits as computing them inside the call
    st = ops.layer_norm_stats(x.to(dev))
    ref_mean = x.float().mean(dim=1)
    assert (st[:, 0].cpu() - ref_mean).abs().max() <= 1e-5 * (1 + ref_mean.abs().max())
    q2, s2, _ = ops.svdq_quantize_w4a4_act_fuse_lora_cuda(x.to(dev), lora_down=None if ld is None else ld.to(dev),
                                                          smooth=lin["smooth_factor"].to(dev), norm=(scale.to(dev), shift.to(dev), st))  # fmt: skip
    assert torch.equal(q2[:M], q[:M]) and torch.equal(s2[:, :M].view(torch.int16), s[:, :M].view(torch.int16))
    # scale / shift as interleaved slices of one projection output (element stride 6), used where they lie
    emb = torch.zeros(batches, K, 6, dtype=dtype, device=dev)
    emb[:, :, 1], emb[:, :, 0] = scale.to(dev), shift.to(dev)
    q3, s3, _ = ops.svdq_quantize_w4a4_act_fuse_lora_cuda(x.to(dev), lora_down=None if ld is None else ld.to(dev),
                                                          smooth=lin["smooth_factor"].to(dev), norm=(emb[:, :, 1], emb[:, :, 0], st))  # fmt: skip
    assert torch.equal(q3[:M], q[:M]) and torch.equal(s3[:, :M].view(torch.int16), s[:, :M].view(torch.int16))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,R", [(1, 64, 16), (17, 512, 32), (33, 4096, 48), (16, 4160, 16), (31, 8192, 0), (18, 8256, 32), (4100, 128, 16)])
def test_statistics_inside_the_quantizer(dev, M, K, R, dtype):
    """The row statistics a norm prologue computes for itself are layer_norm_stats' own, bit for bit: rows kept in registers
    up to K = 4096 there and 8192 here, read twice beyond; ends of the row blocks; one and several workgroups to a row block."""
    from nunchaku_rocm_amd import ops

    g = torch.Generator(device=dev).manual_seed(M + K)
    x = (torch.randn(M, K, generator=g, device=dev) * 1.7 + 0.3).to(dtype)
    scale, shift = (1 + 0.3 * torch.randn(K, generator=g, device=dev)).to(dtype), (0.2 * torch.randn(K, generator=g, device=dev)).to(dtype)
    down = torch.randn(K, R, generator=g, device=dev).to(dtype) if R else None
    for eps in (1e-6, 0.25, 0.0):
        own = ops.svdq_quantize_w4a4_act_fuse_lora_cuda(x, lora_down=down, norm=(scale, shift), norm_eps=eps)
        given = ops.svdq_quantize_w4a4_act_fuse_lora_cuda(x, lora_down=down, norm=(scale, shift, ops.layer_norm_stats(x, eps)), norm_eps=eps)
        torch.cuda.synchronize()
        assert torch.equal(own[0][:M], given[0][:M]) and torch.equal(own[1][:, :M].view(torch.int16), given[1][:, :M].view(torch.int16))
        assert torch.equal(own[2][:M], given[2][:M])


@pytest.mark.parametrize("M,K", [(1, 64), (33, 512), (17, 8256)])
def test_statistics_at_any_float(dev, M, K):
    """Row statistics are written and read where they lie: four bytes of alignment are enough."""
    from nunchaku_rocm_amd import _lib, ops

    x = (torch.randn(M, K, device=dev) * 3 + 1).to(torch.bfloat16)
    scale, shift = torch.rand(K, device=dev).to(x.dtype) + 0.5, torch.rand(K, device=dev).to(x.dtype)
    want = ops.layer_norm_stats(x)
    buf = torch.full((2 * M + 2,), -7.0, device=dev)
    stats = buf[1:-1].view(M, 2)
    assert stats.data_ptr() % 8 == 4
    _lib.check(_lib.load().svdq_row_stats(x.data_ptr(), stats.data_ptr(), M, K, K, _lib.dtype_code(x.dtype), 1e-6, _lib.stream_of(x)))
    assert torch.equal(stats, want) and buf[0] == buf[-1] == -7.0
    for a, b in zip(*(ops.quantize_w4a4_act_fuse_lora(x, norm=(scale, shift, s))[:2] for s in (stats, want))):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


@pytest.mark.parametrize("eps", [1e-50, 1e-46, 1e-44])
def test_norm_with_an_eps_that_32_bits_lose(dev, eps):
    """The norm is applied, with the eps that 32 bits hold, by native and Python checks alike."""
    from nunchaku_rocm_amd import ops

    x = (torch.randn(33, 512, device=dev) * 3 + 1).to(torch.bfloat16)
    scale, shift = torch.rand(512, device=dev).to(x.dtype) + 0.5, torch.rand(512, device=dev).to(x.dtype)
    want = ops.quantize_w4a4_act_fuse_lora(x, norm=(scale, shift, ops.layer_norm_stats(x, eps)))
    out = [ops.quantize_w4a4_act_fuse_lora(x, norm=(scale, shift), norm_eps=eps)]
    buf = torch.zeros_like(want[0]), torch.zeros_like(want[1])
    out.append(ops.quantize_w4a4_act_fuse_lora(x, *buf, norm=(scale, shift), norm_eps=eps))
    plain = ops.quantize_w4a4_act_fuse_lora(x)
    torch.cuda.synchronize()
    for q, s, _ in out:
        assert torch.equal(q, want[0]) and torch.equal(s, want[1]) and not torch.equal(q, plain[0])


@pytest.mark.parametrize("M,K,R,launches", [(4096, 128, 64, 1), (4097, 128, 64, 2), (17, 4096, 32, 1), (17, 4160, 32, 2), (512, 192, 256, 1), (530, 192, 256, 2)])
def test_statistics_in_a_launch_of_their_own(dev, monkeypatch, M, K, R, launches):
    """Where a statistics launch in front is the faster way it is made, by native and Python checks alike; the bits are the same."""
    from nunchaku_rocm_amd import _lib, ops
    from nunchaku_rocm_amd.ops import quantize as Q

    g = torch.Generator(device=dev).manual_seed(M + K)
    x = (torch.randn(M, K, generator=g, device=dev) * 1.7 + 0.3).to(torch.bfloat16)
    scale, shift = (1 + 0.3 * torch.randn(K, generator=g, device=dev)).to(x.dtype), (0.2 * torch.randn(K, generator=g, device=dev)).to(x.dtype)
    down = torch.randn(K, R, generator=g, device=dev).to(x.dtype)
    lib, seen = _lib.load(), []

    class Lib:
        def __getattr__(self, name):
            if name in ("svdq_row_stats", "svdq_quantize_act"):
                seen.append(name)
            return getattr(lib, name)

    monkeypatch.setattr(_lib, "load", lambda: Lib())
    run = lambda: ops.svdq_quantize_w4a4_act_fuse_lora_cuda(x, lora_down=down, norm=(scale, shift))  # noqa: E731
    results = []
    for _ in range(3):  # the third call finds its copy of the weight made and complete: the native checks
        seen.clear()
        results.append(run())
        torch.cuda.synchronize()
        assert seen == ["svdq_row_stats", "svdq_quantize_act"][2 - launches :]
    monkeypatch.setattr(Q, "_stats_first", lambda args, device: None)
    results.append(run())  # its own, whatever the size
    torch.cuda.synchronize()
    for r in results[1:]:
        assert torch.equal(r[0][:M], results[0][0][:M]) and torch.equal(r[1][:, :M].view(torch.int16), results[0][1][:, :M].view(torch.int16))
        assert torch.equal(r[2][:M], results[0][2][:M])


def test_plain_aliases_and_quantized_product(dev):
    """quantize_w4a4_act / quantize_w4a4_wgt (no smoothing, no LoRA): bit-equal to the oracle, and their outputs are the
    GEMM's natural-layout operands: the int4 product tracks the dense one within the quantization noise."""
    from nunchaku_rocm_amd import ops

    g = torch.Generator().manual_seed(77)
    M, N, K = 96, 160, 512
    x = torch.randn(M, K, generator=g).to(torch.bfloat16)
    w = (torch.randn(N, K, generator=g) * 0.05).to(torch.bfloat16)
    qa, sa = ops.quantize_w4a4_act(x.to(dev))
    qw, sw = ops.quantize_w4a4_wgt(w.to(dev))
    torch.cuda.synchronize()
    ra = O.quantize_act(x)
    rw = O.quantize_act(w)
    assert qa.shape == (M, K // 2) and sa.shape == (K // 64, M) and qw.shape == (N, K // 2) and sw.shape == (K // 64, N)
    assert torch.equal(qa.cpu(), ra[0]) and torch.equal(sa.cpu(), ra[1])
    assert torch.equal(qw.cpu(), rw[0]) and torch.equal(sw.cpu(), rw[1])
    out = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    ops.svdq_gemm_w4a4_cuda(qa, qw, out=out, ascales=sa, wscales=sw)
    torch.cuda.synchronize()
    ref = O.gemm_w4a4(ra[0], rw[0], ra[1], rw[1])
    assert O.max_rel_err(out.cpu(), ref) <= 1e-2
    dense = x.float() @ w.float().t()
    # int4 x int4 with per-group absmax scales: relative error of a dot product of 512 terms is a few percent
    assert O.cosine(out.cpu().float(), dense) >= 0.98
    with pytest.raises(NotImplementedError):
        ops.quantize_w4a4_wgt(w.to(dev), fp4=True)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,R", [(48, 256, 32), (130, 384, 0), (257, 1024, 48)])
def test_gelu_prologue(dev, M, K, R, dtype):
    """fuse_gelu: tanh-GELU, LoRA-down on its rounded value, + 0.171875, smoothing, unsigned codes.  exp() differs
    between implementations by an ulp, so codes carry the reference's own bar: off by at most one, rarely."""
    from nunchaku_rocm_amd.ops.quantize import quantize_w4a4_act_fuse_lora

    print(f"case M={M} K={K} R={R} {dtype}", flush=True)
    lin = O.make_svdq_linear(K, 64, R=max(R, 16), seed=K + R, dtype=dtype)
    x = (O.make_activations(M, K, seed=M, dtype=dtype).float() * 0.3).to(dtype)
    ld = lin["proj_down"][:, :R].contiguous() if R else None
    sm = lin["smooth_factor"]
    out, osc, la = quantize_w4a4_act_fuse_lora(x.to(dev), lora_down=ld.to(dev) if R else None, smooth=sm.to(dev),
                                               fuse_gelu=True, shift_value=O.GELU_SHIFT, unsigned=True)  # fmt: skip
    torch.cuda.synchronize()
    rp, rs, rl, rc = O.quantize_act(x, ld, sm, unsigned=True, shift=O.GELU_SHIFT, fuse_gelu=True)
    assert_requantized_like_the_reference(O.unpack_int4(out.cpu(), False), rc, osc.cpu(), rs.to(dtype), dtype)
    if R:
        assert (la.cpu() - rl).abs().max() <= 1e-2 * rl.abs().max()
    with pytest.raises(NotImplementedError):
        quantize_w4a4_act_fuse_lora(torch.zeros(16, 128, dtype=dtype, device=dev), fuse_gelu=True, fuse_glu=True)


def test_full_size_invariants(dev):
    """On the whole (4608, 3072) input, on the GPU: multiplying the input by two leaves the codes alone and doubles the
    scales and the LoRA hidden state exactly; permuting the rows permutes every output."""
    from nunchaku_rocm_amd.ops.quantize import quantize_w4a4_act_fuse_lora

    M, K, R = 4608, 3072, 32
    lin = O.make_svdq_linear(K, 64, R=R, seed=3)
    x = O.make_activations(M, K, seed=4).to(dev)
    ld, sm = lin["proj_down"].to(dev), lin["smooth_factor"].to(dev)
    q0, s0, l0 = quantize_w4a4_act_fuse_lora(x, lora_down=ld, smooth=sm)
    q1, s1, l1 = quantize_w4a4_act_fuse_lora(x * 2, lora_down=ld, smooth=sm)
    assert torch.equal(q0, q1) and torch.equal(s1, s0 * 2) and torch.equal(l1, l0 * 2)
    pm = torch.randperm(M, generator=torch.Generator(device=dev).manual_seed(5), device=dev)
    q2, s2, l2 = quantize_w4a4_act_fuse_lora(x[pm].contiguous(), lora_down=ld, smooth=sm)
    assert torch.equal(q2, q0[pm]) and torch.equal(s2, s0[:, pm]) and torch.equal(l2, l0[pm])
    # every group uses its full range: the largest code magnitude of a group with a non-zero scale is 7 (or -8 never
    # without a 7-magnitude partner: |x| / (absmax / 7) <= 7)
    codes = O.unpack_int4(q0.cpu(), True).view(M, K // 64, 64)
    nz = s0.cpu().t().float() != 0
    assert bool((codes.abs().amax(dim=2)[nz] == 7).all()) and int(codes.min()) >= -7


@pytest.mark.parametrize("norm", [False, True, "given"])
@pytest.mark.parametrize("M,K,R", [(333, 2048, 64), (1201, 3072, 48), (2048, 1536, 32), (2064, 1536, 32), (4096, 1536, 16), (2048, 1472, 32), (4097, 256, 32), (4100, 192, 32), (4112, 128, 32), (5120, 320, 32),
                                   (5136, 512, 16), (5456, 256, 32), (5457, 256, 32), (8208, 512, 32), (4112, 256, 48), (4608, 64, 32)])  # fmt: skip
def test_row_blocks_behind_the_last_whole_round(dev, M, K, R, norm):
    """On 256 CUs: sixteen wavefronts with the norm prologue up to one workgroup to a CU (4096 rows; 2048: with rows that only quantize)
    from K = 1536 on, four (to 5120 rows) and three (to 5456) workgroups to a block of the rest, three where there are three groups (192),
    none with fewer (128, 64) or a second chunk of ranks -- against the same rows, normalised before, a few blocks at a time, which take none of these routes."""
    from nunchaku_rocm_amd import ops
    from nunchaku_rocm_amd.layout import block_scales

    print(f"case M={M} K={K} R={R} norm={norm}", flush=True)
    g = torch.Generator().manual_seed(M + K)
    T = torch.bfloat16
    x = O.make_activations(M, K, seed=M, dtype=T).to(dev)
    down, smooth = (torch.randn(K, R, generator=g) * 0.02).to(T).to(dev), (torch.rand(K, generator=g) + 0.5).to(T).to(dev)
    scale, shift = (1 + 0.3 * torch.randn(K, generator=g)).to(T).to(dev), (0.2 * torch.randn(K, generator=g)).to(T).to(dev)
    vecs, xm = None, x
    if norm:
        stats = ops.layer_norm_stats(x)
        vecs = (scale, shift, stats) if norm == "given" else (scale, shift)
        xm = ((x.float() - stats[:, :1]) * stats[:, 1:]).to(T)
        xm = ((xm.float() * scale.float()).to(T).float() + shift.float()).to(T)

    def run(rows, blocked, norm=None):
        return ops.svdq_quantize_w4a4_act_fuse_lora_cuda(rows, lora_down=down, smooth=smooth, norm=norm, pad_size=32, out_blocked=blocked)

    unblocked = None
    for blocked in (0, 2, 3) if K % 512 == 0 else (0, 2):
        codes, scales, la = run(x, blocked, vecs)
        if blocked == 3:
            full = M // 32 * 32
            assert torch.equal(scales.view(-1)[: full * K // 64].cpu(), block_scales(unblocked.cpu()).view(-1)[: full * K // 64])
        unblocked = scales
        for i in range(0, M, 1024):
            n = min(1024, M - i)
            c, s, a = run(xm[i : i + n], blocked)
            whole = n // 32 * 32 if blocked else n  # (rows of the padding are not written)
            assert torch.equal(codes[i : i + whole], c[:whole]) and (blocked == 3 or torch.equal(scales[:, i : i + n], s[:, :n]))
            assert torch.equal(la[i : i + n], a[:n])
    # fp32 sums of K products, 32 at a time
    exact, terms = xm.double() @ down.double(), xm.double().abs() @ down.double().abs()
    assert ((la[:M].double() - exact).abs() <= (K // 32 + 8) * 2.0**-24 * terms).all()


@pytest.mark.parametrize("given", [False, True])
@pytest.mark.parametrize("K,R", [(1536, 32), (3072, 48), (4096, 128)])
def test_low_rank_state_of_a_row_whatever_stands_beside_it(dev, K, R, given):
    """Two batches with scale and shift of their own, in launches of one row block to several for each CU: eight and sixteen wavefronts, row
    blocks shared or not, one to three workgroups that quantize beside those that project."""
    from nunchaku_rocm_amd import ops

    g = torch.Generator().manual_seed(K)
    T = torch.bfloat16
    x = O.make_activations(2 * 4608, K, seed=K, dtype=T).to(dev)
    down = (torch.randn(K, R, generator=g) * 0.02).to(T).to(dev)
    scale, shift = (1 + 0.3 * torch.randn(2, K, generator=g)).to(T).to(dev), (0.2 * torch.randn(2, K, generator=g)).to(T).to(dev)
    stats = ops.layer_norm_stats(x)
    first = None
    for rows in (16, 336, 512, 640, 1024, 2048, 4608):  # of a batch
        print(f"case K={K} R={R} rows={rows} given={given}", flush=True)
        both = torch.cat([x[:rows], x[4608 : 4608 + rows]])
        vecs = (scale, shift, torch.cat([stats[:rows], stats[4608 : 4608 + rows]])) if given else (scale, shift)
        _, _, la = ops.svdq_quantize_w4a4_act_fuse_lora_cuda(both, lora_down=down, norm=vecs, pad_size=32, out_blocked=2)
        head = torch.cat([la[:16], la[rows : rows + 16]])
        first = head if first is None else first
        assert torch.equal(head, first)
    xm = torch.cat([x[:16], x[4608:4624]])
    st = torch.cat([stats[:16], stats[4608:4624]])
    xm = ((xm.float() - st[:, :1]) * st[:, 1:]).to(T).view(2, 16, K)
    xm = ((xm.float() * scale[:, None].float()).to(T).float() + shift[:, None].float()).to(T).view(32, K)
    exact, terms = xm.double() @ down.double(), xm.double().abs() @ down.double().abs()
    assert ((first.double() - exact).abs() <= (K // 32 + 8) * 2.0**-24 * terms).all()
