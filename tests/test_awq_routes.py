"""Which route a call of the AWQ product takes: the kernel that decodes the weight inside, or the decode to memory and a library
product, which carries gradients, tangents, transforms and subclasses of the activations along."""

import pytest
import torch
from torch.autograd import forward_ad

from oracle import svdq_oracle as O

N, K, GROUP = 64, 256, 128


class _Marked(torch.Tensor):
    pass


def _weight(n=N, k=K, group=GROUP, dtype=torch.float16, seed=0):
    g = torch.Generator().manual_seed(seed)
    q = torch.randint(0, 16, (n, k), generator=g, dtype=torch.int32)
    s = (torch.rand(k // group, n, generator=g) * 0.015 + 0.005).to(dtype)
    z = (-torch.randint(0, 16, s.shape, generator=g).float() * s.float()).to(dtype)
    packed = O.awq_pack(q)
    return packed.view(torch.int32), s, z, O.awq_dequantize(packed, s, z, group)


@pytest.fixture
def routes(monkeypatch):
    """The operators on CPU tensors: the decode by the oracle, the kernel's launch noted instead of made."""
    from nunchaku_rocm_amd import _lib
    from nunchaku_rocm_amd.ops import gemv

    launches = []

    class Stub:
        def svdq_awq_gemm_w4a16(self, args, group, stream):
            launches.append(args)
            return 0

        def svdq_awq_gemv_w4a16_bias(self, args, bias, stream):
            launches.append((args, bias))
            return 0

    import contextlib

    monkeypatch.setattr(_lib, "load", Stub)
    monkeypatch.setattr(_lib, "require_cuda", lambda *t: torch.device("cpu"))
    monkeypatch.setattr(_lib, "stream_of", lambda t: 0)
    monkeypatch.setattr(_lib, "on_device", lambda d: contextlib.nullcontext())
    monkeypatch.setattr(gemv, "awq_dequantize", lambda kernel, s, z, n, k, group, dtype: O.awq_dequantize(kernel.view(torch.int16), s, z, group))
    return launches


def test_plain_activations_take_the_kernel(routes):
    from nunchaku_rocm_amd import ops

    qw, s, z, _ = _weight()
    x = torch.randn(5, K).half()
    ops.awq_gemm_w4a16(x, qw, s, z, group_size=GROUP)
    with torch.no_grad():  # nobody will ask for the gradient
        ops.awq_gemm_w4a16(x.clone().requires_grad_(), qw, s, z, group_size=GROUP)
    ops.awq_gemv_w4a16_cuda(x, qw, s, z, 5, N, K, group_size=GROUP)
    with forward_ad.dual_level():  # a level is open, the activations have no part in it
        ops.awq_gemm_w4a16(x, qw, s, z, group_size=GROUP)
    assert len(routes) == 4


def test_too_few_columns_for_a_long_k_take_the_library_product(routes):
    """A workgroup of the kernel walks all of K; sizes on either side of the line, with what was measured (kernel, library)."""
    from nunchaku_rocm_amd import ops
    from nunchaku_rocm_amd.ops.gemv import _decodes_inside

    for m, n, k in [(1, 512, 12288), (17, 1024, 12288), (32, 2048, 12288), (1024, 512, 12288), (1, 512, 4096), (2049, 10240, 4096), (0, 4096, 4096)]:
        assert not _decodes_inside(m, n, k)  # 49 / 24, 50 / 31, 50 / 41, 51 / 45, 19 / 16 us
    for m, n, k in [(1, 4096, 12288), (256, 4096, 12288), (77, 4096, 4096), (2048, 10240, 4096), (1, 4, 64), (2048, 128, 2048), (1024, 2048, 12288)]:
        assert _decodes_inside(m, n, k)  # 50 / 55, 54 / 79, 20 / 36, 171 / 175 us, ..., 70 / 92
    qw, s, z, w = _weight(k=2304)
    x = torch.randn(5, 2304).half()
    out = ops.awq_gemm_w4a16(x, qw, s, z, group_size=GROUP)
    assert not routes and torch.equal(out, x @ w.t())


def test_what_the_kernel_does_not_carry_is_carried_on(routes):
    from nunchaku_rocm_amd import ops

    qw, s, z, w = _weight()
    x, t = torch.randn(5, K).half(), torch.randn(5, K).half()
    call = lambda a: ops.awq_gemm_w4a16(a, qw, s, z, group_size=GROUP)  # noqa: E731
    # the same product up to the order of K fp32 additions and the rounding to fp16
    close = lambda a, b: torch.testing.assert_close(a.float(), b.float(), rtol=2.0**-9, atol=2e-2)  # noqa: E731

    a = x.clone().requires_grad_()
    call(a).backward(t[:, :N])
    close(a.grad, t[:, :N] @ w)
    with forward_ad.dual_level():
        out = forward_ad.unpack_dual(call(forward_ad.make_dual(x, t)))
        close(out.primal, x @ w.t())
        close(out.tangent, t @ w.t())
    close(torch.func.jvp(call, (x,), (t,))[1], t @ w.t())
    close(torch.func.vmap(call)(torch.stack([x, t])), torch.stack([x, t]) @ w.t())
    close(call(torch._neg_view(x)), -x @ w.t())
    assert type(call(x.as_subclass(_Marked))) is _Marked
    assert not routes


@pytest.mark.gpu
@pytest.mark.parametrize("m", [3, 300, 2048, 2049])
def test_gradients_on_both_sides_of_the_row_limit(dev, m):
    from nunchaku_rocm_amd.linear import AWQW4A16Linear

    dtype = torch.bfloat16
    qw, s, z, w = _weight(dtype=dtype)
    mod = AWQW4A16Linear(K, N, group_size=GROUP, torch_dtype=dtype, device=dev)
    mod.qweight.data, mod.wscales.data, mod.wzeros.data = qw.to(dev), s.to(dev), z.to(dev)
    mod.bias.data.fill_(0.5)
    g = torch.Generator().manual_seed(m)
    x, grad = torch.randn(m, K, generator=g).to(dtype), torch.randn(m, N, generator=g).to(dtype)
    a = x.to(dev).requires_grad_()
    out = mod(a)
    out.backward(grad.to(dev))
    ref = grad.double() @ w.double()
    # one rounding to bf16, and N fp32 additions of exact products in any order
    bound = ref.abs() * 2.0**-8 + N * 2.0**-24 * (grad.double().abs() @ w.double().abs()) + 1e-6
    assert ((a.grad.cpu().double() - ref).abs() <= bound).all()
    with torch.no_grad():  # the kernel, where it runs: the same product before the bias within two roundings
        plain = mod(a)
    ref = x.double() @ w.double().t() + 0.5
    bound = (ref.abs() + 1) * 2.0**-7 + K * 2.0**-24 * (x.double().abs() @ w.double().abs().t())
    assert ((plain.cpu().double() - ref).abs() <= bound).all() and ((out.detach().cpu().double() - ref).abs() <= bound).all()


@pytest.mark.gpu
def test_autocast_decides_on_the_type(dev):
    from nunchaku_rocm_amd import ops

    qw, s, z, w = (t.to(dev) for t in _weight(dtype=torch.bfloat16))
    x = torch.randn(5, K, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).to(dev)
    with torch.autocast("cuda", torch.float16):
        out = ops.awq_gemm_w4a16(x, qw, s, z, group_size=GROUP)
    assert out.dtype == torch.float16 and torch.equal(out, x.half() @ w.half().t())
    with torch.autocast("cuda", torch.bfloat16):
        assert torch.equal(ops.awq_gemm_w4a16(x, qw, s, z, group_size=GROUP), ops.awq_gemm_w4a16(x, qw, s, z, group_size=GROUP))
    assert ops.awq_gemm_w4a16(x, qw, s, z, group_size=GROUP).dtype == torch.bfloat16


def test_a_bias_the_kernel_cannot_carry_is_added_behind_it(routes):
    from nunchaku_rocm_amd.ops.gemv import awq_gemv_bias

    qw, s, z, _ = _weight(group=64)
    x, bias, tangent = torch.zeros(2, K).half(), torch.randn(N).half(), torch.randn(N).half()
    call = lambda b: awq_gemv_bias(x, qw, s, z, b, 2, N, K)  # noqa: E731
    call(bias)
    assert routes[-1][1] == bias.data_ptr()
    with forward_ad.dual_level():
        call(bias)
        assert routes[-1][1] == bias.data_ptr()
        out = call(forward_ad.make_dual(bias, tangent))
        assert torch.equal(forward_ad.unpack_dual(out).tangent, tangent.expand(2, N)) and routes[-1][1] is None
    assert call(bias.clone().requires_grad_()).requires_grad and routes[-1][1] is None
    call(torch._neg_view(bias))
    assert routes[-1][1] is None


def _laid_out(x: torch.Tensor) -> dict:
    """The values of ``x`` in the layouts the library product takes."""
    m, k = x.shape
    odd = torch.empty(1 + m * k, dtype=x.dtype, device=x.device)[1:].view(m, k)
    wide = torch.empty(m, k + 4, dtype=x.dtype, device=x.device)[:, 2 : 2 + k]
    padded = torch.empty(m, k + 8, dtype=x.dtype, device=x.device)[:, :k]
    turned = torch.empty(k, m, dtype=x.dtype, device=x.device).t()
    views = {"one piece at an odd address": odd, "odd columns": wide, "aligned rows apart": padded, "transposed": turned}
    for v in views.values():
        v.copy_(x)
    views["one row over and over"] = x[:1].expand(m, k)
    return views


@pytest.mark.parametrize("m", [1, 2, 5])
def test_rows_are_handed_over_aligned(routes, m):
    from nunchaku_rocm_amd import ops

    qw, s, z, _ = _weight()
    views = _laid_out(torch.randn(m, K).half())
    for name, x in views.items():
        ops.awq_gemm_w4a16(x, qw, s, z, group_size=GROUP)
        args = routes[-1]
        assert args.x % 16 == 0 and args.ld_x >= K and args.ld_x % 8 == 0, name
        if name == "aligned rows apart":
            assert args.x == x.data_ptr() and (m == 1 or args.ld_x == K + 8)
    assert len(routes) == len(views)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 2, 40])
def test_layouts_of_the_activations(dev, m):
    from nunchaku_rocm_amd import ops

    qw, s, z, _ = (t.to(dev) for t in _weight())
    x = torch.randn(m, K, generator=torch.Generator().manual_seed(m)).half().to(dev)
    for name, v in _laid_out(x).items():
        print(f"case m={m} {name}", flush=True)
        assert torch.equal(ops.awq_gemm_w4a16(v, qw, s, z, group_size=GROUP), ops.awq_gemm_w4a16(v.clone(memory_format=torch.contiguous_format), qw, s, z, group_size=GROUP))
