"""The checks in native code (csrc/host.cpp) against the operators' Python code: the same argument block for every form the
native code accepts, and nothing accepted that is not the ordinary case."""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

NAMES = ("quantize_buffers", "quantize", "gemm", "gemv", "attention")


class _Off:
    """The extension with every shortcut declined."""

    def __getattr__(self, name):
        return lambda *a: False


@pytest.fixture
def calls(monkeypatch):
    """``run(f, fresh)``: the argument blocks ``f()`` hands to the library, by native code and by Python, as dicts without the
    addresses in ``fresh`` (allocated in the call); and how many of the native functions did their part."""
    from nunchaku_rocm_amd import _lib

    lib, native = _lib.load(), _lib.host()
    blocks, taken = [], []

    class Lib:
        def __getattr__(self, name):
            entry = getattr(lib, name)
            if name not in ("svdq_quantize_act", "svdq_gemm_w4a4", "svdq_awq_gemv_w4a16_bias", "svdq_attention_fp16"):
                return entry

            def call(args, *more):
                blocks.append((name, {f: getattr(args, f) for f, _ in args._fields_}, *(m or 0 for m in more)))
                return entry(args, *more)

            return call

    class Host:
        def __getattr__(self, name):
            def call(*a):
                result = getattr(native, name)(*a)
                if name in NAMES:
                    taken.append(result is not False)
                return result

            return call

    def run(f, fresh=()):
        monkeypatch.setattr(_lib, "load", lambda: Lib())
        out = []
        for host in (Host(), _Off()):
            monkeypatch.setattr(_lib, "host", lambda: host)
            blocks.clear()
            f()
            torch.cuda.synchronize()
            out.append([(b[0], {k: v for k, v in b[1].items() if k not in fresh}, *b[2:]) for b in blocks])
        did = list(taken)
        taken.clear()
        monkeypatch.setattr(_lib, "load", lambda: lib)
        monkeypatch.setattr(_lib, "host", lambda: native)
        return out[0], out[1], did

    return run


def _linear(k, n, rank, dtype, dev, **kw):
    from nunchaku_rocm_amd.linear import SVDQW4A4Linear

    g = torch.Generator(device=dev).manual_seed(k + n)
    lin = SVDQW4A4Linear(k, n, rank=rank, torch_dtype=dtype, device=dev, **kw)
    with torch.no_grad():
        lin.qweight.copy_(torch.randint(-128, 128, lin.qweight.shape, device=dev, generator=g, dtype=torch.int16).to(torch.int8))
        for p in (lin.wscales, lin.smooth_factor, lin.proj_down, lin.proj_up, *([lin.bias] if lin.bias is not None else [])):
            p.copy_(torch.rand(p.shape, device=dev, generator=g).to(dtype) * 0.1 + 0.01)
    return lin.requires_grad_(False)


def _warm(*fs):
    """Working copies are made, and known to be complete, before the native code reads them."""
    for f in fs:
        for _ in range(2):
            f()
            torch.cuda.synchronize()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,blocked,norm", [(1, 512, 0, None), (33, 576, 1, "1d"), (300, 1024, 2, "2d"), (65, 512, 3, "stats"), (17, 1536, 3, "strided"), (40, 640, 2, None)])
def test_quantizer_blocks(dev, calls, M, K, blocked, norm, dtype):
    from nunchaku_rocm_amd import ops

    lin = _linear(K, 256, 32, dtype, dev)
    x = torch.randn(M, K + 64, device=dev).to(dtype)[:, :K]  # rows of another stride
    emb = torch.rand(1, K, 6, device=dev).to(dtype)
    nm = {None: None, "1d": (emb[0, :, 0].contiguous(), emb[0, :, 1].contiguous()), "2d": (emb[:, :, 0].contiguous(), emb[:, :, 1].contiguous()),
          "strided": (emb[:, :, 1], emb[:, :, 0])}.get(norm)  # fmt: skip
    if norm == "stats":
        nm = (emb[0, :, 0].contiguous(), emb[0, :, 1].contiguous(), ops.layer_norm_stats(x))
    rows = -(-M // 256) * 256
    buf = dict(output=torch.zeros(rows, K * 3 // 4 if blocked >= 2 else K // 2, dtype=torch.uint8, device=dev),
               oscales=torch.zeros(K // 64, rows, dtype=dtype, device=dev), lora_act_out=torch.zeros(rows, 32, device=dev))  # fmt: skip
    f = lambda **kw: ops.svdq_quantize_w4a4_act_fuse_lora_cuda(x, lora_down=lin.proj_down, smooth=lin.smooth_factor, norm=nm, out_blocked=blocked, **kw)  # noqa: E731
    _warm(lambda: f(**buf))
    lone = ("ld_x",) if M == 1 else ()  # the distance of a lone row's neighbours: reshape() makes one up
    a, b, taken = calls(lambda: f(**buf), fresh=lone)
    assert a == b and len(a) == 1 and taken == [True]
    a, b, taken = calls(f, fresh=("out", "scales", "lora_act", *lone))  # buffers allocated in the call
    assert a == b and len(a) == 1 and taken == [True, True]
    a, b, taken = calls(lambda: f(output=buf["output"], oscales=buf["oscales"].float().to(dtype), lora_act_out=buf["lora_act_out"]), fresh=("scales", *lone))
    assert a == b and taken == [True]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("epilogue,blocked,rank,bias", [("plain", 0, 32, True), ("plain", 2, 0, False), ("plain", 3, 48, True), ("qkv", 3, 32, True), ("qkv", 1, 16, False),
                                                       ("gelu", 3, 32, True), ("gelu", 2, 16, True), ("swiglu", 3, 32, False), ("gelu", 0, 0, True)])  # fmt: skip
def test_gemm_blocks(dev, calls, epilogue, blocked, rank, bias, dtype):
    from nunchaku_rocm_amd import ops

    M, K, N = 160, 512, 384 if epilogue == "qkv" else 1024
    lin = _linear(K, N, max(rank, 16), dtype, dev, bias=bias)
    x = torch.randn(M, K, device=dev).to(dtype)
    q, s, la = ops.svdq_quantize_w4a4_act_fuse_lora_cuda(x, lora_down=lin.proj_down, smooth=lin.smooth_factor, out_blocked=blocked)
    kw = dict(act=q, wgt=lin.qweight, ascales=s, wscales=lin.wscales, lora_act_in=la if rank else None, lora_up=lin.proj_up if rank else None,
              bias=lin.bias, act_blocked=blocked)  # fmt: skip
    if epilogue in ("plain", "qkv"):
        kw["out"] = torch.empty(M, N + 32, dtype=dtype, device=dev)[:, :N]
        if epilogue == "qkv":
            w = torch.nn.Parameter(torch.rand(128, device=dev).to(dtype), requires_grad=False)
            kw.update(norm_q=w, norm_k=w, rotary_emb=torch.randn(M, 64, 1, 2, device=dev))
    else:
        nq = N // 2 if epilogue == "swiglu" else N
        nxt = _linear(nq, 128, max(rank, 16), dtype, dev)
        qb = blocked if nq % 512 == 0 or blocked < 3 else 2
        kw.update(qout=torch.empty(q.shape[0], nq * 3 // 4 if qb >= 2 else nq // 2, dtype=torch.uint8, device=dev), fuse_swiglu=epilogue == "swiglu",
                  oscales=torch.empty(nq // 64, q.shape[0], dtype=dtype, device=dev), smooth_factor=nxt.smooth_factor, qout_blocked=qb)  # fmt: skip
        if rank:
            kw.update(lora_down=nxt.proj_down, lora_act_out=torch.empty(q.shape[0], nxt.proj_down.shape[1], device=dev))
    f = lambda: ops.svdq_gemm_w4a4_cuda(**kw)  # noqa: E731
    _warm(f)
    a, b, taken = calls(f, fresh=("scratch",))
    assert a == b and len(a) == 1 and taken == [True]


@pytest.mark.parametrize("M,N,R2,swiglu", [(16, 128, 16, False), (160, 1024, 48, True), (272, 1152, 32, False)])
def test_scratch_memory_is_what_the_library_asks_for(dev, monkeypatch, M, N, R2, swiglu):
    from nunchaku_rocm_amd import _lib, ops
    from nunchaku_rocm_amd.ops import gemm as G

    k, nq, dtype = 128, N // 2 if swiglu else N, torch.bfloat16
    byte = lambda *s: torch.zeros(*s, dtype=torch.uint8, device=dev)  # noqa: E731
    val = lambda *s: torch.ones(*s, dtype=dtype, device=dev)  # noqa: E731
    kw = dict(act=byte(M, k // 2), wgt=byte(N, k // 2), ascales=val(k // 64, M), wscales=val(k // 64, N), fuse_swiglu=swiglu, qout=byte(M, nq // 2),
              oscales=val(nq // 64, M), lora_down=val(nq, R2), lora_act_out=torch.empty(M, R2, device=dev))  # fmt: skip
    native, made = _lib.host(), []

    class Host:
        def __getattr__(self, name):
            return getattr(native, name)

        def gemm(self, *a):
            made.append(native.gemm(*a))
            return made[-1]

    monkeypatch.setattr(_lib, "host", lambda: Host())
    monkeypatch.setattr(G, "USE_WEIGHT_PLANES", "all")
    for _ in range(3):
        ops.svdq_gemm_w4a4_cuda(**kw)
        torch.cuda.synchronize()
    epilogue = _lib.EPI_SWIGLU_QUANT if swiglu else _lib.EPI_GELU_QUANT
    assert made and made[-1].nbytes == _lib.load().svdq_gemm_w4a4_scratch_bytes(M, N, R2, epilogue)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,bias", [(1, True), (8, False), (32, True)])
def test_gemv_blocks(dev, calls, m, bias, dtype):
    from nunchaku_rocm_amd.ops.gemv import awq_gemv_bias

    n, k = 96, 512
    w = torch.randint(-(2**31), 2**31 - 1, (n // 4, k // 2), device=dev, dtype=torch.int32)
    s = torch.rand(k // 64, n + 32, device=dev).to(dtype)[:, :n]
    b = torch.rand(n, device=dev).to(dtype) if bias else None
    x = torch.randn(m, k + 8, device=dev).to(dtype)[:, :k]
    one, two, taken = calls(lambda: awq_gemv_bias(x, w, s, s, b, m, n, k, 64), fresh=("out", "ld_x") if m == 1 else ("out",))
    assert one == two and len(one) == 1 and taken == [True]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,q,kv,d", [(1, 2, 65, 65, 128), (2, 3, 40, 77, 64), (2, 1, 1, 1, 128)])
def test_attention_blocks(dev, calls, B, H, q, kv, d, dtype):
    from nunchaku_rocm_amd import ops

    def views(t, parts):
        x = torch.randn(B, t, parts * H * d, device=dev).to(dtype)
        return [p.view(B, t, H, d).transpose(1, 2) for p in x.chunk(parts, dim=-1)]

    (a,), (k, v) = views(q, 1), views(kv, 2)
    outs = []
    one, two, taken = calls(lambda: outs.append(ops.scaled_dot_product_attention(a, k, v)), fresh=("o",))
    assert one == two and len(one) == 1 and taken == [True]
    assert outs[0].shape == outs[1].shape and outs[0].stride() == outs[1].stride() and torch.equal(outs[0], outs[1])


def test_norm_without_scale_or_shift(dev):
    """A norm whose scale and shift are missing is refused, not quantized without the norm."""
    from nunchaku_rocm_amd import ops

    x = torch.randn(16, 512, device=dev).to(torch.bfloat16)
    v = torch.ones(512, device=dev, dtype=x.dtype)
    buf = (torch.zeros(16, 256, dtype=torch.uint8, device=dev), torch.zeros(8, 16, dtype=x.dtype, device=dev))
    ops.quantize_w4a4_act_fuse_lora(x, *buf, norm=(v, v))
    for norm in ((None, None), (None, None, None), (v, None), (None, v), (None, None, ops.layer_norm_stats(x))):
        with pytest.raises((AttributeError, TypeError)):
            ops.quantize_w4a4_act_fuse_lora(x, *buf, norm=norm)


def test_allocations_let_other_threads_run(dev):
    """While the native code allocates, another Python thread gets the interpreter's lock, as inside torch.empty.  (The lock changes hands
    only where it is let go of: no switches by time here.)"""
    import sys
    import threading

    from nunchaku_rocm_amd import _lib

    host, gate, ran = _lib.host(), threading.Lock(), []
    x = torch.zeros(16, 2048, device=dev, dtype=torch.bfloat16)
    gate.acquire()
    thread = threading.Thread(target=lambda: (gate.acquire(), ran.append(1)))
    torch.cuda.empty_cache()  # the allocation asks the device for memory, which takes long enough for a thread to wake up
    thread.start()
    old = sys.getswitchinterval()
    sys.setswitchinterval(60.0)
    try:
        gate.release()
        buffers = host.quantize_buffers(x, 0, 1 << 23, 0)  # 8 GB of codes
        during = list(ran)
    finally:
        sys.setswitchinterval(old)
        thread.join()
    assert buffers is not False and during == [1]
    del buffers
    torch.cuda.empty_cache()


def test_what_is_left_to_python(dev):
    """Not the ordinary case: declined, and the block is not touched."""
    from nunchaku_rocm_amd import _lib

    host, dt = _lib.host(), torch.bfloat16

    class Sub(torch.Tensor):
        pass

    n, k = 64, 128
    x, w = torch.randn(2, k, device=dev).to(dt), torch.zeros(n // 4, k // 2, dtype=torch.int32, device=dev)
    s, b = torch.rand(k // 64, n, device=dev).to(dt), torch.rand(n, device=dev).to(dt)
    args = _lib.AwqGemvArgs()
    gemv = lambda x=x, w=w, s=s, z=s, b=b, m=2, n=n, k=k: host.gemv(args, x, w, s, z, b, m, n, k)  # noqa: E731
    empty = bytes(args)
    assert gemv() is not False
    ctypes.memset(ctypes.byref(args), 0, ctypes.sizeof(args))
    wrong = [dict(x=x.cpu()), dict(x=x.as_subclass(Sub)), dict(x=x.float()), dict(x=x[:, ::2], k=64), dict(x=x[1:], m=2), dict(x=x[None], m=2),
             dict(w=w[:-1]), dict(w=w.t()), dict(s=s.t().contiguous().t()), dict(z=s[:, :32]), dict(b=b.float()), dict(b=b[:32]),
             dict(b=b.clone().requires_grad_()), dict(b=b.as_subclass(Sub)), dict(b=torch.rand(2 * n, device=dev).to(dt)[::2]), dict(n=48, b=None), dict(m=33), dict(m=0)]  # fmt: skip
    for kw in wrong:
        assert gemv(**kw) is False and bytes(args) == empty, kw
    with torch.autograd.forward_ad.dual_level():
        assert gemv(b=torch.autograd.forward_ad.make_dual(b, b)) is False
    assert torch.func.vmap(lambda v: torch.as_tensor(float(gemv(x=v) is False), device=dev).expand(1))(x[None].expand(2, 2, k)).sum() == 2
    with torch.no_grad():
        assert gemv(b=b.clone().requires_grad_()) is not False
    att = _lib.AttentionArgs()
    q = torch.randn(1, 2, 8, 64, device=dev).to(dt)
    empty = bytes(att)
    for t in ((q.float(),) * 3, (q, q.half(), q), (q, q[:, :, :0], q[:, :, :0]), (q[..., ::2],) * 3, (q, q, q[:, :, 1:]), (q.cpu(),) * 3, (q[0],) * 3):
        assert host.attention(att, *t) is False and bytes(att) == empty
    assert host.same_source((0, w.untyped_storage(), 0, w.shape, w.stride()), w.cpu()) is None
    assert host.same_source((w._version, w.untyped_storage(), 0, w.shape, w.stride()), w) is True
    assert host.same_source((w._version, w.untyped_storage(), 4, w.shape, w.stride()), w) is False
    w.add_(1)
    assert host.same_source((w._version - 1, w.untyped_storage(), 0, w.shape, w.stride()), w) is False
