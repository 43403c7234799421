"""AWQ W4A16 operators: the group-64 GEMV, the dense decode and the GEMM built on it (reference:
nunchaku/ops/gemv.py:10-56, nunchaku/ops/dispatch.py:19-49, nunchaku/ops/triton/awq.py:83-118, 186-251)."""

from __future__ import annotations

import torch
from torch.autograd import forward_ad

from .. import _lib

_MAX_ROWS = 32  # rows one launch handles; more rows re-stream the weights per block of 32


def awq_gemv_w4a16_cuda(
    in_feats: torch.Tensor,
    kernel: torch.Tensor,
    scaling_factors: torch.Tensor,
    zeros: torch.Tensor,
    m: int,
    n: int,
    k: int,
    group_size: int = 64,
) -> torch.Tensor:
    """
    ``out = in_feats @ (q * scaling_factors + zeros).T`` with ``q`` the TinyChat-packed uint4 weight
    (``kernel`` ``(n // 4, k // 2)`` int32).  Group size 64 runs the fused GEMV kernel (weights read once for all ``m``
    rows).  Two cases take :func:`awq_gemm_w4a16` (the weight rounded to 16 bits, the reference's own route for everything
    but group size 64, ops/triton/awq.py:226-228): other group sizes or ``n % 32 != 0``, and shapes whose per-group tables
    do not fit the kernel's 64 KB of LDS (``k = 12288`` with more than 16 rows; no FLUX shape).  Weights of 4 GiB and more
    are refused (``RuntimeError``): the kernels address them with 32-bit offsets.  Returns ``in_feats.shape[:-1] + (n,)``
    in the input dtype.
    """
    return awq_gemv_bias(in_feats, kernel, scaling_factors, zeros, None, m, n, k, group_size)


def awq_gemv_bias(in_feats, kernel, scaling_factors, zeros, bias: torch.Tensor | None, m: int, n: int, k: int, group_size: int = 64) -> torch.Tensor:
    """:func:`awq_gemv_w4a16_cuda`, then ``+ bias`` (``(n,)``, rounded again as an addition of its own would) in the kernel's
    last step where the fused kernel runs and the bias is a contiguous tensor of the output dtype and no more than its values
    (a gradient or a tangent wanted through it: an addition of its own)."""
    if group_size == 64:  # the ordinary call, checked in native code; anything else is left to what follows
        args = _lib.AwqGemvArgs()
        ready = _lib.host().gemv(args, in_feats, kernel, scaling_factors, zeros, bias, m, n, k)
        if ready:
            rc = _lib.load().svdq_awq_gemv_w4a16_bias(args, ready[1], _lib.stream_of(in_feats))
            if rc != _lib.E_UNSUPPORTED:
                _lib.check(rc)
                return ready[0]
    _lib.require_cuda(in_feats, kernel, scaling_factors, zeros)
    x = in_feats.reshape(m, k)
    if group_size != 64 or n % 32:
        return _plus_bias(_product(x, kernel, scaling_factors, zeros, n, k, group_size).reshape(*in_feats.shape[:-1], n), bias)
    if x.stride(1) != 1 or x.stride(0) % 8 or x.data_ptr() % 16:
        x = x.contiguous()
    if kernel.element_size() * kernel.numel() != n * k // 2 or not kernel.is_contiguous():
        raise ValueError(f"unexpected packed AWQ weight shape {tuple(kernel.shape)} for n={n}, k={k}")
    if scaling_factors.stride(1) != 1 or zeros.stride() != scaling_factors.stride():
        raise ValueError("scaling_factors and zeros must share a row-major (k // 64, n) layout")
    if scaling_factors.dtype != x.dtype or zeros.dtype != x.dtype:
        raise ValueError("scaling_factors / zeros must have the input dtype")
    if n * k // 2 >= 1 << 32:
        raise RuntimeError(f"AWQ weight of {n * k // 2} bytes: 4 GiB and more are not supported (32-bit offsets)")
    out = torch.empty(m, n, dtype=x.dtype, device=x.device)
    fused = None  # the bias' address where the kernel adds it
    if bias is not None and _is_plain(bias) and bias.dtype == x.dtype and bias.device == x.device and bias.shape == (n,) and bias.is_contiguous():
        fused = bias.data_ptr()
    lib = _lib.load()
    with _lib.on_device(x.device):
        for r0 in range(0, m, _MAX_ROWS):
            rows = min(_MAX_ROWS, m - r0)
            args = _lib.AwqGemvArgs(
                x=x[r0:].data_ptr(),
                qweight=kernel.data_ptr(),
                scales=scaling_factors.data_ptr(),
                zeros=zeros.data_ptr(),
                out=out[r0:].data_ptr(),
                M=rows,
                N=n,
                K=k,
                ld_x=x.stride(0),
                ld_scales=scaling_factors.stride(0),
                ld_out=out.stride(0),
                dtype=_lib.dtype_code(x.dtype),
            )
            rc = lib.svdq_awq_gemv_w4a16_bias(args, fused, _lib.stream_of(x))
            if rc == _lib.E_UNSUPPORTED:
                # the kernel's per-group tables do not fit LDS (K = 12288 with more than 16 rows, longer K with fewer):
                # the GEMM, as for other group sizes (the other refusal, a weight of 4 GiB and more, was raised above)
                return _plus_bias(_product(x, kernel, scaling_factors, zeros, n, k, group_size).reshape(*in_feats.shape[:-1], n), bias)
            _lib.check(rc)
    out = out.reshape(*in_feats.shape[:-1], n)
    return out if fused else _plus_bias(out, bias)


def _plus_bias(out: torch.Tensor, bias: torch.Tensor | None) -> torch.Tensor:
    return out if bias is None else out.add_(bias.view([1] * (out.ndim - 1) + [-1]))


class AwqGemvBatch:
    """Several AWQ W4A16 GEMVs of one shape, all on the same input, in one launch (``svdq_awq_gemv_w4a16_batched``).

    The adaLN projections of a diffusion transformer all take ``silu(temb)`` and depend on nothing else in the model
    (nunchaku/models/normalization.py), so the model can compute them together; one 32 MB weight is too short a read to
    reach the HBM rate, many behind each other are not.  Built once from the layers' tensors (``kernels[i]``
    ``(n // 4, k // 2)`` int32, ``scales[i]`` / ``zeros[i]`` ``(k // 64, n)``); ``__call__`` copies the input into the
    batch's own buffer and returns ``(count, m, n)``, a buffer the next call overwrites.  Results are bit-identical to
    :func:`awq_gemv_w4a16_cuda` layer by layer.  Up to eight rows, group size 64.  No counterpart in the reference.
    """

    def __init__(self, kernels, scales, zeros, m: int, n: int, k: int):
        import ctypes

        if not 1 <= m <= 8:
            raise ValueError(f"m={m}: a batched launch takes up to eight rows")
        _lib.require_cuda(*kernels, *scales, *zeros)
        count, dev, dtype = len(kernels), kernels[0].device, scales[0].dtype
        if count == 0 or len(scales) != count or len(zeros) != count:
            raise ValueError("kernels, scales and zeros must be equally long, non-empty lists")
        if n * k // 2 >= 1 << 32:
            raise RuntimeError(f"AWQ weight of {n * k // 2} bytes: 4 GiB and more are not supported (32-bit offsets)")
        self.m, self.n, self.k, self.count = m, n, k, count
        self.x = torch.zeros(m, k, dtype=dtype, device=dev)
        self.out = torch.empty(count, m, n, dtype=dtype, device=dev)
        self._keep = (list(kernels), list(scales), list(zeros))
        table = (_lib.AwqGemvArgs * count)()
        for i, (q, sc, z) in enumerate(zip(kernels, scales, zeros)):
            if q.element_size() * q.numel() != n * k // 2 or not q.is_contiguous() or q.data_ptr() % 16:
                raise ValueError(f"problem {i}: unexpected packed AWQ weight {tuple(q.shape)} for n={n}, k={k}")
            for name, t in (("scales", sc), ("zeros", z)):
                if t.shape != (k // 64, n) or t.dtype != dtype or t.stride() != (n, 1) or t.data_ptr() % 16 or t.device != dev:
                    raise ValueError(f"problem {i}: {name} must be a contiguous ({k // 64}, {n}) {dtype} tensor on {dev}")
            table[i] = _lib.AwqGemvArgs(x=self.x.data_ptr(), qweight=q.data_ptr(), scales=sc.data_ptr(), zeros=z.data_ptr(),
                                        out=self.out[i].data_ptr(), M=m, N=n, K=k, ld_x=k, ld_scales=n, ld_out=n,
                                        dtype=_lib.dtype_code(dtype))  # fmt: skip
        self._first = table[0]
        raw = torch.frombuffer(bytearray(bytes(table)), dtype=torch.uint8)
        self._table = raw.to(dev)  # the device copy the kernel reads its pointers from

    def __call__(self, in_feats: torch.Tensor) -> torch.Tensor:
        self.x.copy_(in_feats.reshape(self.m, self.k))
        with _lib.on_device(self.x.device):
            _lib.check(_lib.load().svdq_awq_gemv_w4a16_batched(self._first, self._table.data_ptr(), self.count, _lib.stream_of(self.x)))
        return self.out


def _check_weight(kernel, scaling_factors, zeros, n: int, k: int, group_size: int, dtype: torch.dtype):
    _lib.require_cuda(kernel, scaling_factors, zeros)
    if kernel.element_size() * kernel.numel() != n * k // 2 or not kernel.is_contiguous():
        raise ValueError(f"unexpected packed AWQ weight shape {tuple(kernel.shape)} for n={n}, k={k}")
    if group_size <= 0 or k % group_size:
        raise ValueError(f"group_size={group_size} does not divide k={k}")
    groups = k // group_size
    if scaling_factors.shape != (groups, n) or zeros.shape != (groups, n):
        raise ValueError(f"scaling_factors / zeros must be ({groups}, {n})")
    if scaling_factors.dtype != dtype or zeros.dtype != dtype:
        raise ValueError("scaling_factors / zeros must have the output dtype")
    if scaling_factors.stride(1) != 1 or zeros.stride() != scaling_factors.stride():
        scaling_factors, zeros = scaling_factors.contiguous(), zeros.contiguous()
    return scaling_factors, zeros


def _decodes_inside(m: int, n: int, k: int) -> bool:
    """Whether the GEMM that decodes the weight inside is the faster one, or a decode to memory and a library product is.

    Rows: beyond 2048 the decode to memory is paid once for many (K = 4096: N = 10240 169 us in the kernel against 173 at 2048
    rows, 241 against 200 at 3000; N = 4096 63 against 73, 108 against 91).
    Columns and K: a workgroup of the kernel walks all of K, 3.7 us per 1024 of it however few workgroups there are, while the
    decode costs by the weight's size and the library product may split K.  So it needs columns (and, less, rows) for its K.  The
    line is a fit to 1098 sizes (K 1024 to 24576, N 128 to 10240, 1 to 2048 rows) on which it takes no size that is more than 2 %
    slower in the kernel.  Kernel against library, us, 32 rows: K = 12288, N = 512 50 against 28, 1024 50 against 36, 4096 50
    against 58; K = 4096, N = 512 19 against 14, 1536 20 against 22; K = 2048, N = 128 11.5 against 11.6.  Past 12288 the library
    product slows down by more than K."""
    return 0 < m <= 2048 and (k <= 2048 or n * (512 + m) >= 128 * (2400 + min(k, 12288)))


_PLAIN_TYPES = frozenset((torch.Tensor, torch.nn.Parameter))
_is_wrapped = torch._C._functorch.is_functorch_wrapped_tensor


def _is_plain(t: torch.Tensor) -> bool:
    """Whether ``t`` is no more than the values in its memory: a kernel that is handed an address carries no gradient, tangent,
    batch dimension of a transform, subclass or pending negation along."""
    if type(t) not in _PLAIN_TYPES or (t.requires_grad and torch.is_grad_enabled()) or t.is_neg() or _is_wrapped(t):
        return False
    return forward_ad._current_level < 0 or forward_ad.unpack_dual(t).tangent is None


def _cast_by_autocast(x: torch.Tensor) -> bool:
    return torch.is_autocast_enabled("cuda") and torch.get_autocast_dtype("cuda") != x.dtype


def _aligned_rows(x: torch.Tensor) -> tuple[torch.Tensor, int]:
    """The 2-D ``x`` with 16-byte aligned rows of unit stride, and the distance of its rows: itself, or a copy (``contiguous()``
    makes none of a tensor that lies in one piece at an odd address).  The stride of a lone row means nothing."""
    m, k = x.shape
    ld = x.stride(0) if m > 1 else k
    if x.stride(1) == 1 and ld >= k and ld % 8 == 0 and x.data_ptr() % 16 == 0:
        return x, ld
    return x.clone(memory_format=torch.contiguous_format), k


def _product(x: torch.Tensor, kernel, scaling_factors, zeros, n: int, k: int, group_size: int) -> torch.Tensor:
    """``x @ T(q * s + z).T`` for a 2-D ``x``: the weight decoded inside the GEMM (``svdq_awq_gemm_w4a16``), or decoded to
    memory first for a library product where that is faster or where ``x`` is more than its values: the product is
    differentiable in ``x``, forward and backward, can be mapped over it, and follows an enclosing autocast."""
    scaling_factors, zeros = _check_weight(kernel, scaling_factors, zeros, n, k, group_size, x.dtype)
    m = x.shape[0]
    if _decodes_inside(m, n, k) and x.shape[1] == k and _is_plain(x) and not _cast_by_autocast(x):
        x, ld_x = _aligned_rows(x)
        out = torch.empty(m, n, dtype=x.dtype, device=x.device)
        args = _lib.AwqGemvArgs(x=x.data_ptr(), qweight=kernel.data_ptr(), scales=scaling_factors.data_ptr(), zeros=zeros.data_ptr(),
                                out=out.data_ptr(), M=m, N=n, K=k, ld_x=ld_x, ld_scales=scaling_factors.stride(0), ld_out=n,
                                dtype=_lib.dtype_code(x.dtype))  # fmt: skip
        with _lib.on_device(x.device):
            rc = _lib.load().svdq_awq_gemm_w4a16(args, group_size, _lib.stream_of(x))
        if rc != _lib.E_UNSUPPORTED:  # tensors too large for its 32-bit offsets
            _lib.check(rc)
            return out
    w = awq_dequantize(kernel, scaling_factors, zeros, n, k, group_size, x.dtype)
    return torch.matmul(x, w.t())


def awq_dequantize(
    kernel: torch.Tensor,
    scaling_factors: torch.Tensor,
    zeros: torch.Tensor,
    n: int,
    k: int,
    group_size: int,
    dtype: torch.dtype,
) -> torch.Tensor:
    """
    Unpack a TinyChat-packed AWQ W4 weight to a dense ``(n, k)`` tensor ``q * scaling_factors + zeros`` of ``dtype``
    (reference: nunchaku/ops/triton/awq.py:83-118).
    """
    scaling_factors, zeros = _check_weight(kernel, scaling_factors, zeros, n, k, group_size, dtype)
    out = torch.empty(n, k, dtype=dtype, device=kernel.device)
    with _lib.on_device(kernel.device):
        _lib.check(_lib.load().svdq_awq_dequantize(kernel.data_ptr(), scaling_factors.data_ptr(), zeros.data_ptr(),
                                                   out.data_ptr(), n, k, group_size, scaling_factors.stride(0),
                                                   out.stride(0), _lib.dtype_code(dtype), _lib.stream_of(kernel)))  # fmt: skip
    return out


def awq_gemm_w4a16(
    in_feats: torch.Tensor,
    kernel: torch.Tensor,
    scaling_factors: torch.Tensor,
    zeros: torch.Tensor,
    group_size: int = 128,
) -> torch.Tensor:
    """
    AWQ W4A16 GEMM for larger batches (reference: nunchaku/ops/triton/awq.py:232-251, there a dense decode and a library
    product): the weight is decoded, and rounded to the input dtype, inside the GEMM; with more than 2048 rows, too few columns
    for a long ``k``, or where ``in_feats`` wants a gradient or is under a transform, it is decoded to memory once by
    :func:`awq_dequantize` for a library product.
    """
    _lib.require_cuda(in_feats, kernel, scaling_factors, zeros)
    shape = in_feats.shape
    k = shape[-1]
    x = in_feats.reshape(-1, k)
    n = scaling_factors.shape[-1]
    return _product(x, kernel, scaling_factors, zeros, n, k, group_size).reshape(*shape[:-1], n)


def gemv_awq(in_feats, kernel, scaling_factors, zeros, m: int, n: int, k: int, group_size: int) -> torch.Tensor:
    """The reference's dispatcher name for :func:`awq_gemv_w4a16_cuda` (nunchaku/ops/dispatch.py:19-34)."""
    return awq_gemv_w4a16_cuda(in_feats, kernel, scaling_factors, zeros, m, n, k, group_size)


def gemm_awq(in_feats, kernel, scaling_factors, zeros) -> torch.Tensor:
    """The reference's dispatcher name for :func:`awq_gemm_w4a16` (nunchaku/ops/dispatch.py:37-49)."""
    return awq_gemm_w4a16(in_feats, kernel, scaling_factors, zeros)
