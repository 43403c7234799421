"""Composite operators (reference: nunchaku/ops/fused.py:15-253): quantize -> GEMM (fused epilogue) -> GEMM."""

from __future__ import annotations

import torch

from .gemm import svdq_gemm_w4a4_cuda

SWIGLU_BLOCK = 16


def _ceil_divide(a: int, b: int) -> int:
    return (a + b - 1) // b


def _row_block(pad_size: int) -> int:
    """What the buffers between the two GEMMs are padded to.  fc1's epilogue requantizes every row of its buffers, so rows up to
    ``pad_size`` are computed for nobody; the kernels ask for whole blocks of 32 only.  us per call, 256 / 32 (bf16,
    K = 3072, hidden 12288): SwiGLU 32 rows 67.3 / 53.1, 333 rows 97.0 / 91.9, 1100 rows 188 / 183, GELU 2100 rows 217 / 211;
    K = 1536, hidden 6144: GELU 32 rows 38.5 / 34.7, 600 rows 47.8 / 44.1; multiples of 256 as before.
    (Fewer rows may bring in the kernel that splits K: the last bits of a row's sums are then that kernel's.)"""
    return 32 if pad_size > 0 and pad_size % 32 == 0 else pad_size


def fused_gelu_mlp(x: torch.Tensor, fc1, fc2, pad_size: int = 256, norm: tuple | None = None) -> torch.Tensor:
    """``fc2(gelu_tanh(fc1(x)))`` for two ``SVDQW4A4Linear`` layers: fc1's GEMM applies GELU, fc2's LoRA-down and
    fc2's (unsigned, +0.171875) int4 quantization in its epilogue, so the hidden activation never reaches memory in
    16 bits.  ``x`` is ``(B, S, C_in)``; returns ``(B, S, C_out)``.  ``norm``: LayerNorm + modulate of ``x`` inside
    fc1's quantizer (see ``ops.quantize``; not in the reference's signature)."""
    batch_size, seq_len, channels = x.shape
    x = x.view(batch_size * seq_len, channels)
    in_pad = 256  # (buffers padded otherwise than fc1's input are refused by the GEMM)
    if _ceil_divide(batch_size * seq_len, pad_size) * pad_size == _ceil_divide(batch_size * seq_len, in_pad) * in_pad:
        in_pad = pad_size = _row_block(pad_size)
    in_blocked = fc1.takes_blocked(batch_size * seq_len, in_pad)     # fc1's input and fc2's input (fc1's requantized output)
    mid_blocked = fc2.takes_blocked(batch_size * seq_len, pad_size)  # in the order their GEMMs read them
    quantized_x, ascales, lora_act = fc1.quantize(x, pad_size=in_pad, norm=norm, blocked=in_blocked)

    batch_size_pad = _ceil_divide(batch_size * seq_len, pad_size) * pad_size
    qout_act = torch.empty(batch_size_pad, fc1.out_features * (3 if mid_blocked >= 2 else 2) // 4, dtype=torch.uint8, device=x.device)
    qout_ascales = torch.empty(fc1.out_features // 64, batch_size_pad, dtype=x.dtype, device=x.device)
    qout_lora_act = torch.empty(batch_size_pad, fc2.proj_down.shape[1], dtype=torch.float32, device=x.device)

    svdq_gemm_w4a4_cuda(
        act=quantized_x,
        wgt=fc1.qweight,
        qout=qout_act,
        ascales=ascales,
        wscales=fc1.wscales,
        oscales=qout_ascales,
        lora_act_in=lora_act,
        lora_up=fc1.proj_up,
        lora_down=fc2.proj_down,
        lora_act_out=qout_lora_act,
        bias=fc1.bias,
        smooth_factor=fc2.smooth_factor,
        fp4=False,
        alpha=fc1.wtscale,
        wcscales=fc1.wcscales,
        act_blocked=in_blocked,
        qout_blocked=mid_blocked,
    )
    output = torch.empty(batch_size * seq_len, fc2.out_features, dtype=x.dtype, device=x.device)
    output = fc2.forward_quant(qout_act, qout_ascales, qout_lora_act, output=output, act_blocked=mid_blocked)
    return output.view(batch_size, seq_len, -1)


def interleave_swiglu(n: int, device=None) -> torch.Tensor:
    """Row order for a ``[gate (n/2) | up (n/2)]`` projection: 16-row blocks gate, up, gate, up, ...
    (reference: nunchaku/ops/triton/native/w4a4.py:350-360)."""
    h, b = n // 2, SWIGLU_BLOCK
    g = torch.arange(h, device=device).view(h // b, b)
    return torch.stack([g, g + h], dim=1).reshape(-1)


def interleave_swiglu_linear_(linear, up_first: bool = False) -> None:
    """Reorder a SwiGLU input projection's output rows in place for :func:`fused_swiglu_mlp` (call once)."""
    assert linear.precision != "nvfp4" and linear.out_features % 64 == 0
    if hasattr(linear, "restore_packed_weight"):
        linear.restore_packed_weight()  # a released packed weight is rebuilt first: its rows are about to move
    idx = interleave_swiglu(linear.out_features, linear.qweight.device)
    if up_first:
        idx = (idx + linear.out_features // 2) % linear.out_features
    with torch.no_grad():
        linear.qweight.data = linear.qweight.data[idx].contiguous()
        linear.wscales.data = linear.wscales.data[:, idx].contiguous()
        linear.proj_up.data = linear.proj_up.data[idx].contiguous()
        if linear.bias is not None:
            linear.bias.data = linear.bias.data[idx].contiguous()


def fused_swiglu_mlp(x: torch.Tensor, fc1, fc2, pad_size: int = 256) -> torch.Tensor:
    """``fc2(silu(gate) * up)`` with ``[gate | up] = fc1(x)``; fc1's rows interleaved by
    :func:`interleave_swiglu_linear_`; SwiGLU and fc2's signed int4 quantization fused into fc1's GEMM."""
    shape = x.shape
    x = x.reshape(-1, shape[-1])
    M = x.shape[0]
    pad_size = _row_block(pad_size)
    in_blocked, mid_blocked = fc1.takes_blocked(M, pad_size), fc2.takes_blocked(M, pad_size)
    quantized_x, ascales, lora_act = fc1.quantize(x, pad_size=pad_size, blocked=in_blocked)
    M_pad = quantized_x.shape[0]
    H = fc2.in_features
    qout_act = torch.empty(M_pad, H * (3 if mid_blocked >= 2 else 2) // 4, dtype=torch.uint8, device=x.device)
    qout_ascales = torch.empty(H // 64, M_pad, dtype=x.dtype, device=x.device)
    qout_lora_act = torch.empty(M_pad, fc2.proj_down.shape[1], dtype=torch.float32, device=x.device)
    svdq_gemm_w4a4_cuda(
        act=quantized_x,
        wgt=fc1.qweight,
        ascales=ascales,
        wscales=fc1.wscales,
        bias=fc1.bias,
        lora_act_in=lora_act,
        lora_up=fc1.proj_up,
        qout=qout_act,
        oscales=qout_ascales,
        smooth_factor=fc2.smooth_factor,
        lora_down=fc2.proj_down,
        lora_act_out=qout_lora_act,
        act_unsigned=fc1.act_unsigned,
        fuse_swiglu=True,
        act_blocked=in_blocked,
        qout_blocked=mid_blocked,
    )
    output = torch.empty(M, fc2.out_features, dtype=x.dtype, device=x.device)
    output = fc2.forward_quant(qout_act, qout_ascales, qout_lora_act, output=output, act_blocked=mid_blocked)
    return output.view(*shape[:-1], fc2.out_features)


def fused_qkv_norm_rottary(
    x: torch.Tensor,
    proj,
    norm_q=None,
    norm_k=None,
    rotary_emb: torch.Tensor | None = None,
    output: torch.Tensor | tuple[torch.Tensor, torch.Tensor, torch.Tensor] | None = None,
    attn_tokens: int = 0,
    norm: tuple | None = None,
) -> torch.Tensor:
    """Quantized QKV projection with per-head RMSNorm on Q and K and RoPE fused into the GEMM epilogue.
    ``norm_q``/``norm_k`` are RMSNorm modules without bias (their ``weight`` is used); ``rotary_emb`` is the natural
    ``(S, 64, 1, 2)`` float32 (sin, cos) table.  The tuple-output form (packed Q/K/V for the reference's fp16
    attention kernel) is not implemented.  ``norm``: LayerNorm + modulate of ``x`` inside the quantizer (see
    ``ops.quantize``; not in the reference's signature)."""
    for nm in (norm_q, norm_k):
        assert nm is None or (hasattr(nm, "weight") and getattr(nm, "bias", None) is None)
    batch_size, seq_len, channels = x.shape
    x = x.view(batch_size * seq_len, channels)
    blocked = proj.takes_blocked(batch_size * seq_len)
    quantized_x, ascales, lora_act = proj.quantize(x, norm=norm, blocked=blocked)
    if output is None:
        output = torch.empty(batch_size * seq_len, proj.out_features, dtype=x.dtype, device=x.device)
    if isinstance(output, tuple):
        assert len(output) == 3
        svdq_gemm_w4a4_cuda(
            act=quantized_x, wgt=proj.qweight, ascales=ascales, wscales=proj.wscales, lora_act_in=lora_act,
            lora_up=proj.proj_up, bias=proj.bias, alpha=proj.wtscale, wcscales=proj.wcscales,
            norm_q=norm_q.weight if norm_q is not None else None, norm_k=norm_k.weight if norm_k is not None else None,
            rotary_emb=rotary_emb, out_q=output[0], out_k=output[1], out_v=output[2], attn_tokens=attn_tokens,
            act_blocked=blocked,
        )  # fmt: skip
        return output
    svdq_gemm_w4a4_cuda(
        act=quantized_x,
        wgt=proj.qweight,
        out=output,
        ascales=ascales,
        wscales=proj.wscales,
        lora_act_in=lora_act,
        lora_up=proj.proj_up,
        bias=proj.bias,
        fp4=False,
        alpha=proj.wtscale,
        wcscales=proj.wcscales,
        norm_q=norm_q.weight if norm_q is not None else None,
        norm_k=norm_k.weight if norm_k is not None else None,
        rotary_emb=rotary_emb,
        act_blocked=blocked,
    )
    return output.view(batch_size, seq_len, -1)
