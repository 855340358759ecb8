"""`attention` with the reference's signature (python/ac4k_kernel/ops/attention.py:193-241): for
precision="nvfp4" the three quantize calls of `_nvfp4_attention` (:100-133) followed by the HIP `mha_nvfp4_fwd`;
for precision="int8+fp8e4m3" the front end of `_int8_x_fp8_attention` (:137-190: K minus its token mean, per-token-block
int8 quantization of Q and K, per-row e4m3 quantization of V) followed by the HIP `mha_int8_x_fp8_fwd`.  Head dims up to 128."""
from __future__ import annotations

import math

import torch

from .. import _rocm_ops
from .quant import quantize

mha_nvfp4_fwd = _rocm_ops.mha_nvfp4_fwd
mha_int8_x_fp8_fwd = _rocm_ops.mha_int8_x_fp8_fwd


def _int8_quantize(x, layout, dim, type="token", BLOCK_SIZE=64, HDIM_ALIGN=16):
    """python/ac4k_kernel/ops/attention.py:51-99: -> (y int8 [B,H,N,align_up(D,16)], scale fp32 [B,H,ceil(N/BLOCK_SIZE)])."""
    assert HDIM_ALIGN == 16, "HDIM_ALIGN must be 16"
    assert type == "token", "Only support token quantization yet."
    assert BLOCK_SIZE >= 16
    assert (BLOCK_SIZE & (BLOCK_SIZE - 1)) == 0
    assert layout in ["BNHD", "BHND"], "Unsupported layout: {}".format(layout)
    assert dim in ([1, 3] if layout == "BNHD" else [2, 3])
    if x.stride(3) != 1:
        x = x.contiguous()
    x_bhnd = x.permute(0, 2, 1, 3) if layout == "BNHD" else x
    B, H, N, D = x_bhnd.shape
    scale = torch.empty([B, H, -(-x.shape[dim] // BLOCK_SIZE)], device=x.device, dtype=torch.float32)
    y = torch.empty([B, H, N, (D + 15) // 16 * 16], device=x.device, dtype=torch.int8)
    _rocm_ops.quantize_int8_token_block(y, scale, x_bhnd, BLOCK_SIZE)
    return y, scale


def _as_bhnd(layout, *operands):
    """Views of [B,H,N,D]; operands of [B,N,H,D] with another number of dims are refused here (RuntimeError)."""
    return tuple(t.permute(0, 2, 1, 3) for t in operands) if layout == "BNHD" else operands


def _int8_x_fp8_attention(q, k, v, layout, Q_QUANTIZE_BLOCK_SIZE=64, K_QUANTIZE_BLOCK_SIZE=128, out=None):
    """INT8 (QK) x FP8 (PV) attention (python/ac4k_kernel/ops/attention.py:137-190)."""
    assert layout in ["BNHD", "BHND"], f"Unsupported layout: {layout}"
    B, Dqk = q.shape[0], q.shape[-1]
    Dv = v.shape[-1]
    if layout == "BNHD":
        Nq, H = q.shape[1], q.shape[2]
    else:
        H, Nq = q.shape[1], q.shape[2]
    if out is None:
        out_shape = (B, Nq, H, Dv) if layout == "BNHD" else (B, H, Nq, Dv)
        out = torch.empty(out_shape, dtype=torch.bfloat16, device=q.device)
    # the operator takes dense V only; everything else goes operator by operator
    if (Q_QUANTIZE_BLOCK_SIZE, K_QUANTIZE_BLOCK_SIZE) == (64, 128) and v.is_contiguous() and _rocm_ops.attention_int8_x_fp8(
            out, q, k, v, 2.25, 1 / math.sqrt(Dqk), layout == "BNHD"):
        return out
    o_bhnd = _as_bhnd(layout, out, q, k, v)[0]  # the kernel writes through the strides
    n_dim = 1 if layout == "BNHD" else 2
    k = k - k.mean(dim=n_dim, keepdim=True)
    q_int8, q_sf = _int8_quantize(q, layout, n_dim, BLOCK_SIZE=Q_QUANTIZE_BLOCK_SIZE)
    k_int8, k_sf = _int8_quantize(k, layout, n_dim, BLOCK_SIZE=K_QUANTIZE_BLOCK_SIZE)
    v_fp8, v_sf = quantize(v, 3, n_dim, swizzle=True, max_scale=2.25, precision="fp8e4m3")
    mha_int8_x_fp8_fwd(o_bhnd, q_int8, q_sf, Q_QUANTIZE_BLOCK_SIZE, k_int8, k_sf, K_QUANTIZE_BLOCK_SIZE, v_fp8, v_sf,
                       1 / math.sqrt(Dqk))
    return out


def _nvfp4_attention(q, k, v, layout, out=None):
    assert layout in ["BNHD", "BHND"], f"Unsupported layout: {layout}"
    B, Dqk = q.shape[0], q.shape[-1]
    Dv = v.shape[-1]
    if layout == "BNHD":
        Nq, H = q.shape[1], q.shape[2]
    else:
        H, Nq = q.shape[1], q.shape[2]
    if out is None:
        out_shape = (B, Nq, H, Dv) if layout == "BNHD" else (B, H, Nq, Dv)
        out = torch.empty(out_shape, dtype=torch.bfloat16, device=q.device)
    # the quantizers take dense tensors only; everything else goes operator by operator
    if q.is_contiguous() and k.is_contiguous() and v.is_contiguous() and _rocm_ops.attention_nvfp4(
            out, q, k, v, 1 / math.sqrt(Dqk), layout == "BNHD"):
        return out
    o_bhnd = _as_bhnd(layout, out, q, k, v)[0]  # the kernel writes through the strides
    n_dim = 1 if layout == "BNHD" else 2
    q_fp4, q_sf, q_alpha = quantize(q, n_dim, 3)
    k_fp4, k_sf, k_alpha = quantize(k, n_dim, 3)
    v_fp4, v_sf, v_alpha = quantize(v, 3, n_dim, swizzle=True)
    mha_nvfp4_fwd(o_bhnd, q_fp4, q_sf, q_alpha, k_fp4, k_sf, k_alpha, v_fp4, v_sf, v_alpha, 1 / math.sqrt(Dqk))
    return out


def attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, *, layout: str = "BNHD", precision: str = "int8+fp8e4m3",
              out: torch.Tensor = None) -> torch.Tensor:
    """Multi-head attention on bf16 q, k, v of [B, N, H, D] (layout "BNHD") or [B, H, N, D] ("BHND"); returns bf16 in
    the same layout.  precision "int8+fp8e4m3" (the reference's default): QK^T on int8, PV on e4m3; "nvfp4": both
    products on NVFP4 operands.  Head dim at most 128."""
    assert q.dtype == torch.bfloat16, "q dtype must be bfloat16"
    assert k.dtype == torch.bfloat16, "k dtype must be bfloat16"
    assert v.dtype == torch.bfloat16, "v dtype must be bfloat16"
    assert layout in ["BNHD", "BHND"], f"Unsupported layout: {layout}"
    assert precision in ["nvfp4", "int8+fp8e4m3"], f"Unsupported precision: {precision}"
    if out is not None:
        assert out.dtype == torch.bfloat16, "out dtype must be bfloat16"
    if precision == "int8+fp8e4m3":
        return _int8_x_fp8_attention(q, k, v, layout, out=out)
    return _nvfp4_attention(q, k, v, layout, out=out)
