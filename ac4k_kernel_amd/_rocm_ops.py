"""Tensor-level binding over the C ABI: the module the reference's package would import as
`ac4k_kernel._rocm_ops` (python/ac4k_kernel/__init__.py:39-48), with the function names and
positional arguments of `_cuda_ops` (lib/cuda_bindings.cc:64-85, include/ac4k_kernel/ops.h:27-48).

All functions write into caller-provided tensors, return None, enqueue on the current
torch stream and never synchronise.  Argument checks mirror the reference host launchers'
TORCH_CHECKs and raise RuntimeError.
"""
from __future__ import annotations

import torch

from . import _lib

_L = _lib.load()

__arch__ = _L.ac4k_arch().decode()
__arch_description__ = _L.ac4k_arch_description().decode()
__backend__ = _L.ac4k_backend().decode()
__version__ = _L.ac4k_version().decode()

_DTYPE_TAG = {torch.bfloat16: 0, torch.float16: 1, torch.float32: 2}


def _check(cond: bool, msg: str, *args) -> None:
    """RuntimeError(msg.format(*args)) unless cond; the message is only built on failure."""
    if not cond:
        raise RuntimeError(msg.format(*args) if args else msg)


def _check_tensor(t, dtype, name: str, suffix: str = "") -> None:
    # one combined test on the hot path; the individual messages are only built on failure
    if isinstance(t, torch.Tensor) and t.is_cuda and t.dtype == dtype and t.is_contiguous():
        return
    name += suffix
    _check(isinstance(t, torch.Tensor), "{} must be a tensor", name)
    _check(t.is_cuda, "{} must be a CUDA tensor", name)
    _check(t.is_contiguous(), "{} must be contiguous", name)
    _check(t.dtype == dtype, "Inconsistency of Tensor type: {} must be {}", name, dtype)


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_current_device = getattr(torch._C, "_cuda_getDevice", torch.cuda.current_device)  # operands on a GPU: torch is initialised


def _stream() -> int:
    """hipStream_t of torch's current stream on the current device."""
    if _raw_stream is not None:
        return _raw_stream(_current_device())
    return torch.cuda.current_stream().cuda_stream


def _align_up(a: int, b: int) -> int:
    return (a + b - 1) // b * b


def _quant_geometry(inp: torch.Tensor, cross_dim: int, reduce_dim: int):
    """Checks shared by the three quantizers (quantize_nvfp4.cu:171-190,226-241)."""
    _check_tensor(inp, torch.bfloat16, "in")
    _check(2 <= inp.dim() <= 4, "in must be 2-4D")
    _check(0 <= cross_dim < inp.dim(), "cross_dim must be less than in.dim()")
    _check(0 <= reduce_dim < inp.dim(), "reduce_dim must be less than in.dim()")
    _check(cross_dim != reduce_dim, "cross_dim and reduce_dim must be different")
    if inp.dim() == 2:
        shape, stride = inp.shape, inp.stride()
        _check(shape[0] > 0 and shape[1] > 0, "in must not be empty")
        return [], (1, 1, shape[cross_dim], shape[reduce_dim], 0, 0, stride[cross_dim], stride[reduce_dim])
    shape, stride = list(inp.shape), list(inp.stride())
    lead = [i for i in range(inp.dim()) if i not in (cross_dim, reduce_dim)]
    lead_shape = [shape[i] for i in lead]
    ld = [(shape[i], stride[i]) for i in lead]
    while len(ld) < 2:
        ld.insert(0, (1, 0))
    (d0, s0), (d1, s1) = ld
    _check(inp.numel() > 0, "in must not be empty")
    return lead_shape, (d0, d1, shape[cross_dim], shape[reduce_dim], s0, s1, stride[cross_dim], stride[reduce_dim])


def global_scale(out: torch.Tensor, inp: torch.Tensor, max_scale: float) -> None:
    """out (0-dim fp32) = amax(|inp|) / max_scale  (python/ac4k_kernel/ops/quant.py:33-59)."""
    _check_tensor(inp, torch.bfloat16, "in")
    _check_tensor(out, torch.float32, "global_scale")
    _check(out.dim() == 0, "global_scale must be a scalar")
    _lib.check(_L.ac4k_global_scale_bf16(out.data_ptr(), inp.data_ptr(), inp.numel(), float(max_scale), _stream()))


def quantize_nvfp4(out, sf, inp, global_scale, cross_dim: int, reduce_dim: int, swizzle: bool) -> None:
    lead_shape, geom = _quant_geometry(inp, cross_dim, reduce_dim)
    R, K = geom[2], geom[3]
    _check_tensor(global_scale, torch.float32, "global_scale")
    _check(global_scale.dim() == 0, "global_scale must be a scalar")
    _check_tensor(out, torch.uint8, "out")
    _check(list(out.shape) == lead_shape + [R, _align_up(K, 64) // 2],
           "out must have shape [.., cross, align_up(reduce, 64) / 2]")
    _check_tensor(sf, torch.float8_e4m3fn, "sf")
    _check(list(sf.shape) == lead_shape + [_align_up(K, 64) // 64, _align_up(R, 16), 4], "meet invalid sf shape")
    _lib.check(_L.ac4k_quantize_nvfp4(out.data_ptr(), sf.data_ptr(), inp.data_ptr(), global_scale.data_ptr(),
                                      *geom, int(bool(swizzle)), _stream()))


def quantize_nvfp4_with_global_scale(out, sf, global_scale, inp, cross_dim: int, reduce_dim: int, swizzle: bool,
                                     max_scale: float) -> None:
    """global_scale (written) = amax(|inp|) / max_scale, then quantize_nvfp4 with it: the nvfp4 branch
    of the reference's Ac4kQuantizeOp.forward (quant.py:187-242) behind one C call."""
    lead_shape, geom = _quant_geometry(inp, cross_dim, reduce_dim)
    R, K = geom[2], geom[3]
    _check_tensor(global_scale, torch.float32, "global_scale")
    _check(global_scale.dim() == 0, "global_scale must be a scalar")
    _check_tensor(out, torch.uint8, "out")
    _check(list(out.shape) == lead_shape + [R, _align_up(K, 64) // 2],
           "out must have shape [.., cross, align_up(reduce, 64) / 2]")
    _check_tensor(sf, torch.float8_e4m3fn, "sf")
    _check(list(sf.shape) == lead_shape + [_align_up(K, 64) // 64, _align_up(R, 16), 4], "meet invalid sf shape")
    _quantize_nvfp4_bf16(out, sf, global_scale, inp, geom, swizzle, max_scale)


def quantize_nvfp4_new(inp, cross_dim: int, reduce_dim: int, swizzle: bool, max_scale: float):
    """The same into tensors made here, which need no checks: (out, sf, global_scale)."""
    lead_shape, geom = _quant_geometry(inp, cross_dim, reduce_dim)
    R, Kp = geom[2], (geom[3] + 63) // 64 * 64
    dev = inp.device
    out = torch.empty([*lead_shape, R, Kp // 2], dtype=torch.uint8, device=dev)
    sf = torch.empty([*lead_shape, Kp // 64, (R + 15) // 16 * 16, 4], dtype=torch.float8_e4m3fn, device=dev)
    global_scale = torch.empty((), dtype=torch.float32, device=dev)
    _quantize_nvfp4_bf16(out, sf, global_scale, inp, geom, swizzle, max_scale)
    return out, sf, global_scale


def _quantize_nvfp4_bf16(out, sf, global_scale, inp, geom, swizzle, max_scale) -> None:
    _lib.check(_L.ac4k_quantize_nvfp4_bf16(out.data_ptr(), sf.data_ptr(), global_scale.data_ptr(), inp.data_ptr(),
                                           *geom, int(bool(swizzle)), float(max_scale), _stream()))


def _quantize_rowwise(fn, out, out_dtype, sf, inp, scale_max, scale_dtype, cross_dim, reduce_dim, *extra):
    lead_shape, geom = _quant_geometry(inp, cross_dim, reduce_dim)
    R, K = geom[2], geom[3]
    _check_tensor(scale_max, scale_dtype, "scale_max")
    _check(scale_max.dim() == 0, "scale_max must be a scalar")
    _check_tensor(out, out_dtype, "out")
    _check(list(out.shape) == lead_shape + [R, _align_up(K, 16)], "out must have shape [.., cross, align_up(reduce, 16)]")
    _check_tensor(sf, torch.float32, "sf")
    _check(list(sf.shape) == lead_shape + [_align_up(R, 16)], "meet invalid sf shape")
    _lib.check(fn(out.data_ptr(), sf.data_ptr(), inp.data_ptr(), scale_max.data_ptr(), *geom, *extra, _stream()))


def quantize_fp8(out, sf, inp, scale_max, cross_dim: int, reduce_dim: int, swizzle: bool) -> None:
    _quantize_rowwise(_L.ac4k_quantize_fp8, out, torch.float8_e4m3fn, sf, inp, scale_max, torch.float32,
                      cross_dim, reduce_dim, int(bool(swizzle)))


def quantize_int8(out, sf, inp, scale_max, cross_dim: int, reduce_dim: int) -> None:
    _quantize_rowwise(_L.ac4k_quantize_int8, out, torch.int8, sf, inp, scale_max, torch.int32,
                      cross_dim, reduce_dim)


def _check_linear_operand(x, x_sf, x_gs, rows, name):
    # one pass over the attributes of a well-formed operand; what is wrong with another one is found out below
    if isinstance(x, torch.Tensor) and isinstance(x_sf, torch.Tensor) and isinstance(x_gs, torch.Tensor) and x.dim() == 2:
        K = x.size(1) * 2
        if (x.dtype is torch.uint8 and x.is_cuda and x.is_contiguous()
                and x_sf.dtype is torch.float8_e4m3fn and x_sf.is_cuda and x_sf.is_contiguous()
                and x_sf.shape == ((K + 63) // 64, (rows + 15) // 16 * 16, 4)
                and x_gs.dtype is torch.float32 and x_gs.is_cuda and x_gs.dim() == 0):
            return K
    _check(x.dim() == 2, "{} must be a 2d matrix", name)
    _check_tensor(x, torch.uint8, name)
    K = x.size(1) * 2
    _check(x_sf.dim() == 3, "scale_{} must be a 3d matrix", name)
    _check_tensor(x_sf, torch.float8_e4m3fn, "scale_", name)
    _check(x_sf.shape == ((K + 63) // 64, _align_up(rows, 16), 4), "scale_{} has an invalid shape", name)
    _check_tensor(x_gs, torch.float32, "global_scale_", name)
    _check(x_gs.dim() == 0, "{}_global_scale must be a scalar", name)
    return K


def _bias_args(bias, N):
    if bias is None:
        return None, 0
    _check(bias.dtype in _DTYPE_TAG, "bias must be bfloat16, half or float")
    _check(bias.is_cuda and bias.is_contiguous(), "bias must be contiguous")
    _check(bias.dim() == 2, "bias must be a 2d matrix")
    _check(bias.size(0) == 1, "bias shape[0] must be 1")
    _check(bias.size(1) == N, "bias shape[1] must be {}", N)
    return bias.data_ptr(), _DTYPE_TAG[bias.dtype]


def _check_output(D):
    if isinstance(D, torch.Tensor) and D.dim() == 2 and D.is_cuda and D.is_contiguous():
        tag = _DTYPE_TAG.get(D.dtype)
        if tag is not None:
            return D.size(0), D.size(1), tag
    _check(isinstance(D, torch.Tensor) and D.dim() == 2, "d must be a 2d matrix")
    _check(D.dtype in _DTYPE_TAG, "d must be bfloat16, half or float")
    _check(False, "d must be contiguous")


def linear_nvfp4(D, A, A_sf, A_global_scale, B, B_sf, B_global_scale, bias=None) -> None:
    """Checks of linear_nvfp4.cu:759-805.  Shapes for which the library asks for scratch (too few output
    tiles for the GPU, long K) get a workspace tensor and the split-K kernels; everything else goes to
    the reference-shaped entry point, which allocates nothing and picks its kernel by shape."""
    M, N, tag = _check_output(D)
    if A.dim() != 2 or A.size(0) != M:
        _check(False, "A size(0) must be {}", M)
    K = _check_linear_operand(A, A_sf, A_global_scale, M, "a")
    if K % 16 != 0:
        _check(False, "A size(1)*2 must be multiple of 16 but see {}", K)
    if B.dim() != 2 or B.size(1) * 2 != K:
        _check(False, "B size(1) must equal A size(1)")
    if B.size(0) != N:
        _check(False, "B size(0) must be {}", N)
    _check_linear_operand(B, B_sf, B_global_scale, N, "b")
    bias_ptr, bias_tag = (None, 0) if bias is None else _bias_args(bias, N)
    if M == 0 or N == 0:
        return
    nbytes = _L.ac4k_linear_nvfp4_scratch_bytes(M, N, K)
    if nbytes > 0:
        ws = D.new_empty((nbytes,), dtype=torch.uint8)
        _lib.check(_L.ac4k_linear_nvfp4_workspace(D.data_ptr(), tag, A.data_ptr(), A_sf.data_ptr(),
                                                  A_global_scale.data_ptr(), B.data_ptr(), B_sf.data_ptr(),
                                                  B_global_scale.data_ptr(), bias_ptr, bias_tag, M, N, K,
                                                  ws.data_ptr(), nbytes, _stream()))
        return
    _lib.check(_L.ac4k_linear_nvfp4(D.data_ptr(), tag, A.data_ptr(), A_sf.data_ptr(),
                                    A_global_scale.data_ptr(), B.data_ptr(), B_sf.data_ptr(),
                                    B_global_scale.data_ptr(), bias_ptr, bias_tag, M, N, K, _stream()))


def prepack_weight_nvfp4(B, B_sf) -> torch.Tensor:
    """Weight image of B [N, K/2] / B_sf [K/64, align_up(N,16), 4] for linear_nvfp4_prepacked: a uint8
    tensor of ac4k_prepack_weight_nvfp4_bytes(N, K) bytes.  K must be a multiple of 128."""
    _check(B.dim() == 2, "b must be a 2d matrix")
    _check_tensor(B, torch.uint8, "b")
    N, K = B.size(0), B.size(1) * 2
    _check(B_sf.dim() == 3, "scale_b must be a 3d matrix")
    _check_tensor(B_sf, torch.float8_e4m3fn, "scale_", "b")
    _check(B_sf.shape == ((K + 63) // 64, _align_up(N, 16), 4), "scale_b has an invalid shape")
    nbytes = _L.ac4k_prepack_weight_nvfp4_bytes(N, K)
    _check(nbytes > 0, "no weight image for N = {}, K = {}: K must be a multiple of 128", N, K)
    image = torch.empty((nbytes,), dtype=torch.uint8, device=B.device)
    _lib.check(_L.ac4k_prepack_weight_nvfp4(image.data_ptr(), B.data_ptr(), B_sf.data_ptr(), N, K, _stream()))
    return image


def linear_nvfp4_prepacked(D, A, A_sf, A_global_scale, W_image, B_global_scale, bias=None) -> None:
    """linear_nvfp4 on a weight image made by prepack_weight_nvfp4 (N = D.size(1), K = 2 * A.size(1))."""
    M, N, tag = _check_output(D)
    _check(A.dim() == 2 and A.size(0) == M, "A size(0) must be {}", M)
    K = _check_linear_operand(A, A_sf, A_global_scale, M, "a")
    _check_tensor(W_image, torch.uint8, "w_image")
    _check(N > 0 and W_image.numel() == _L.ac4k_prepack_weight_nvfp4_bytes(N, K) and W_image.numel() > 0,
           "w_image is not the weight image of a [{}, {}] weight", N, K)
    _check_tensor(B_global_scale, torch.float32, "global_scale_", "b")
    _check(B_global_scale.dim() == 0, "b_global_scale must be a scalar")
    bias_ptr, bias_tag = _bias_args(bias, N)
    if M == 0:
        return
    nbytes = _L.ac4k_linear_nvfp4_prepacked_workspace_bytes(M, N, K)
    ws = D.new_empty((nbytes,), dtype=torch.uint8) if nbytes > 0 else None
    _lib.check(_L.ac4k_linear_nvfp4_prepacked(D.data_ptr(), tag, A.data_ptr(), A_sf.data_ptr(),
                                              A_global_scale.data_ptr(), W_image.data_ptr(),
                                              B_global_scale.data_ptr(), bias_ptr, bias_tag, M, N, K,
                                              None if ws is None else ws.data_ptr(), nbytes, _stream()))


def linear_nvfp4_fused(D, X, X_q, X_sf, X_global_scale, B, B_sf, B_global_scale, bias=None) -> None:
    """quantize(X, 0, 1) + linear_nvfp4 for a bf16 activation X [M, K], 1 <= M <= 32;
    X_q / X_sf / X_global_scale receive the quantized activation."""
    M, N, tag = _check_output(D)
    K = _check_fused_activation(X, M)
    _check_tensor(X_q, torch.uint8, "x_q")
    _check(list(X_q.shape) == [M, K // 2], "x_q must be [M, K/2]")
    _check_linear_operand(X_q, X_sf, X_global_scale, M, "x")
    _check(B.dim() == 2 and B.size(0) == N and B.size(1) == K // 2, "weight must be [N, K/2]")
    _check_linear_operand(B, B_sf, B_global_scale, N, "b")
    bias_ptr, bias_tag = _bias_args(bias, N)
    if K % 256 != 0:  # the C entry point takes whole stages of the kernels it began with: the composition itself, same kernels
        quantize_nvfp4_with_global_scale(X_q, X_sf, X_global_scale, X, 0, 1, False, 2688.0)
        linear_nvfp4(D, X_q, X_sf, X_global_scale, B, B_sf, B_global_scale, bias)
        return
    nbytes = _L.ac4k_linear_nvfp4_workspace_bytes(M, N, K)  # 0: one K range per tile, no scratch
    ws = D.new_empty((nbytes,), dtype=torch.uint8) if nbytes > 0 else None
    _lib.check(_L.ac4k_linear_nvfp4_fused_bf16(D.data_ptr(), tag, X.data_ptr(), X_q.data_ptr(),
                                               X_sf.data_ptr(), X_global_scale.data_ptr(), B.data_ptr(),
                                               B_sf.data_ptr(), B_global_scale.data_ptr(), bias_ptr, bias_tag,
                                               M, N, K, None if ws is None else ws.data_ptr(), nbytes, _stream()))


def _check_fused_activation(X, M):
    _check_tensor(X, torch.bfloat16, "x")
    _check(X.dim() == 2 and X.size(0) == M, "x must be [{}, K]", M)
    _check(1 <= M <= 32, "the fused linear takes 1 <= M <= 32")
    K = X.size(1)
    _check(K % 64 == 0, "K must be a multiple of 64")
    return K


def linear_nvfp4_fused_scratch(D, X, B, B_sf, B_global_scale, bias=None) -> bool:
    """linear_nvfp4_fused for a caller who does not ask for the quantized activation: it and the workspace are one allocation.
    False, with nothing done, for a K that runs as the composition."""
    M, N, tag = _check_output(D)
    K = _check_fused_activation(X, M)
    if K == 0 or K % 256 != 0:
        return False
    _check(B.dim() == 2 and B.size(0) == N and B.size(1) == K // 2, "weight must be [N, K/2]")
    _check_linear_operand(B, B_sf, B_global_scale, N, "b")
    bias_ptr, bias_tag = (None, 0) if bias is None else _bias_args(bias, N)
    nbytes = _L.ac4k_linear_nvfp4_workspace_bytes(M, N, K)  # 0: one K range per tile, no scratch
    q_bytes, sf_bytes = _align_up(M * K // 2, 256), K // 64 * _align_up(M, 16) * 4  # (a multiple of 256: K % 256 == 0)
    ws_bytes = _align_up(nbytes, 256)
    ws = D.new_empty((ws_bytes + q_bytes + sf_bytes + 4,), dtype=torch.uint8)
    at = ws.data_ptr()
    q = at + ws_bytes
    _lib.check(_L.ac4k_linear_nvfp4_fused_bf16(D.data_ptr(), tag, X.data_ptr(), q, q + q_bytes, q + q_bytes + sf_bytes, B.data_ptr(),
                                               B_sf.data_ptr(), B_global_scale.data_ptr(), bias_ptr, bias_tag,
                                               M, N, K, at if nbytes > 0 else None, nbytes, _stream()))
    return True


def _check_attention_operand(x, x_sf, x_gs, B, H, rows, width, name):
    """One packed operand of mha_nvfp4_fwd: x [B,H,rows,width/2], x_sf [B,H,ceil(width/64),align_up(rows,16),4]
    (mha_nvfp4.cu:917-1003)."""
    _check_tensor(x, torch.uint8, name)
    _check(x.dim() == 4 and list(x.shape) == [B, H, rows, width // 2], "{} must be [{}, {}, {}, {}]", name, B, H, rows, width // 2)
    _check_tensor(x_sf, torch.float8_e4m3fn, name + "_sf")
    _check(x_sf.dim() == 5, "{}_sf must be a 5D tensor", name)
    _check(list(x_sf.shape) == [B, H, (width + 63) // 64, _align_up(rows, 16), 4], "Meet invalid {}_sf size", name)
    _check_tensor(x_gs, torch.float32, name + "_global_scale")
    _check(x_gs.dim() == 0, "{}_global_scale must be a float tensor", name)


def mha_nvfp4_fwd(o, q, q_sf, q_global_scale, k, k_sf, k_global_scale, v, v_sf, v_global_scale, sm_scale: float) -> None:
    """Checks of mha_nvfp4.cu:917-1012.  o may be a permuted view (the reference's caller passes one): only its
    shape [B,H,Nq,Dv], dtype and device are checked."""
    _check(isinstance(q, torch.Tensor) and q.dim() == 4, "Q must be a 4D tensor")
    B, H, Nq = q.size(0), q.size(1), q.size(2)
    Dqk = q.size(3) * 2
    _check(Dqk % 16 == 0, "Dqk must be multiple of 16")
    _check(Dqk <= 128, "Dqk must be less than 128")
    _check(isinstance(k, torch.Tensor) and k.dim() == 4, "K must be a 4D tensor")
    _check(k.size(0) == B, "K must have the same batch size as Q")
    _check(k.size(1) == H, "K must have the same head number as Q")
    _check(k.size(3) == q.size(3), "K must have the same dim as Q")
    Nkv = k.size(2)
    _check(isinstance(v, torch.Tensor) and v.dim() == 4, "V must be a 4D tensor")
    Dv = v.size(2)
    _check(Dv <= 128, "Dv must be less than 128")
    _check(v.size(3) * 2 == _align_up(Nkv, 64), "V must have the same sequence length as K")
    _check_attention_operand(q, q_sf, q_global_scale, B, H, Nq, Dqk, "q")
    _check_attention_operand(k, k_sf, k_global_scale, B, H, Nkv, Dqk, "k")
    _check_attention_operand(v, v_sf, v_global_scale, B, H, Dv, _align_up(Nkv, 64), "v")
    _check(isinstance(o, torch.Tensor) and o.is_cuda, "O must be a CUDA tensor")
    _check(o.dtype == torch.bfloat16, "O must be a bfloat16 tensor")
    _check(o.dim() == 4 and list(o.shape) == [B, H, Nq, Dv], "O must be [{}, {}, {}, {}]", B, H, Nq, Dv)
    if B == 0 or H == 0 or Nq == 0:
        return
    _check(Nkv > 0, "K must not be empty")
    _lib.check(_L.ac4k_mha_nvfp4_fwd(o.data_ptr(), *o.stride(), q.data_ptr(), q_sf.data_ptr(), q_global_scale.data_ptr(),
                                     k.data_ptr(), k_sf.data_ptr(), k_global_scale.data_ptr(), v.data_ptr(), v_sf.data_ptr(),
                                     v_global_scale.data_ptr(), B, H, Nq, Nkv, Dqk, Dv, float(sm_scale), _stream()))


def mha_int8_x_fp8_fwd(o, q, q_sf, q_quantize_block_size: int, k, k_sf, k_quantize_block_size: int, v, v_sf,
                       sm_scale: float) -> None:
    """Checks of mha_int8_x_fp8.cu:982-1044.  o may be a permuted view: only its shape [B,H,Nq,Dv], dtype and
    device are checked."""
    _check_tensor(q, torch.int8, "Q")
    _check(q.dim() == 4, "Q must be a 4D tensor")
    B, H, Nq, Dqk = q.size(0), q.size(1), q.size(2), q.size(3)
    _check(Dqk % 16 == 0, "Dqk must be multiple of 16")
    _check(Dqk <= 128, "Dqk must be less than 128")
    _check_tensor(q_sf, torch.float32, "Q_SF")
    _check(q_sf.dim() == 3, "Q_SF must be a 3D tensor")
    _check(list(q_sf.shape) == [B, H, -(-Nq // q_quantize_block_size)], "Meet invalid Q_SF size")
    _check_tensor(k, torch.int8, "K")
    _check(k.dim() == 4, "K must be a 4D tensor")
    _check(k.size(0) == B, "K must have the same batch size as Q")
    _check(k.size(1) == H, "K must have the same head number as Q")
    _check(k.size(3) == Dqk, "K must have the same dim as Q")
    Nkv = k.size(2)
    _check_tensor(k_sf, torch.float32, "K_SF")
    _check(k_sf.dim() == 3, "K_SF must be a 3D tensor")
    _check(list(k_sf.shape) == [B, H, -(-Nkv // k_quantize_block_size)], "Meet invalid K_SF size")
    _check_tensor(v, torch.float8_e4m3fn, "V")
    _check(v.dim() == 4, "V must be a 4D tensor")
    _check(v.size(0) == B, "V must have the same batch size as Q")
    _check(v.size(1) == H, "V must have the same head number as Q")
    Dv = v.size(2)
    _check(v.size(3) == _align_up(Nkv, 16), "Meet invalid v size(3) with {}=={}", v.size(3), _align_up(Nkv, 16))
    _check(Dv <= 128, "Dv must be less than 128")
    _check_tensor(v_sf, torch.float32, "V_SF")
    _check(v_sf.dim() == 3 and list(v_sf.shape) == [B, H, _align_up(Dv, 16)], "Meet invalid v_sf size")
    _check(isinstance(o, torch.Tensor) and o.is_cuda, "O must be a CUDA tensor")
    _check(o.dtype == torch.bfloat16, "O must be a bfloat16 tensor")
    _check(o.dim() == 4 and list(o.shape) == [B, H, Nq, Dv], "O must be [{}, {}, {}, {}]", B, H, Nq, Dv)
    if B == 0 or H == 0 or Nq == 0:
        return
    _check(Nkv > 0, "K must not be empty")
    _lib.check(_L.ac4k_mha_int8_x_fp8_fwd(o.data_ptr(), *o.stride(), q.data_ptr(), q_sf.data_ptr(), int(q_quantize_block_size),
                                          k.data_ptr(), k_sf.data_ptr(), int(k_quantize_block_size), v.data_ptr(),
                                          v_sf.data_ptr(), B, H, Nq, Nkv, Dqk, Dv, float(sm_scale), _stream()))


def _attention(entry, workspace_bytes, o, q, k, v, scale: float, sm_scale: float, bnhd: bool) -> bool:
    try:
        if bnhd:
            (B, Nq, H, Dqk), (k_B, Nkv, k_H, k_D), (v_B, v_N, v_H, Dv), (o_B, o_N, o_H, o_D) = q.shape, k.shape, v.shape, o.shape
        else:
            (B, H, Nq, Dqk), (k_B, k_H, Nkv, k_D), (v_B, v_H, v_N, Dv), (o_B, o_H, o_N, o_D) = q.shape, k.shape, v.shape, o.shape
    except ValueError:  # not 4D
        return False
    dev, bf16 = q.get_device(), torch.bfloat16  # -1 on the CPU
    if not (B == k_B == v_B == o_B and H == k_H == v_H == o_H and Nkv == v_N and Nq == o_N and Dqk == k_D and Dv == o_D
            and dev >= 0 and dev == k.get_device() == v.get_device() == o.get_device()
            and q.dtype is bf16 and k.dtype is bf16 and v.dtype is bf16 and o.dtype is bf16):
        return False
    if bnhd:
        (q_b, q_n, q_h, q_d), (k_b, k_n, k_h, k_d), (v_b, v_n, v_h, v_d), (o_b, o_n, o_h, o_d) = q.stride(), k.stride(), v.stride(), o.stride()
    else:
        (q_b, q_h, q_n, q_d), (k_b, k_h, k_n, k_d), (v_b, v_h, v_n, v_d), (o_b, o_h, o_n, o_d) = q.stride(), k.stride(), v.stride(), o.stride()
    if q_d != 1 or k_d != 1 or v_d != 1:
        return False
    nbytes = workspace_bytes(B, H, Nq, Nkv, Dqk, Dv)
    if nbytes < 0:
        return False
    ws = q.new_empty((nbytes,), dtype=torch.uint8)
    _lib.check(entry(o.data_ptr(), o_b, o_h, o_n, o_d, q.data_ptr(), q_b, q_h, q_n, k.data_ptr(), k_b, k_h, k_n, v.data_ptr(), v_b, v_h, v_n,
                     B, H, Nq, Nkv, Dqk, Dv, scale, sm_scale, ws.data_ptr(), nbytes, _stream()))
    return True


def attention_int8_x_fp8(o, q, k, v, v_scale_max: float, sm_scale: float, bnhd: bool = False) -> bool:
    """The whole `_int8_x_fp8_attention` (python/ac4k_kernel/ops/attention.py:137-190) behind one C call on bf16 q, k, v
    of [B,H,N,D], or of [B,N,H,D] with `bnhd` (any batch, head and token strides).  False, with nothing done, for operands this call does not
    take - odd shapes, other dtypes and the ones an operator-by-operator call rejects with its own message."""
    return _attention(_L.ac4k_attention_int8_x_fp8_bf16, _L.ac4k_attention_int8_x_fp8_workspace_bytes, o, q, k, v, v_scale_max, sm_scale, bnhd)


def attention_nvfp4(o, q, k, v, sm_scale: float, bnhd: bool = False) -> bool:
    """The same for `_nvfp4_attention` (python/ac4k_kernel/ops/attention.py:100-133) on dense q, k, v."""
    return _attention(_L.ac4k_attention_nvfp4_bf16, _L.ac4k_attention_nvfp4_workspace_bytes, o, q, k, v, 2688.0, sm_scale, bnhd)


def quantize_int8_token_block(y, scale, x_bhnd, block: int) -> None:
    """y int8 [B,H,N,align_up(D,16)], scale fp32 [B,H,ceil(N/block)] <- x bf16 viewed as [B,H,N,D] (any batch, head and
    token strides, head dim contiguous): the per-token-block quantizer of python/ac4k_kernel/ops/attention.py:18-99."""
    _check(isinstance(x_bhnd, torch.Tensor) and x_bhnd.is_cuda and x_bhnd.dtype == torch.bfloat16, "x must be a CUDA bfloat16 tensor")
    _check(x_bhnd.dim() == 4 and x_bhnd.stride(3) == 1, "x must be 4D with a contiguous head dim")
    B, H, N, D = x_bhnd.shape
    _check_tensor(y, torch.int8, "y")
    _check(list(y.shape) == [B, H, N, _align_up(D, 16)], "Meet invalid y size")
    _check_tensor(scale, torch.float32, "scale")
    _check(list(scale.shape) == [B, H, -(-N // block)], "Meet invalid scale size")
    if x_bhnd.numel() == 0:
        return
    _lib.check(_L.ac4k_quantize_int8_token_block_bf16(y.data_ptr(), scale.data_ptr(), x_bhnd.data_ptr(), B, H, N, D,
                                                      x_bhnd.stride(0), x_bhnd.stride(1), x_bhnd.stride(2), int(block), _stream()))
