"""MXFP8 (OCP MX: E4M3 + one E8M0 scale per 32 elements along K) quantisation and GEMM, with an
optional fused SwiGLU epilogue, on the MI355X scaled fp8 matrix cores.

Counterparts of ``torch_npu.npu_dynamic_mx_quant`` and ``torch_npu.npu_quant_matmul(...,
group_sizes=[1, 1, 32])`` as used by the reference's MXFP8 linear layer
(mindiesd/quantization/layer.py:334-361)."""
import torch

from ... import _native
from ...utils.exception import ParametersInvalid


def mx_quantize(x):
    """[M, K] bf16/fp16 (row stride a multiple of 8, K % 32 == 0) ->
    (float8_e4m3fn [M, K], float8_e8m0fnu [M, K/32])."""
    if not isinstance(x, torch.Tensor) or x.dim() != 2 or not x.is_cuda or x.dtype not in _native.DTYPE_CODE:
        raise ParametersInvalid("mx_quantize needs a 2-D bf16/fp16 GPU tensor.")
    m, k = x.shape
    if k % 32 != 0:
        raise ParametersInvalid(f"mx_quantize needs K % 32 == 0, but got K = {k}.")
    if x.stride(1) != 1 or x.stride(0) % 8 != 0 or x.data_ptr() % 16 != 0:
        x = x.contiguous()
    q = torch.empty((m, k), dtype=torch.uint8, device=x.device)
    e = torch.empty((m, k // 32), dtype=torch.uint8, device=x.device)
    with _native.on_device(x.device):
        rc = _native.lib().mindiesd_mx_quant(x.data_ptr(), q.data_ptr(), e.data_ptr(), _native.DTYPE_CODE[x.dtype], m, k,
                                             x.stride(0), _native.stream_ptr(x.device))
    _native.check(rc, "mindiesd_mx_quant")
    return q.view(torch.float8_e4m3fn), e.view(torch.float8_e8m0fnu)


def _as_u8(t, what, shape):
    if t.dtype not in (torch.uint8, torch.float8_e4m3fn, torch.float8_e8m0fnu) or not t.is_cuda:
        raise ParametersInvalid(f"{what} must be a 1-byte (fp8 / e8m0 / uint8) GPU tensor, but got {t.dtype}.")
    t = t.reshape(shape)
    return t.contiguous().view(torch.uint8)


def _as_bias(bias, device, nw):
    bias = bias.to(device=device, dtype=torch.float32).contiguous()
    if bias.numel() != nw:
        raise ParametersInvalid("bias must have one entry per weight row.")
    return bias


def _check_matmul(same_k, k, w_q, out_dtype, swiglu):
    """What the GEMM asks of its shapes and output type; returns the number of weight rows."""
    if not same_k:
        raise ParametersInvalid("mxfp8_matmul needs x_q [M, K] and w_q [N, K].")
    nw = w_q.shape[0]
    if k % 128 != 0:
        raise ParametersInvalid(f"mxfp8_matmul needs K % 128 == 0, but got K = {k}.")
    if nw % (16 if swiglu else 8) != 0:
        raise ParametersInvalid(f"mxfp8_matmul needs the weight row count to be a multiple of "
                                f"{16 if swiglu else 8}, but got {nw}.")
    if out_dtype not in _native.DTYPE_CODE:
        raise ParametersInvalid(f"out_dtype must be bf16 or fp16, but got {out_dtype}.")
    return nw


def mxfp8_matmul(x_q, x_scale, w_q, w_scale, bias=None, out_dtype=torch.bfloat16, swiglu=False):
    """``act(x @ w.T + bias)`` on MX-quantised operands: x_q [M, K] E4M3, x_scale [M, K/32] E8M0,
    w_q [Nw, K], w_scale [Nw, K/32] (also accepted as [Nw, K/64, 2], the reference's storage shape).
    ``swiglu=True``: w = [gate rows | up rows], result [M, Nw/2] = silu(gate) * up; else [M, Nw]."""
    same_k = x_q.dim() == 2 and w_q.dim() == 2 and x_q.shape[1] == w_q.shape[1]
    nw = _check_matmul(same_k, x_q.shape[-1], w_q, out_dtype, swiglu)
    m, k = x_q.shape
    xq, wq = _as_u8(x_q, "x_q", (m, k)), _as_u8(w_q, "w_q", (nw, k))
    xs, ws = _as_u8(x_scale, "x_scale", (m, k // 32)), _as_u8(w_scale, "w_scale", (nw, k // 32))
    if bias is not None:
        bias = _as_bias(bias, xq.device, nw)
    out = torch.empty((m, nw // 2 if swiglu else nw), dtype=out_dtype, device=xq.device)
    with _native.on_device(xq.device):
        rc = _native.lib().mindiesd_mxfp8_gemm(xq.data_ptr(), xs.data_ptr(), wq.data_ptr(), ws.data_ptr(),
                                               bias.data_ptr() if bias is not None else None, out.data_ptr(),
                                               _native.DTYPE_CODE[out_dtype], m, k, nw, int(bool(swiglu)),
                                               _native.stream_ptr(xq.device))
    _native.check(rc, "mindiesd_mxfp8_gemm")
    return out


_CODE_DTYPES = (torch.uint8, torch.float8_e4m3fn, torch.float8_e8m0fnu)


def mxfp8_linear(x, w_q, w_scale, bias=None, out_dtype=torch.bfloat16, swiglu=False):
    """``mxfp8_matmul(*mx_quantize(x), w_q, w_scale, bias, out_dtype, swiglu)`` as one native call, for x [..., K] bf16/fp16
    with any leading dimensions; result [..., Nw] or [..., Nw/2].  A layer on a few hundred tokens is
    over sooner than the host has made the two calls with their tensors, views and checks (28 us a layer, with this one call
    17 us, of which 2 are the layer's views), so the codes and scales share one allocation, and only what is not contiguous is viewed or copied."""
    if not isinstance(x, torch.Tensor) or x.dim() < 1 or not x.is_cuda or x.dtype not in _native.DTYPE_CODE:
        raise ParametersInvalid("mx_quantize needs a 2-D bf16/fp16 GPU tensor.")
    *lead, k = x.shape
    if k % 32 != 0:
        raise ParametersInvalid(f"mx_quantize needs K % 32 == 0, but got K = {k}.")
    nw = _check_matmul(w_q.dim() == 2 and w_q.shape[1] == k, k, w_q, out_dtype, swiglu)
    m, x_ss, x_ptr = x.numel() // max(k, 1), k, x.data_ptr()
    if x_ptr % 16 != 0 or not x.is_contiguous():
        x = x.reshape(m, k)
        x_ss, x_s1 = x.stride()
        if x_s1 != 1 or x_ss % 8 != 0 or x.data_ptr() % 16 != 0:
            x, x_ss = x.contiguous(), k
        x_ptr = x.data_ptr()
    for t, cols in ((w_q, k), (w_scale, k // 32)):
        if t.dtype not in _CODE_DTYPES or not t.is_cuda or t.numel() != nw * cols or not t.is_contiguous():
            w_q, w_scale = _as_u8(w_q, "w_q", (nw, k)), _as_u8(w_scale, "w_scale", (nw, k // 32))
            break
    device = x.device
    if bias is not None:
        bias = _as_bias(bias, device, nw)
    out = torch.empty((*lead, nw // 2 if swiglu else nw), dtype=out_dtype, device=device)
    codes = torch.empty(m * (k + k // 32), dtype=torch.uint8, device=device)
    code_ptr = codes.data_ptr()
    with _native.on_device(device):
        rc = _native.lib().mindiesd_mxfp8_linear(
            x_ptr, _native.DTYPE_CODE[x.dtype], x_ss, code_ptr, code_ptr + m * k, w_q.data_ptr(), w_scale.data_ptr(),
            None if bias is None else bias.data_ptr(), out.data_ptr(), _native.DTYPE_CODE[out_dtype], m, k, nw,
            1 if swiglu else 0, _native.stream_ptr(device))
    _native.check(rc, "mindiesd_mxfp8_linear")
    return out


def mxfp8_gemm_swiglu(x, w_q, w_scale, bias=None, out_dtype=None):
    """DiT FFN up-projection: quantise the activations ``x`` [..., K] on the fly, multiply with the
    MX-quantised weight [gate | up] ([2F, K]) and return ``silu(gate) * up`` [..., F]."""
    return mxfp8_linear(x, w_q, w_scale, bias, out_dtype or x.dtype, swiglu=True)
