"""Callers of the C ABI for torch-owned device buffers: the library's Python entry points.

torch supplies device memory and the current HIP stream; every computation is a
call into libcaifx.so.  The calls of a training or serving step go through native code
(csrc/torch_calls.cpp: checks, result and workspace allocation, stream), the rest through
ctypes.  Function names follow the reference's CAIF_Ops entry points
(src/caif_ops.cpp:504-680); argument meaning is the same.
"""
import torch

from . import capi
from .capi import F32, F16, BF16, W_INT8, W_INT4_GROUP, W_F32, W_F16, W_BF16

TORCH_DTYPE = {F32: torch.float32, F16: torch.float16, BF16: torch.bfloat16}
CODE_OF = {v: k for k, v in TORCH_DTYPE.items()}


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _ptr(t):
    return 0 if t is None else t.data_ptr()


def _need_cuda(*ts):
    for t in ts:
        if t is not None and not t.is_cuda:
            # CAIF_Ops quantise entry points throw for Host_e tensors (src/caif_ops.cpp:514-517)
            raise RuntimeError("host backend not supported")
        if t is not None and not t.is_contiguous():
            raise RuntimeError("tensor must be contiguous")


_native = None


def _calls():
    global _native
    if _native is None:
        _native = capi.calls()
    return _native


def _done(r, name):
    """The native call's result; a status other than CAIFX_OK comes back as an int."""
    if r.__class__ is int:
        capi.check(r, name)
    return r


# ------------------------------------------------------------------ CAIF_Ops::Quantize* / Dequantize*
def quantize_int8(x, per_channel):
    """CAIF_Ops::QuantizeInt8 (src/caif_ops_device.cpp:1517-1573).  Returns (codes, scales)."""
    return _done((_native or _calls()).quantize_int8(x, per_channel),
                 "caifx_quantize_int8_per_channel" if per_channel else "caifx_quantize_int8_per_tensor")


def dequantize_int8(q, scales, per_channel):
    """CAIF_Ops::DequantizeInt8 (src/caif_ops_device.cpp:1584-1640)."""
    _need_cuda(q, scales)
    out = torch.empty(q.shape, dtype=torch.float32, device=q.device)
    if not per_channel:
        if scales.numel() != 1:
            raise RuntimeError("DequantizeInt8 PerTensor: scales must have 1 element")
        capi.call("caifx_dequantize_int8_per_tensor", _ptr(q), _ptr(out), _ptr(scales), q.numel(), _stream())
        return out
    if q.dim() != 2:
        raise RuntimeError("DequantizeInt8 PerChannel: input must be 2D")
    rows, cols = q.shape
    if scales.numel() != cols:
        raise RuntimeError("DequantizeInt8 PerChannel: scales length must equal cols")
    capi.call("caifx_dequantize_int8_per_channel", _ptr(q), _ptr(out), _ptr(scales), rows, cols, _stream())
    return out


def quantize_int4_per_group(x, group_size):
    """CAIF_Ops::QuantizeInt4PerGroup (src/caif_ops_device.cpp:1651-1687).  Returns (packed, fp16 scales)."""
    return _done((_native or _calls()).quantize_int4(x, group_size), "caifx_quantize_to_int4")


def dequantize_int4_per_group(packed, scales, n, group_size):
    """CAIF_Ops::DequantizeInt4PerGroup (src/caif_ops_device.cpp:1698-1734)."""
    _need_cuda(packed, scales)
    if group_size == 0:
        raise RuntimeError("DequantizeInt4PerGroup: group_size must be > 0")
    if scales.numel() != (n + group_size - 1) // group_size:
        raise RuntimeError("DequantizeInt4PerGroup: scales length must equal num_groups")
    out = torch.empty(n, dtype=torch.float32, device=packed.device)
    capi.call("caifx_dequantize_int4", _ptr(packed), _ptr(scales), _ptr(out), n, group_size, _stream())
    return out


_CASTS = {
    (torch.float32, torch.float16): "caifx_convert_fp32_to_fp16",
    (torch.float16, torch.float32): "caifx_convert_fp16_to_fp32",
    (torch.float32, torch.bfloat16): "caifx_convert_fp32_to_bf16",
    (torch.bfloat16, torch.float32): "caifx_convert_bf16_to_fp32",
    (torch.float32, torch.int8): "caifx_convert_fp32_to_int8",
    (torch.int8, torch.float32): "caifx_convert_int8_to_fp32",
}


def convert(x, dtype):
    """The cast kernels behind CAIF_DeviceTensor::To (src/caif_device_tensor.cpp:604-706)."""
    _need_cuda(x)
    out = torch.empty(x.shape, dtype=dtype, device=x.device)
    capi.call(_CASTS[(x.dtype, dtype)], _ptr(x), _ptr(out), x.numel(), _stream())
    return out


# ------------------------------------------------------------------ frozen linear
class FrozenWeight:
    """Device storage of one CAIF_DeviceFrozenLinear: codes, scales and the scale scheme."""

    def __init__(self, wq, w_kind, scales, N, K, scale_period=1, group_size=128):
        self.wq, self.w_kind, self.scales = wq, w_kind, scales
        self.N, self.K, self.scale_period, self.group_size = N, K, scale_period, group_size


def qlinear_forward(x, fw, compute_dtype, y_dtype=F32, out=None, workspace=None, addend=None):
    """caifx_qlinear_forward on x [..., K]; returns y [M, N].  With `addend` [M, N] of y_dtype:
    caifx_qlinear_forward_add, y = T(float(T(x W^T)) + float(addend))."""
    return _done((_native or _calls()).qlinear(0, x, fw, compute_dtype, y_dtype, out, workspace, addend),
                 "caifx_qlinear_forward")


def probe_mfma_bf16(a_values, b_values, iters):
    """caifx_probe_mfma_bf16: launches the matrix-pipe-only loop on the first 16384 bf16 values of each tensor;
    returns the floating-point operations of the launch (time it with events around the call)."""
    import ctypes
    _need_cuda(a_values)
    a = a_values.reshape(-1)[:16384].to(torch.bfloat16).contiguous()
    b = b_values.reshape(-1)[:16384].to(torch.bfloat16).contiguous()
    assert a.numel() == 16384 and b.numel() == 16384
    sink = torch.empty(512, dtype=torch.float32, device=a.device)
    flops = ctypes.c_int64(0)
    capi.call("caifx_probe_mfma_bf16", _ptr(a), _ptr(b), int(iters), _ptr(sink), ctypes.byref(flops), _stream())
    return flops.value, (a, b, sink)


def qlinear_backward_input(dy, fw, compute_dtype, dx_dtype=F32, out=None, workspace=None, addend=None):
    """caifx_qlinear_backward_input on dy [..., N]; returns dx [M, K] (plus `addend` [M, K], see qlinear_forward)."""
    return _done((_native or _calls()).qlinear(1, dy, fw, compute_dtype, dx_dtype, out, workspace, addend),
                 "caifx_qlinear_backward_input")


class GroupedFrozenWeights:
    """E frozen linears of one shape (one per expert), addressed through device pointer arrays."""

    def __init__(self, weights):
        w0 = weights[0]
        self.weights = weights
        self.N, self.K, self.w_kind = w0.N, w0.K, w0.w_kind
        self.scale_period, self.group_size = w0.scale_period, w0.group_size
        dev = w0.wq.device
        self.wq_ptrs = torch.tensor([w.wq.data_ptr() for w in weights], dtype=torch.int64, device=dev)
        self.scales_ptrs = None
        if w0.scales is not None:
            self.scales_ptrs = torch.tensor([w.scales.data_ptr() for w in weights], dtype=torch.int64, device=dev)


def _check_grouped(x, in_dim, rows, offsets, E, results, out_dim, out_dtype):
    """The C ABI sees raw pointers: sizes and dtypes are checked here, before anything is launched."""
    if x.numel() != rows * in_dim:
        raise ValueError(f"input has {x.numel()} elements, not a multiple of the reduction length {in_dim}")
    if offsets.dtype != torch.int32 or offsets.numel() != E + 1:
        raise ValueError(f"offsets must be int32 [{E + 1}]")
    for t in results:
        _need_cuda(t)
        if t.dtype != out_dtype or t.numel() != rows * out_dim:
            raise ValueError(f"result / gating tensors must be {out_dtype} with {rows} x {out_dim} elements")


def qlinear_grouped_forward(x, offsets, gw, compute_dtype, y_dtype=F32, out=None, workspace=None):
    return _done((_native or _calls()).grouped(0, x, offsets, gw, compute_dtype, y_dtype, out, workspace, None),
                 "caifx_qlinear_grouped_forward")


def qlinear_grouped_backward_input(dy, offsets, gw, compute_dtype, dx_dtype=F32, out=None, workspace=None,
                                   addend=None):
    return _done((_native or _calls()).grouped(1, dy, offsets, gw, compute_dtype, dx_dtype, out, workspace, addend),
                 "caifx_qlinear_grouped_backward_input")


def qlinear_grouped_forward_swiglu(x, offsets, gw_up, gate, compute_dtype, out=None):
    """Up projection with the gating in its store: returns (up, hidden), both of gate's dtype and shape."""
    _need_cuda(x, offsets, gate)
    rows = x.numel() // gw_up.K
    up, hidden = out if out is not None else (torch.zeros_like(gate), torch.zeros_like(gate))
    _check_grouped(x, gw_up.K, rows, offsets, len(gw_up.weights), (gate, up, hidden), gw_up.N, gate.dtype)
    capi.call("caifx_qlinear_grouped_forward_swiglu", len(gw_up.weights), _ptr(offsets), rows, gw_up.N, gw_up.K, _ptr(x),
              CODE_OF[x.dtype], compute_dtype, _ptr(gw_up.wq_ptrs), gw_up.w_kind, _ptr(gw_up.scales_ptrs),
              gw_up.scale_period, gw_up.group_size, _ptr(gate), _ptr(up), _ptr(hidden), CODE_OF[gate.dtype], _stream())
    return up, hidden


def qlinear_grouped_backward_input_swiglu(dy, offsets, gw_down, gate, up, compute_dtype, out=None):
    """Input gradient of the down projection with the gating's backward in its store: returns (grad_gate, grad_up)."""
    _need_cuda(dy, offsets, gate, up)
    rows = dy.numel() // gw_down.N
    grad_gate, grad_up = out if out is not None else (torch.zeros_like(gate), torch.zeros_like(gate))
    _check_grouped(dy, gw_down.N, rows, offsets, len(gw_down.weights), (gate, up, grad_gate, grad_up), gw_down.K, gate.dtype)
    capi.call("caifx_qlinear_grouped_backward_input_swiglu", len(gw_down.weights), _ptr(offsets), rows, gw_down.N, gw_down.K,
              _ptr(dy), CODE_OF[dy.dtype], compute_dtype, _ptr(gw_down.wq_ptrs), gw_down.w_kind, _ptr(gw_down.scales_ptrs),
              gw_down.scale_period, gw_down.group_size, _ptr(gate), _ptr(up), _ptr(grad_gate), _ptr(grad_up),
              CODE_OF[gate.dtype], _stream())
    return grad_gate, grad_up


# ------------------------------------------------------------------ element-wise
def _ew(op, name, a, b=None, out=None):
    return _done((_native or _calls()).elementwise(op, a, b, out), name)


def silu(x):
    return _ew(0, "caifx_silu", x)


def silu_backward(x, grad_out):
    return _ew(1, "caifx_silu_backward", x, grad_out)


def multiply(a, b):
    return _ew(2, "caifx_multiply", a, b)


def add(a, b):
    return _ew(3, "caifx_add", a, b)


def silu_multiply(gate, up, out=None):
    return _ew(4, "caifx_silu_multiply", gate, up, out)


def swiglu_backward(gate, up, grad_hidden, out_gate=None, out_up=None):
    """(grad_gate, grad_up) of hidden = silu(gate) * up in one pass, bit-identical to
    multiply(grad_hidden, silu(gate)) and silu_backward(gate, multiply(grad_hidden, up))."""
    return _done((_native or _calls()).swiglu_backward(gate, up, grad_hidden, out_gate, out_up), "caifx_swiglu_backward")


# ------------------------------------------------------------------ MoE token routing
def moe_build_dispatch_map(expert_indices, num_experts, capacity_per_expert=0):
    """(dispatch_map [T, top_k] int32, expert_offsets [E+1] int32), built on the device without a host
    round trip; expert_offsets[-1] is the number of assigned rows."""
    return _done((_native or _calls()).moe_build_dispatch_map(expert_indices, num_experts, capacity_per_expert),
                 "caifx_moe_build_dispatch_map")


def moe_dispatch(x, expert_indices, dispatch_map, expert_offsets, total_rows, out=None):
    return _done((_native or _calls()).moe_dispatch(x, expert_indices, dispatch_map, expert_offsets, total_rows, out),
                 "caifx_moe_dispatch")


def moe_combine(expert_buffer, expert_indices, expert_weights, dispatch_map, expert_offsets, out=None):
    return _done((_native or _calls()).moe_combine(expert_buffer, expert_indices, expert_weights, dispatch_map,
                                                   expert_offsets, out), "caifx_moe_combine")


def moe_combine_backward_grad_expert(grad_output, expert_indices, expert_weights, dispatch_map, expert_offsets,
                                     total_rows, out=None):
    return _done((_native or _calls()).moe_combine_backward_grad_expert(
        grad_output, expert_indices, expert_weights, dispatch_map, expert_offsets, total_rows, out),
        "caifx_moe_combine_backward_grad_expert")


def moe_dispatch_backward(grad_expert_buffer, expert_indices, dispatch_map, expert_offsets, out=None):
    return _done((_native or _calls()).moe_dispatch_backward(grad_expert_buffer, expert_indices, dispatch_map,
                                                             expert_offsets, out), "caifx_moe_dispatch_backward")


def moe_combine_backward_grad_weights(grad_output, expert_buffer, expert_indices, dispatch_map, expert_offsets):
    return _done((_native or _calls()).moe_combine_backward_grad_weights(
        grad_output, expert_buffer, expert_indices, dispatch_map, expert_offsets),
        "caifx_moe_combine_backward_grad_weights")
