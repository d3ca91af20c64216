"""torch.library custom ops over the C ABI of libhynomas_fp8.so.

Each op is opaque to torch.compile (a fake implementation gives shapes only),
launches on the current stream of the input's device, and raises on CPU
tensors: the FP8 path has no CPU fallback. The custom-op + register_fake
pattern is the one the reference uses for its FP8 GEMM
(hymm/models/vae/pixelumm_decoder/cutlass_fp8.py:47-57).

Plain eager inference calls an op's implementation without the dispatcher
(``eager_op``): the trip through torch's custom-op layers costs more host time
than a launch, and the small calls are bound by it.
"""
from __future__ import annotations

import contextlib
import ctypes
import functools
import math
from typing import Optional

import torch

from . import _lib as L

FP8 = torch.float8_e4m3fn


def _gpu(*tensors) -> None:
    for t in tensors:
        if t is not None and not t.is_cuda:
            raise RuntimeError("hy-nomas_amd FP8 kernels need GPU tensors (there is no CPU path)")


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _stream(t: torch.Tensor) -> int:
    if _raw_stream is None:  # a torch without the short form
        return torch.cuda.current_stream(t.device).cuda_stream
    return _raw_stream(t.device.index)


def _on(device: torch.device):
    """``torch.cuda.device(device)``, or nothing where it is current already."""
    return contextlib.nullcontext() if device.index == torch.cuda.current_device() else torch.cuda.device(device)


_TENSOR = (torch.Tensor, torch.nn.Parameter)
_KINDS = {"Tensor": _TENSOR, "Optional[Tensor]": (*_TENSOR, type(None)), "int": (int,), "float": (float, int),
          "Optional[float]": (float, int, type(None))}


try:
    _OBSERVERS = (torch._C._get_tracing_state, torch._C._len_torch_function_stack,
                  torch._C._len_torch_dispatch_stack, torch._C._functorch.peek_interpreter_stack,
                  torch.autograd._profiler_enabled)
    _forward_ad = torch.autograd.forward_ad
    _forward_ad._current_level
except AttributeError:  # a torch without one of these private names: no direct calls
    _OBSERVERS = None


def _observed() -> bool:
    """Whether something other than the kernel would see a call of an op: a
    trace, a torch_function or torch_dispatch mode, a functorch transform,
    forward-mode AD or the autograd profiler."""
    if _OBSERVERS is None:
        return True
    trace, function_modes, dispatch_modes, transform, profiled = _OBSERVERS
    return bool(trace() is not None or function_modes() or dispatch_modes() or transform() is not None
                or _forward_ad._current_level >= 0 or profiled())


def eager_op(op_name: str, mutates_args=()):
    """``torch.library.custom_op`` whose plain eager calls skip the dispatcher.

    A call goes straight to the implementation when every argument is of
    exactly its schema's type (plain tensors and numbers, no subclass), every tensor
    is on a GPU with its values in memory as they are (meta tensors have a fake kernel;
    the dispatcher resolves negated views), no tensor would be recorded by autograd and
    nothing observes the call (_observed, or torch.compile); every other call, and every
    call of an op that a program has registered a kernel or rule on, goes through the
    registered op. Mutated tensors get the version bump that the op gives
    them. Host time of an FP8
    linear 45 -> 24 us, of a K/V cache write 41 -> 31 us."""
    def wrap(fn):
        op = torch.library.custom_op(op_name, fn, mutates_args=mutates_args)
        args = op._opoverload._schema.arguments
        names = [a.name for a in args]
        kinds = [_KINDS[str(a.type)] for a in args]
        by_name = dict(zip(names, kinds))
        required = sum(not a.has_default_value() for a in args)
        mutated = [(i, n) for i, n in enumerate(names) if n in mutates_args]

        def plain(pos, kw) -> bool:
            if len(pos) > len(kinds) or (len(pos) < required and any(n not in kw for n in names[len(pos):required])):
                return False
            grad = torch.is_grad_enabled()
            for v, kind in zip(pos, kinds):
                t = type(v)
                if t not in kind or (t in _TENSOR and (not v.is_cuda or v.is_neg()
                                                       or (grad and v.requires_grad))):
                    return False
            for n, v in kw.items():
                t = type(v)
                if t not in by_name.get(n, ()) or (t in _TENSOR and (not v.is_cuda or v.is_neg()
                                                                     or (grad and v.requires_grad))):
                    return False
            return not _observed()

        registered = []  # kernels and rules of the caller's own: calls then meet the op

        @functools.wraps(fn)
        def call(*pos, **kw):
            if torch.compiler.is_compiling() or registered or not plain(pos, kw):
                return op(*pos, **kw)
            out = fn(*pos, **kw)
            if mutated:
                seen = [pos[i] if i < len(pos) else kw.get(n) for i, n in mutated]
                torch.autograd.graph.increment_version([t for t in seen if t is not None and not t.is_inference()])
            return out

        def rule(name):
            def register(*pos, **kw):
                registered.append(name)
                return getattr(op, name)(*pos, **kw)
            return register

        for name in dir(op):  # custom_op's own registration methods
            if name.startswith("register_") or name == "set_kernel_enabled":
                setattr(call, name, rule(name))
        call.register_fake = op.register_fake
        call.impl = fn
        return call
    return wrap


def _bytes(t: torch.Tensor) -> torch.Tensor:
    return t.view(torch.uint8) if t.dtype in (FP8, torch.int8) else t


# --------------------------------------------------------------------------
# quantizers

@eager_op("hy_nomas_amd::quantize_rows_fp8", mutates_args=())
def quantize_rows_fp8(x: torch.Tensor, scale_mode: int = L.HN_SCALE_CLAMP,
                      amax_floor: float = 1e-4) -> tuple[torch.Tensor, torch.Tensor]:
    """Per-row e4m3 codes and fp32 scales of a bf16 [..., C] tensor."""
    _gpu(x)
    if x.dtype != torch.bfloat16:
        raise TypeError("quantize_rows_fp8 expects bf16 input")
    q, s = _quantize_matrix(x if x.ndim == 2 else x.reshape(-1, x.shape[-1]), scale_mode, amax_floor)
    return (q, s) if x.ndim == 2 else (q.view(x.shape), s.view(x.shape[:-1]))


def _quantize_matrix(x, scale_mode: int, amax_floor: float):
    if x.stride(-1) != 1:
        x = x.contiguous()
    rows, cols = x.shape
    device = x.device
    q = torch.empty((rows, cols), dtype=FP8, device=device)
    s = torch.empty((rows,), dtype=torch.float32, device=device)
    with _on(device):
        L.check(L.load().hn_quantize_rows_fp8(
            x.data_ptr(), rows, cols, x.stride(0), scale_mode, amax_floor,
            q.data_ptr(), s.data_ptr(), _stream(x)), "hn_quantize_rows_fp8")
    return q, s


@quantize_rows_fp8.register_fake
def _(x, scale_mode=L.HN_SCALE_CLAMP, amax_floor=1e-4):
    return x.new_empty(x.shape, dtype=FP8), x.new_empty(x.shape[:-1], dtype=torch.float32)


def ln_modulate_quantize_fp8(x, shift, scale, eps: float = 1e-6, amax_floor: float = 1e-4, *,
                             residual=None):
    """LayerNorm (no affine) + adaLN modulate + per-token e4m3 quantization of a
    bf16 [B, L, C] tensor in one pass: the codes and scales of
    quantize_rows_fp8(modulate(layer_norm(x), shift, scale)) with shift and
    scale bf16 [B, C] (nomas_compile_prepost.py:14-15,40-43,81-84). Returns
    codes [B*L, C] and fp32 scales [B*L].

    With ``residual`` = (y [B, L, C], gate [B, C]) x is first replaced by
    gated_residual(x, y, gate) in the same pass; returns that x too, before the
    codes and scales."""
    if residual is None:
        return _ln_modulate_quantize_op(x, shift, scale, eps, amax_floor)
    return _residual_ln_modulate_quantize_op(x, *residual, shift, scale, eps, amax_floor)


@eager_op("hy_nomas_amd::ln_modulate_quantize_fp8", mutates_args=())
def _ln_modulate_quantize_op(x: torch.Tensor, shift: torch.Tensor, scale: torch.Tensor,
                             eps: float = 1e-6,
                             amax_floor: float = 1e-4) -> tuple[torch.Tensor, torch.Tensor]:
    _gpu(x, shift, scale)
    if x.dtype != torch.bfloat16 or shift.dtype != torch.bfloat16 or scale.dtype != torch.bfloat16:
        raise TypeError("ln_modulate_quantize_fp8 expects bf16 tensors")
    if x.ndim != 3 or shift.shape != (x.shape[0], x.shape[2]) or scale.shape != shift.shape:
        raise ValueError("ln_modulate_quantize_fp8: x [B, L, C] with shift and scale [B, C]")
    x = x.contiguous()
    shift = shift.contiguous()
    scale = scale.contiguous()
    B, Lt, C = x.shape
    q = torch.empty((B * Lt, C), dtype=FP8, device=x.device)
    s = torch.empty((B * Lt,), dtype=torch.float32, device=x.device)
    with _on(x.device):
        L.check(L.load().hn_ln_mod_quantize_fp8(
            x.data_ptr(), B * Lt, C, max(Lt, 1), shift.data_ptr(), scale.data_ptr(), C, eps,
            amax_floor, q.data_ptr(), s.data_ptr(), _stream(x)), "hn_ln_mod_quantize_fp8")
    return q, s


@_ln_modulate_quantize_op.register_fake
def _(x, shift, scale, eps=1e-6, amax_floor=1e-4):
    n = x.shape[0] * x.shape[1]
    return x.new_empty((n, x.shape[2]), dtype=FP8), x.new_empty((n,), dtype=torch.float32)


def _rows16(t: torch.Tensor) -> torch.Tensor:
    """t contiguous and 16-byte aligned, as the kernels load it (a copy where it is not)."""
    t = t.contiguous()
    return t.clone() if t.data_ptr() % 16 else t


def _residual_args(x, y, gate, what: str):
    """Checks of x and y bf16 [B, L, C] and gate bf16 [B, C]; x, y and gate for the kernel."""
    _gpu(x, y, gate)
    if x.dtype != torch.bfloat16 or y.dtype != torch.bfloat16 or gate.dtype != torch.bfloat16:
        raise TypeError(f"{what} expects bf16 tensors")
    if x.ndim != 3 or y.shape != x.shape or gate.shape != (x.shape[0], x.shape[2]):
        raise ValueError(f"{what}: x and y [B, L, C] with gate [B, C]")
    return _rows16(x), _rows16(y), _rows16(gate)


@eager_op("hy_nomas_amd::gated_residual", mutates_args=())
def gated_residual(x: torch.Tensor, y: torch.Tensor, gate: torch.Tensor) -> torch.Tensor:
    """x + y * gate for bf16 [B, L, C] x and y and a [B, C] gate, with the bf16
    roundings of the two tensor ops (nomas_compile_prepost.py:75-88)."""
    x, y, gate = _residual_args(x, y, gate, "gated_residual")
    B, Lt, C = x.shape
    out = torch.empty_like(x)
    with _on(x.device):
        L.check(L.load().hn_gated_residual(x.data_ptr(), y.data_ptr(), gate.data_ptr(), C, out.data_ptr(),
                                           B * Lt, C, max(Lt, 1), _stream(x)), "hn_gated_residual")
    return out


@gated_residual.register_fake
def _(x, y, gate):
    return x.new_empty(x.shape)


@eager_op("hy_nomas_amd::residual_ln_modulate_quantize_fp8", mutates_args=())
def _residual_ln_modulate_quantize_op(
        x: torch.Tensor, y: torch.Tensor, gate: torch.Tensor, shift: torch.Tensor, scale: torch.Tensor,
        eps: float = 1e-6, amax_floor: float = 1e-4) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    x, y, gate = _residual_args(x, y, gate, "ln_modulate_quantize_fp8")
    _gpu(shift, scale)
    if shift.dtype != torch.bfloat16 or scale.dtype != torch.bfloat16:
        raise TypeError("ln_modulate_quantize_fp8 expects bf16 tensors")
    if shift.shape != gate.shape or scale.shape != gate.shape:
        raise ValueError("ln_modulate_quantize_fp8: gate, shift and scale [B, C]")
    shift, scale = shift.contiguous(), scale.contiguous()
    B, Lt, C = x.shape
    out = torch.empty_like(x)
    q = torch.empty((B * Lt, C), dtype=FP8, device=x.device)
    s = torch.empty((B * Lt,), dtype=torch.float32, device=x.device)
    with _on(x.device):
        L.check(L.load().hn_residual_ln_mod_quantize_fp8(
            x.data_ptr(), y.data_ptr(), gate.data_ptr(), C, out.data_ptr(), B * Lt, C, max(Lt, 1),
            shift.data_ptr(), scale.data_ptr(), C, eps, amax_floor, q.data_ptr(), s.data_ptr(), _stream(x)),
            "hn_residual_ln_mod_quantize_fp8")
    return out, q, s


@_residual_ln_modulate_quantize_op.register_fake
def _(x, y, gate, shift, scale, eps=1e-6, amax_floor=1e-4):
    n = x.shape[0] * x.shape[1]
    return (x.new_empty(x.shape), x.new_empty((n, x.shape[2]), dtype=FP8),
            x.new_empty((n,), dtype=torch.float32))


@eager_op("hy_nomas_amd::quantize_blockwise_fp8", mutates_args=())
def quantize_blockwise_fp8(x: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    """128x128 blockwise e4m3 codes [M,K] and scales [ceil(M/128), K/128]."""
    _gpu(x)
    if x.dtype != torch.bfloat16 or x.ndim != 2:
        raise TypeError("quantize_blockwise_fp8 expects a bf16 [M, K] matrix")
    x = x.contiguous()
    m, k = x.shape
    q = torch.empty((m, k), dtype=FP8, device=x.device)
    s = torch.empty(((m + 127) // 128, k // 128), dtype=torch.float32, device=x.device)
    with _on(x.device):
        L.check(L.load().hn_quantize_blockwise_fp8(x.data_ptr(), m, k, q.data_ptr(), s.data_ptr(),
                                                   _stream(x)), "hn_quantize_blockwise_fp8")
    return q, s


@quantize_blockwise_fp8.register_fake
def _(x):
    m, k = x.shape
    return (x.new_empty((m, k), dtype=FP8),
            x.new_empty(((m + 127) // 128, k // 128), dtype=torch.float32))


# --------------------------------------------------------------------------
# GEMMs

@eager_op("hy_nomas_amd::gemm_fp8_rowcol", mutates_args=())
def gemm_fp8_rowcol(a: torch.Tensor, b: torch.Tensor, sa: torch.Tensor, sb: torch.Tensor,
                    bias: Optional[torch.Tensor] = None, act: int = L.HN_ACT_NONE) -> torch.Tensor:
    """act(a b^T * sa[m] * sb[n] + bias[n]) in bf16; a e4m3 [M,K], b e4m3 [N,K]."""
    _gpu(a, b, sa, sb, bias)
    if a.dtype != FP8 or b.dtype != FP8:
        raise TypeError("gemm_fp8_rowcol expects e4m3 operands")
    if sa.dtype != torch.float32 or sb.dtype != torch.float32:
        raise TypeError("gemm_fp8_rowcol expects fp32 scales")
    if bias is not None and bias.dtype != torch.bfloat16:
        raise TypeError("gemm_fp8_rowcol expects a bf16 bias")
    a = a.contiguous()
    b = b.contiguous()
    m, k = a.shape
    n = b.shape[0]
    if b.shape[1] != k or sa.numel() != m or sb.numel() != n or (bias is not None and bias.numel() != n):
        raise ValueError("gemm_fp8_rowcol shape mismatch")
    out = torch.empty((m, n), dtype=torch.bfloat16, device=a.device)
    with _on(a.device):
        L.check(L.load().hn_gemm_fp8_rowcol(
            a.data_ptr(), b.data_ptr(), sa.contiguous().data_ptr(), sb.contiguous().data_ptr(),
            None if bias is None else bias.contiguous().data_ptr(), out.data_ptr(),
            m, n, k, n, act, _stream(a)), "hn_gemm_fp8_rowcol")
    return out


@gemm_fp8_rowcol.register_fake
def _(a, b, sa, sb, bias=None, act=L.HN_ACT_NONE):
    return a.new_empty((a.shape[0], b.shape[0]), dtype=torch.bfloat16)


@eager_op("hy_nomas_amd::gemm_fp8_blockwise", mutates_args=())
def gemm_fp8_blockwise(a: torch.Tensor, b: torch.Tensor, sa: torch.Tensor,
                       sb: torch.Tensor) -> torch.Tensor:
    """The reference extension's gemm(a, b, sa, sb) with 128x128 block scales."""
    _gpu(a, b, sa, sb)
    for t in (a, b, sa, sb):
        if not t.is_contiguous():
            raise RuntimeError("Expected contiguous tensors on one device")
    if a.dtype != FP8 or b.dtype != FP8:
        raise RuntimeError("Expected E4M3 FP8 inputs")
    if sa.dtype != torch.float32 or sb.dtype != torch.float32:
        raise RuntimeError("Expected FP32 scales")
    if a.dim() != 2 or b.dim() != 2:
        raise RuntimeError("Expected matrices")
    m, k = a.shape
    n = b.shape[0]
    if not (m > 0 and n > 0 and k > 0 and b.shape[1] == k and n % 128 == 0 and k % 128 == 0):
        raise RuntimeError("Invalid GEMM shape")
    if sa.dim() != 2 or tuple(sa.shape) != ((m + 127) // 128, k // 128):
        raise RuntimeError("Invalid activation scales")
    if sb.dim() != 2 or tuple(sb.shape) != (n // 128, k // 128):
        raise RuntimeError("Invalid weight scales")
    out = torch.empty((m, n), dtype=torch.bfloat16, device=a.device)
    with _on(a.device):
        L.check(L.load().hn_gemm_fp8_blockwise(a.data_ptr(), b.data_ptr(), sa.data_ptr(),
                                               sb.data_ptr(), out.data_ptr(), m, n, k,
                                               _stream(a)), "hn_gemm_fp8_blockwise")
    return out


@gemm_fp8_blockwise.register_fake
def _(a, b, sa, sb):
    return a.new_empty((a.shape[0], b.shape[0]), dtype=torch.bfloat16)


@eager_op("hy_nomas_amd::linear_fp8", mutates_args=())
def linear_fp8(x: torch.Tensor, weight: torch.Tensor, weight_scale: torch.Tensor,
               bias: Optional[torch.Tensor] = None, act: int = L.HN_ACT_NONE) -> torch.Tensor:
    """Per-token dynamic e4m3 activation quant + per-channel-scaled FP8 GEMM.
    x bf16 [M, K] -> bf16 [M, N]."""
    if x.ndim != 2:
        qx, sx = quantize_rows_fp8.impl(x, L.HN_SCALE_CLAMP, 1e-4)
    else:
        _gpu(x)
        if x.dtype != torch.bfloat16:
            raise TypeError("quantize_rows_fp8 expects bf16 input")
        qx, sx = _quantize_matrix(x, L.HN_SCALE_CLAMP, 1e-4)
    return gemm_fp8_rowcol.impl(qx, weight, sx, weight_scale, bias, act)


@linear_fp8.register_fake
def _(x, weight, weight_scale, bias=None, act=L.HN_ACT_NONE):
    return x.new_empty((x.shape[0], weight.shape[0]), dtype=torch.bfloat16)


# --------------------------------------------------------------------------
# KV cache

def _kv_fmt(codes: torch.Tensor) -> int:
    if codes.dtype == FP8:
        return L.HN_KV_FP8
    if codes.dtype == torch.int8:
        return L.HN_KV_INT8
    raise TypeError("KV codes must be float8_e4m3fn or int8")


def _check_cache_write(codes: torch.Tensor, scale: torch.Tensor, values: torch.Tensor, start: int,
                       what: str) -> int:
    """Geometry of a KV write, checked on the host before any launch: codes
    [B, cap, H, D], fp32 scales [B, cap, H, 1], values [B, L, H, D] and
    0 <= start, start + L <= cap (int8_kv_cache.py:128-135). Returns cap."""
    if codes.ndim != 4 or values.ndim != 4:
        raise ValueError(f"{what}: cache and values must be [B, L, H, D]")
    B, cap, H, D = codes.shape
    if scale.dtype != torch.float32 or tuple(scale.shape) != (B, cap, H, 1):
        raise ValueError(f"{what}: scale must be fp32 [B, cap, H, 1] matching the codes")
    if values.shape[0] != B or values.shape[2] != H or values.shape[3] != D:
        raise ValueError(f"{what}: values [B, L, H, D] do not match the cache's B, H, D")
    if start < 0 or start + values.shape[1] > cap:
        raise ValueError(f"{what}: tokens [{start}, {start + values.shape[1]}) exceed the cache capacity {cap}")
    return cap


def _status_ptr(status: Optional[torch.Tensor]):
    """Device pointer of a KV-write status word (int32, one element), or None."""
    if status is None:
        return None
    if status.dtype != torch.int32 or status.numel() < 1:
        raise TypeError("status must be an int32 tensor of at least one element")
    return status.data_ptr()


# The three cache writers below mutate an optional status word; torch's
# custom-op wrapper finds mutated arguments by position, so each op is
# registered with every argument required and called through a wrapper that
# passes them all.

def kv_quantize_pair_(k_codes, v_codes, k_scale, v_scale, k, v, start: int, status=None) -> None:
    """Quantize bf16 K/V [B,L,H,D] into the caches at token offset ``start``
    (see _kv_quantize_pair_op)."""
    _kv_quantize_pair_op(k_codes, v_codes, k_scale, v_scale, k, v, start, status)


def kv_quantize_(codes, scale, x, start: int, status=None) -> None:
    """Quantize bf16 values [B,L,H,D] into one cache tensor (see _kv_quantize_op)."""
    _kv_quantize_op(codes, scale, x, start, status)


@eager_op("hy_nomas_amd::kv_quantize_pair_",
                         mutates_args=("k_codes", "v_codes", "k_scale", "v_scale", "status"))
def _kv_quantize_pair_op(k_codes: torch.Tensor, v_codes: torch.Tensor, k_scale: torch.Tensor,
                         v_scale: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                         start: int, status: Optional[torch.Tensor]) -> None:
    """Quantize bf16 K/V [B,L,H,D] into the caches at token offset ``start``.

    With ``status`` (int32 on the device), K and V are validated on the device
    first: status[0] becomes 1 and nothing is written if any value is NaN/Inf,
    else 0. No host synchronisation. None: the caller guarantees finite values."""
    fmt = _kv_fmt(k_codes)
    if v_codes.dtype != k_codes.dtype or k.stride() != v.stride() or k.shape != v.shape:
        raise ValueError("K/V caches and values must share dtype and layout")
    if (k_codes.stride() != v_codes.stride() or k_scale.stride() != v_scale.stride()
            or k_codes.shape != v_codes.shape or k_scale.shape != v_scale.shape):
        raise ValueError("K/V caches must share layout")
    cap = _check_cache_write(k_codes, k_scale, k, start, "kv_quantize_pair_")
    sp = _status_ptr(status)
    _gpu(k_codes, v_codes, k_scale, v_scale, k, v, status)
    B, Lt, H, D = k.shape
    with _on(k.device):
        L.check(L.load().hn_kv_quantize_pair(
            fmt, k.data_ptr(), v.data_ptr(), L.strides(k), B, Lt, H, D,
            k_codes.data_ptr(), v_codes.data_ptr(), L.strides(k_codes),
            k_scale.data_ptr(), v_scale.data_ptr(), L.strides(k_scale), cap, start, sp, _stream(k)),
            "hn_kv_quantize_pair")


@_kv_quantize_pair_op.register_fake
def _(k_codes, v_codes, k_scale, v_scale, k, v, start, status):
    return None


@eager_op("hy_nomas_amd::kv_quantize_", mutates_args=("codes", "scale", "status"))
def _kv_quantize_op(codes: torch.Tensor, scale: torch.Tensor, x: torch.Tensor, start: int,
                    status: Optional[torch.Tensor]) -> None:
    """Quantize bf16 values [B,L,H,D] into one cache tensor at ``start``
    (``status`` as in _kv_quantize_pair_op)."""
    fmt = _kv_fmt(codes)
    cap = _check_cache_write(codes, scale, x, start, "kv_quantize_")
    sp = _status_ptr(status)
    _gpu(codes, scale, x, status)
    B, Lt, H, D = x.shape
    with _on(x.device):
        L.check(L.load().hn_kv_quantize(
            fmt, x.data_ptr(), L.strides(x), B, Lt, H, D, codes.data_ptr(), L.strides(codes),
            scale.data_ptr(), L.strides(scale), cap, start, sp, _stream(x)), "hn_kv_quantize")


@_kv_quantize_op.register_fake
def _(codes, scale, x, start, status):
    return None


@eager_op("hy_nomas_amd::kv_dequantize", mutates_args=())
def kv_dequantize(codes: torch.Tensor, scale: torch.Tensor, valid_len: int) -> torch.Tensor:
    """bf16(code * scale) for tokens [0, valid_len): a new [B, valid_len, H, D] tensor."""
    _gpu(codes, scale)
    fmt = _kv_fmt(codes)
    B, _, H, D = codes.shape
    y = torch.empty((B, valid_len, H, D), dtype=torch.bfloat16, device=codes.device)
    if valid_len == 0:
        return y
    with _on(codes.device):
        L.check(L.load().hn_kv_dequantize(
            fmt, codes.data_ptr(), L.strides(codes), scale.data_ptr(), L.strides(scale),
            B, valid_len, H, D, y.data_ptr(), L.strides(y), _stream(codes)), "hn_kv_dequantize")
    return y


@kv_dequantize.register_fake
def _(codes, scale, valid_len):
    B, _, H, D = codes.shape
    return codes.new_empty((B, valid_len, H, D), dtype=torch.bfloat16)


# --------------------------------------------------------------------------
# fused QK RMSNorm + RoPE (+ KV cache write)

def _qk_launch(q, k, v, q_weight, k_weight, cos, sin, eps, cache, start, status=None):
    if not (q.dtype == k.dtype == v.dtype == torch.bfloat16):
        raise TypeError("qk_norm_rope expects bf16 q, k, v")
    if q.stride() != k.stride() or q.stride() != v.stride() or q.shape != k.shape or q.shape != v.shape:
        raise ValueError("q, k and v must share shape and strides")
    B, Lt, H, D = q.shape
    cos = cos.reshape(-1, D)
    sin = sin.reshape(-1, D)
    if cos.dtype != torch.float32 or sin.dtype != torch.float32 or cos.shape[0] < Lt or cos.stride() != sin.stride():
        raise ValueError("cos/sin must be fp32 [L, D] tables with one layout")
    qw = q_weight.to(torch.bfloat16).contiguous()
    kw = k_weight.to(torch.bfloat16).contiguous()
    if cache:
        k_codes, v_codes, k_scale, v_scale = cache
        fmt = _kv_fmt(k_codes)
        if (v_codes.dtype != k_codes.dtype or k_codes.stride() != v_codes.stride()
                or k_scale.stride() != v_scale.stride() or k_codes.shape != v_codes.shape
                or k_scale.shape != v_scale.shape):
            raise ValueError("K/V caches must share dtype and layout")
        cap = _check_cache_write(k_codes, k_scale, k, start, "qk_norm_rope_kv_")
        cargs = (k_codes.data_ptr(), v_codes.data_ptr(), L.strides(k_codes), k_scale.data_ptr(),
                 v_scale.data_ptr(), L.strides(k_scale), cap, start, _status_ptr(status))
    else:
        fmt = L.HN_KV_FP8
        cargs = (None, None, None, None, None, None, 0, start, None)
    _gpu(q, k, v, q_weight, k_weight, cos, sin, status, *(cache or ()))
    with _on(q.device):
        L.check(L.load().hn_qk_norm_rope_kv(
            fmt, q.data_ptr(), k.data_ptr(), v.data_ptr(), L.strides(q), B, Lt, H, D,
            qw.data_ptr(), kw.data_ptr(), cos.data_ptr(), sin.data_ptr(), cos.stride(0), eps,
            *cargs, _stream(q)), "hn_qk_norm_rope_kv")


@eager_op("hy_nomas_amd::qk_norm_rope_", mutates_args=("q", "k"))
def qk_norm_rope_(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, q_weight: torch.Tensor,
                  k_weight: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, eps: float) -> None:
    """In place: q, k <- RoPE(RMSNorm(q)), RoPE(RMSNorm(k)) for bf16 [B, L, H, 128]
    views sharing strides (v is only checked for layout)."""
    _qk_launch(q, k, v, q_weight, k_weight, cos, sin, eps, None, 0)


@qk_norm_rope_.register_fake
def _(q, k, v, q_weight, k_weight, cos, sin, eps):
    return None


def qk_norm_rope_kv_(q, k, v, q_weight, k_weight, cos, sin, eps: float, k_codes, v_codes, k_scale,
                     v_scale, start: int, status=None) -> None:
    """qk_norm_rope_, and the rotated k and v written into the KV caches at
    token offset ``start`` by the same kernel. With ``status`` (int32 on the
    device) the values to be written are validated on the device first:
    status[0] becomes 1 and the cache is left untouched if any is NaN/Inf."""
    _qk_norm_rope_kv_op(q, k, v, q_weight, k_weight, cos, sin, eps, k_codes, v_codes, k_scale, v_scale,
                        start, status)


@eager_op("hy_nomas_amd::qk_norm_rope_kv_",
                         mutates_args=("q", "k", "k_codes", "v_codes", "k_scale", "v_scale", "status"))
def _qk_norm_rope_kv_op(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, q_weight: torch.Tensor,
                        k_weight: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, eps: float,
                        k_codes: torch.Tensor, v_codes: torch.Tensor, k_scale: torch.Tensor,
                        v_scale: torch.Tensor, start: int, status: Optional[torch.Tensor]) -> None:
    _qk_launch(q, k, v, q_weight, k_weight, cos, sin, eps, (k_codes, v_codes, k_scale, v_scale), start,
               status)


@_qk_norm_rope_kv_op.register_fake
def _(q, k, v, q_weight, k_weight, cos, sin, eps, k_codes, v_codes, k_scale, v_scale, start, status):
    return None


# --------------------------------------------------------------------------
# attention

def join_tokens(qa, qb, ka, kb, va, vb):
    """torch.cat([a, b], dim=1) of the q, k and v of two token streams, bf16 [B, L,
    H, 128] each, in one kernel where it reads their layout. Only metadata that a
    trace holds (types, shapes, strides) is looked at here; addresses are looked
    at in the op, so that a compiled caller keeps one graph."""
    pairs = (qa, qb, ka, kb, va, vb)
    joinable = True
    for t in pairs:
        if not (t.is_cuda and t.device == qa.device and t.dtype == torch.bfloat16 and t.ndim == 4
                and t.shape[3] == 128 and t.stride(3) == 1 and t.stride(0) % 8 == 0 and t.stride(1) % 8 == 0
                and t.stride(2) % 8 == 0):
            joinable = False
    if (joinable and ka.shape == qa.shape and va.shape == qa.shape and kb.shape == qb.shape
            and vb.shape == qb.shape and qa.shape[0] == qb.shape[0] and qa.shape[2] == qb.shape[2]):
        return _join_tokens_op(*pairs)
    return torch.cat([qa, qb], dim=1), torch.cat([ka, kb], dim=1), torch.cat([va, vb], dim=1)


@eager_op("hy_nomas_amd::join_tokens")
def _join_tokens_op(qa: torch.Tensor, qb: torch.Tensor, ka: torch.Tensor, kb: torch.Tensor, va: torch.Tensor,
                    vb: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    if any(t.data_ptr() % 16 for t in (qa, qb, ka, kb, va, vb)):  # the kernel loads 16 bytes
        return torch.cat([qa, qb], dim=1), torch.cat([ka, kb], dim=1), torch.cat([va, vb], dim=1)
    B, La, H, D = qa.shape
    Lb = qb.shape[1]
    out = tuple(torch.empty((B, La + Lb, H, D), dtype=torch.bfloat16, device=qa.device) for _ in range(3))

    def pointers(ts):
        return (ctypes.c_void_p * 3)(*(t.data_ptr() for t in ts))

    def strides(ts):
        return (ctypes.c_int64 * 12)(*(s for t in ts for s in t.stride()))

    a, b = (qa, ka, va), (qb, kb, vb)
    with _on(qa.device):
        L.check(L.load().hn_join_tokens(3, pointers(a), strides(a), pointers(b), strides(b), B, La, Lb, H, D,
                                        pointers(out), _stream(qa)), "hn_join_tokens")
    return out


@_join_tokens_op.register_fake
def _(qa, qb, ka, kb, va, vb):
    shape = (qa.shape[0], qa.shape[1] + qb.shape[1], *qa.shape[2:])
    return qa.new_empty(shape), qa.new_empty(shape), qa.new_empty(shape)


def _valid_bytes(mask: Optional[torch.Tensor], rows: int, cols: int, what: str):
    """A key-validity mask as (uint8 view, batch stride): bool or uint8 [rows or
    1, >= cols] with contiguous tokens; a batch of 1 is read by every row."""
    if mask is None:
        return None, 0
    if mask.dtype not in (torch.bool, torch.uint8) or mask.ndim != 2:
        raise TypeError(f"attn_fp8kv: {what} must be a bool [B, L] mask")
    if mask.shape[0] not in (rows, 1) or mask.shape[1] < cols:
        raise ValueError(f"attn_fp8kv: {what} must cover [{rows}, {cols}]")
    if cols and mask.stride(1) != 1:
        mask = mask.contiguous()
    stride = 0 if mask.shape[0] == 1 else mask.stride(0)
    return mask.view(torch.uint8), stride


@eager_op("hy_nomas_amd::attn_fp8kv", mutates_args=())
def attn_fp8kv(q: torch.Tensor, k_codes: torch.Tensor, v_codes: torch.Tensor,
               k_scale: torch.Tensor, v_scale: torch.Tensor, kv_len: int,
               k_cur: Optional[torch.Tensor] = None, v_cur: Optional[torch.Tensor] = None,
               q_pos0: int = 0, chunk_len: int = 0,
               softmax_scale: Optional[float] = None,
               cache_valid: Optional[torch.Tensor] = None,
               cur_valid: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Chunk attention of q [B,Lq,H,D] over cache tokens [0, kv_len) then the
    optional bf16 tail k_cur/v_cur [B,Lc,H,D]; see hn_attn_fp8kv for the mask.

    The cache may hold B slots or one slot that every query batch reads (the
    read-only CFG broadcast). cache_valid (bool [B or 1, >= kv_len]) and
    cur_valid (bool [B, >= Lc]) exclude invalid keys."""
    if q.dtype != torch.bfloat16:
        raise TypeError("attn_fp8kv expects bf16 queries")
    fmt = _kv_fmt(k_codes)
    if q.ndim != 4:
        raise ValueError("attn_fp8kv: q must be [B, Lq, H, D]")
    B, Lq, H, D = q.shape
    if k_codes.ndim != 4 or k_codes.shape[2:] != (H, D) or k_codes.shape[0] not in (B, 1):
        raise ValueError("attn_fp8kv: cache [B or 1, cap, H, D] does not match q")
    if (v_codes.dtype != k_codes.dtype or v_codes.shape != k_codes.shape
            or v_codes.stride() != k_codes.stride()):
        raise ValueError("attn_fp8kv: K and V codes must share dtype, shape and strides")
    cap = k_codes.shape[1]
    if (k_scale.dtype != torch.float32 or v_scale.dtype != torch.float32
            or tuple(k_scale.shape) != (*k_codes.shape[:3], 1) or v_scale.shape != k_scale.shape
            or v_scale.stride() != k_scale.stride()):
        raise ValueError("attn_fp8kv: K and V scales must be fp32 [B, cap, H, 1] with one layout")
    if not 0 <= kv_len <= cap:
        raise ValueError(f"attn_fp8kv: kv_len {kv_len} outside the cache capacity {cap}")
    if softmax_scale is None:
        softmax_scale = D ** -0.5
    if not (softmax_scale > 0 and math.isfinite(softmax_scale)):
        raise ValueError("attn_fp8kv: softmax_scale must be finite and positive")
    if k_codes.shape[0] != B:  # one history slot read by every query batch
        k_codes, v_codes = k_codes.expand(B, -1, -1, -1), v_codes.expand(B, -1, -1, -1)
        k_scale, v_scale = k_scale.expand(B, -1, -1, -1), v_scale.expand(B, -1, -1, -1)
    cur_len = 0 if k_cur is None else k_cur.shape[1]
    if k_cur is not None and (k_cur.ndim != 4 or k_cur.shape[0] != B or k_cur.shape[2:] != (H, D)):
        raise ValueError("attn_fp8kv: k_cur must be [B, Lc, H, D] matching q")
    if cur_len and (v_cur is None or v_cur.shape != k_cur.shape or k_cur.stride() != v_cur.stride()
                    or k_cur.dtype != torch.bfloat16 or v_cur.dtype != torch.bfloat16):
        raise ValueError("k_cur/v_cur must be matching bf16 tensors")
    kvb, kvs = _valid_bytes(cache_valid if kv_len else None, B, kv_len, "cache_valid")
    uvb, uvs = _valid_bytes(cur_valid if cur_len else None, B, cur_len, "cur_valid")
    _gpu(q, k_codes, v_codes, k_scale, v_scale, k_cur, v_cur, kvb, uvb)
    out = torch.empty((B, Lq, H, D), dtype=torch.bfloat16, device=q.device)
    with _on(q.device):
        lib = L.load()
        ws_bytes = lib.hn_attn_fp8kv_workspace_size(B, Lq, H, D, kv_len, cur_len)
        ws = torch.empty((ws_bytes,), dtype=torch.uint8, device=q.device) if ws_bytes else None
        L.check(lib.hn_attn_fp8kv(
            fmt, q.data_ptr(), L.strides(q), B, Lq, H, D,
            k_codes.data_ptr(), v_codes.data_ptr(), L.strides(k_codes),
            k_scale.data_ptr(), v_scale.data_ptr(), L.strides(k_scale), cap, kv_len,
            L.ptr(kvb), kvs,
            None if not cur_len else k_cur.data_ptr(), None if not cur_len else v_cur.data_ptr(),
            L.strides(k_cur) if cur_len else None, cur_len, L.ptr(uvb), uvs, q_pos0, chunk_len,
            float(softmax_scale), out.data_ptr(), L.strides(out),
            None if ws is None else ws.data_ptr(), ws_bytes, _stream(q)), "hn_attn_fp8kv")
    return out


@attn_fp8kv.register_fake
def _(q, k_codes, v_codes, k_scale, v_scale, kv_len, k_cur=None, v_cur=None, q_pos0=0,
      chunk_len=0, softmax_scale=None, cache_valid=None, cur_valid=None):
    return torch.empty_like(q)
