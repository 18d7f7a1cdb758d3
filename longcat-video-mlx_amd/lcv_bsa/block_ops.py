"""Fused row operations of the DiT block (HIP), with torch tensors.

``residual_norm`` covers the block's AdaLN modulation, gated residuals and
the cross-attention pre-norm (longcat_video_dit.py:107-136; blocks.py:
79-119), ``swiglu`` the SwiGLU gate (blocks.py:50-51) and ``head_rms_norm``
the cross-attention's per-head q / k norms (attention.py:325-326).  Each is
one pass over HBM through ``liblcv_bsa.so``; each rounds like the
reference's sequence of fp32 tensor operations followed by a cast.
``adaln_modulation`` gives the fp32 modulation of a timestep embedding
(longcat_video_dit.py:80-138), ``text_attention`` is the cross-attention itself with the q norm inside
(attention.py:318-352).
"""

from __future__ import annotations

import ctypes
from typing import Optional, Sequence

import torch

from . import _lib
from .block_sparse_attention import _dtype_code, _require_device, _stream, _strides

__all__ = ["residual_norm", "swiglu", "head_rms_norm", "adaln_modulation", "text_attention", "plain_tensors",
           "unwatched"]


def unwatched(*ts: torch.Tensor) -> bool:
    """No transform, trace or tensor subclass looks on what torch does with ``ts``."""
    if (torch.autograd.forward_ad._current_level >= 0 or torch._C._functorch.peek_interpreter_stack() is not None
            or torch.compiler.is_compiling() or torch.jit.is_tracing() or torch._C._len_torch_dispatch_stack() > 0):
        return False
    return all(type(t) in (torch.Tensor, torch.nn.Parameter) for t in ts)


def plain_tensors(*ts: Optional[torch.Tensor]) -> bool:
    """Whether a chain of torch operations over these GPU tensors (None skipped)
    may run as one kernel that autograd and torch's tracers do not see: 16-bit
    tensors of one dtype on one device, no gradient wanted from them (reverse or
    forward mode), no transform, trace or tensor subclass looking on."""
    ts = [t for t in ts if t is not None]
    t0 = ts[0]
    if not t0.is_cuda or t0.dtype not in (torch.float16, torch.bfloat16):
        return False
    if torch.is_grad_enabled() and any(t.requires_grad for t in ts):
        return False
    return unwatched(*ts) and all(t.dtype == t0.dtype and t.device == t0.device for t in ts)


def _ptr(t: Optional[torch.Tensor]):
    return None if t is None else t.data_ptr()


def _rows(t: torch.Tensor, name: str, shape) -> torch.Tensor:
    if tuple(t.shape) != tuple(shape):
        raise ValueError(f"{name} must be {tuple(shape)}, got {tuple(t.shape)}")
    return t.contiguous()


def residual_norm(
    x: torch.Tensor,
    a: Optional[torch.Tensor] = None,
    gate: Optional[torch.Tensor] = None,
    *,
    frames: int,
    shift: Optional[torch.Tensor] = None,
    scale: Optional[torch.Tensor] = None,
    weight: Optional[torch.Tensor] = None,
    bias: Optional[torch.Tensor] = None,
    eps: float = 1e-6,
    residual: bool = True,
    norm: bool = True,
):
    """``x``, ``a``: ``[B, N, C]`` fp16 / bf16.  Forms ``r = x``, ``x + a`` or
    ``x + gate * a`` (gate fp32 ``[B, frames, C]`` or ``[B, frames, 1, C]``),
    and ``LayerNorm(r)`` with the affine ``weight`` / ``bias`` or the AdaLN
    ``shift`` / ``scale`` (fp32, per frame).  Returns ``(r, n)`` (each None
    when not asked for; ``r`` is ``x`` itself when ``a`` is None)."""
    _require_device(x)
    B, N, C = x.shape
    x = x.contiguous()
    fshape = (B, frames, C)

    def per_frame(t, name):
        if t is None:
            return None
        t = t.reshape(t.shape[0], t.shape[1], -1) if t.dim() == 4 else t
        if t.dtype != torch.float32:
            raise ValueError(f"{name} must be fp32")
        return _rows(t, name, fshape)

    a = None if a is None else _rows(a, "a", x.shape)
    gate, shift, scale = per_frame(gate, "gate"), per_frame(shift, "shift"), per_frame(scale, "scale")
    if weight is not None:
        weight = _rows(weight.to(x.dtype), "weight", (C,))
        bias = _rows(bias.to(x.dtype), "bias", (C,))
    r = torch.empty_like(x) if (a is not None and residual) else None
    n = torch.empty_like(x) if norm else None
    st = _lib.load().lcv_bsa_block_rows(
        x.data_ptr(), _ptr(a), _dtype_code(x), B, N, C, int(frames), _ptr(gate), _ptr(shift), _ptr(scale),
        _ptr(weight), _ptr(bias), float(eps), _ptr(r), _ptr(n), _stream(x))
    _lib.check(st, "residual_norm")
    return (x if a is None else r), n


def swiglu(h13: torch.Tensor) -> torch.Tensor:
    """``h13``: ``[..., 2 * hidden]`` (w1 output then w3 output) ->
    ``silu(h1) * h3`` of shape ``[..., hidden]``."""
    _require_device(h13)
    h = h13.contiguous()
    hidden = h.shape[-1] // 2
    rows = h.numel() // h.shape[-1]
    out = torch.empty((*h.shape[:-1], hidden), dtype=h.dtype, device=h.device)
    st = _lib.load().lcv_bsa_block_swiglu(h.data_ptr(), _dtype_code(h), rows, hidden, out.data_ptr(), _stream(h))
    _lib.check(st, "swiglu")
    return out


def head_rms_norm(x: torch.Tensor, weight: Optional[torch.Tensor], eps: float = 1e-6,
                  out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """RMSNorm_FP32 over the last dim of a ``[B, H, S, D]`` view (any strides
    with dense D) into ``out`` (default: contiguous ``[B, H, S, D]``)."""
    _require_device(x, *(t for t in (weight, out) if t is not None))
    B, H, S, D = x.shape
    if out is None:
        out = torch.empty((B, H, S, D), dtype=x.dtype, device=x.device)
    if weight is not None:
        weight = _rows(weight.to(x.dtype), "weight", (D,))
    st = _lib.load().lcv_bsa_head_rms_norm(
        x.data_ptr(), _dtype_code(x), B, H, S, D, _strides(x), _ptr(weight), float(eps),
        out.data_ptr(), _strides(out), _stream(x))
    _lib.check(st, "head_rms_norm")
    return out


def adaln_modulation(t: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor, chunks: int) -> torch.Tensor:
    """``silu(t) @ weight^T + bias`` in fp32 for ``t`` ``[B, T, K]`` fp32 and a
    half-precision ``weight`` ``[chunks * C, K]``: ``[chunks, B, T, C]``."""
    _require_device(t, weight, bias)
    B, T, K = t.shape
    C = weight.shape[0] // chunks
    if t.dtype != torch.float32 or bias.dtype != weight.dtype:
        raise ValueError(f"t must be fp32 and bias of weight's dtype, got {t.dtype}, {bias.dtype}, {weight.dtype}")
    t, weight, bias = t.contiguous(), _rows(weight, "weight", (chunks * C, K)), _rows(bias, "bias", (chunks * C,))
    out = torch.empty((chunks, B, T, C), dtype=torch.float32, device=t.device)
    st = _lib.load().lcv_bsa_adaln(t.data_ptr(), weight.data_ptr(), bias.data_ptr(), _dtype_code(weight), B * T, K,
                                   chunks, C, out.data_ptr(), _stream(t))
    _lib.check(st, "adaln_modulation")
    return out


def text_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, text_len: Sequence[int],
                   q_weight: torch.Tensor, eps: float, sm_scale: float, out: torch.Tensor) -> torch.Tensor:
    """``q`` ``[B, H, N, D]`` (normalised here, RMSNorm_FP32) over the packed
    text ``k`` (normalised), ``v`` ``[H, L, D]``: item b attends to the
    ``text_len[b]`` rows after those of the items before it.  Writes ``out``
    ``[B, H, N, D]`` (any strides with dense D)."""
    _require_device(q, k, v, out, q_weight)
    B, H, N, D = q.shape
    L = k.shape[1]
    if tuple(k.shape) != (H, L, D) or tuple(v.shape) != (H, L, D) or tuple(out.shape) != (B, H, N, D):
        raise ValueError(f"k, v must be [{H}, L, {D}] and out {tuple(q.shape)}: got {tuple(k.shape)}, "
                         f"{tuple(v.shape)}, {tuple(out.shape)}")
    if len(text_len) != B:
        raise ValueError(f"{len(text_len)} text lengths for {B} batch items")
    if not (q.dtype == k.dtype == v.dtype == out.dtype) or any(t.stride(-1) != 1 for t in (q, k, v, out)):
        raise ValueError("q, k, v, out must share a dtype and have unit stride in their last dimension")
    weight = _rows(q_weight.to(q.dtype), "q_weight", (D,))
    st = _lib.load().lcv_bsa_text_attn(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), _dtype_code(q), B, H, N, L, D, _strides(q), _strides(k[None]),
        _strides(v[None]), (ctypes.c_int64 * B)(*text_len), weight.data_ptr(), float(eps), float(sm_scale),
        out.data_ptr(), _strides(out), _stream(q))
    _lib.check(st, "text_attention")
    return out
