"""Pre-BSA preparation of q and k: RMSNorm + 3D RoPE + block means, in one pass.

In the DiT's attention layer the BSA inputs are produced by
(longcat_video/models/attention.py:191-201)::

    q, k, v = split(qkv(x))            # [B, H, N, D] views of the QKV output
    q = self.q_norm(q); k = self.k_norm(k)   # RMSNorm_FP32(head_dim, eps=1e-6)
    q, k = self.rope_3d(q, k, shape)

and BSA then pools q and k per block (block_sparse_attention.py:98-104).
``prepare_qk`` does all of it in one HIP pass over q and k
(``lcv_bsa_prepare_qk``), returning the prepared q, k and their fp32 block
means, which ``bsa_attention(..., block_means=(qbar, kbar))`` consumes
instead of pooling again.

RMSNorm_FP32 (longcat_video/models/blocks.py:55-72): ``x * rsqrt(mean(x^2) +
eps)`` in fp32, rounded to the input dtype, then multiplied by the weight in
that dtype.  rope_3d (rope_3d.py:107-128): widened to fp32,
``x*cos + rotate_half(x)*sin``, rounded back.  The cos / sin table is built
here with the reference's angle formula (rope_3d.py:65-93).
"""

from __future__ import annotations

import threading
from typing import Optional, Sequence

import torch

from . import _lib
from .block_sparse_attention import (
    _aligned_rows, _bhsd, _check_shape, _dtype_code, _geom, _require_device, _stream, _strides,
    num_blocks,
)
from .rope_3d import BASE, rope_dims

__all__ = ["rope_table", "prepare_qk", "prepare_qkv", "RMS_EPS"]

RMS_EPS = 1e-6  # q_norm / k_norm, attention.py:53-54


def _axis_table(dim: int, n: int, device) -> tuple[torch.Tensor, torch.Tensor]:
    idx = torch.arange(0, dim, 2, dtype=torch.float32, device=device)[: dim // 2]
    inv = 1.0 / (BASE ** (idx / dim))
    ang = torch.arange(0, n, dtype=torch.float32, device=device)[:, None] * inv[None, :]
    return torch.cos(ang).reshape(-1), torch.sin(ang).reshape(-1)


_TABLES: dict = {}
_TABLES_LOCK = threading.Lock()
_MAX_TABLE_BYTES = 256 << 20  # about 10,000 tables of a 720p grid
_table_bytes = 0              # held now


def rope_table(head_dim: int, grid: Sequence[int], device=None) -> torch.Tensor:
    """The per-axis cos / sin table of ``lcv_bsa_prepare_qk`` (fp32, flat):
    cos_t, sin_t [T, dt/2], cos_h, sin_h [Hl, dh/2], cos_w, sin_w [Wl, dw/2].

    Built once per (head_dim, grid, device) and kept: the kernel only reads
    it, and building it takes about thirty small launches (~0.15 ms at
    720p), which would otherwise recur in every attention layer.  A table is
    complete before it is kept, so that any stream may read it, and none is
    dropped, so that a kernel in flight or in a graph keeps the one it reads.
    Once 256 MiB are held, further ones are built for the caller's stream alone,
    without a wait; so is one built under stream capture, which belongs to that
    graph."""
    global _table_bytes
    dev = torch.device(device) if device is not None else torch.device("cpu")
    if dev.type == "cuda" and dev.index is None:
        dev = torch.device("cuda", torch.cuda.current_device())
    key = (int(head_dim), tuple(int(x) for x in grid), dev)
    table = _TABLES.get(key)
    if table is not None:
        return table
    table = _build_table(head_dim, grid, dev)
    size = table.numel() * table.element_size()
    if _table_bytes + size > _MAX_TABLE_BYTES:
        return table
    if dev.type == "cuda":
        with torch.cuda.device(dev):
            if torch.cuda.is_current_stream_capturing():
                return table
        torch.cuda.current_stream(dev).synchronize()
    with _TABLES_LOCK:
        if key not in _TABLES and _table_bytes + size <= _MAX_TABLE_BYTES:
            _TABLES[key] = table
            _table_bytes += size
        return _TABLES.get(key, table)


def _build_table(head_dim: int, grid: Sequence[int], device) -> torch.Tensor:
    T, Hl, Wl = (int(x) for x in grid)
    dt, dh, dw = rope_dims(head_dim)
    parts = []
    for dim, n in ((dt, T), (dh, Hl), (dw, Wl)):
        parts.extend(_axis_table(dim, n, device))
    return torch.cat(parts).contiguous()


def _norm_weights(ws, q: torch.Tensor):
    D = q.shape[-1]
    for w in ws:
        if w is not None and w.shape != (D,):
            raise ValueError(f"norm weight must be [{D}], got {tuple(w.shape)}")
    return [None if w is None else w.to(device=q.device, dtype=q.dtype).contiguous() for w in ws]


def _device_table(lib, D: int, g, grid: Sequence[int], device) -> torch.Tensor:
    n_tab = lib.lcv_bsa_rope_table_len(D, g)
    if n_tab == 0:
        raise ValueError(f"prepare_qk supports D in {{64, 128}} and RoPE grids up to the table limit "
                         f"(D={D}, grid={tuple(grid)})")
    table = rope_table(D, grid, device)
    assert table.numel() == n_tab
    return table


def _ptr(t: Optional[torch.Tensor]):
    return None if t is None else t.data_ptr()


def prepare_qk(
    q: torch.Tensor,
    k: torch.Tensor,
    grid: Sequence[int],
    *,
    q_weight: Optional[torch.Tensor] = None,
    k_weight: Optional[torch.Tensor] = None,
    eps: float = RMS_EPS,
    shape: Optional[Sequence[int]] = None,
    chunk_thw: Sequence[int] = (4, 4, 4),
):
    """RMSNorm + 3D RoPE of q and k (``[B, H, S, D]``, fp16 / bf16, any row
    strides) over the latent ``grid`` (T, H, W), plus their block means for
    the BSA geometry ``shape`` / ``chunk_thw`` (``shape`` defaults to
    ``grid``; blocks must hold 64 tokens).

    Returns ``(q_out, k_out, q_blocks, k_blocks)``: contiguous q, k in the
    input dtype and fp32 ``[B, H, nb, D]`` means.
    """
    _require_device(q, k)
    q, k = _bhsd(q, "q"), _bhsd(k, "k")
    if q.shape != k.shape or q.dtype != k.dtype:
        raise ValueError("q and k must share shape and dtype")
    B, H, S, D = q.shape
    shape = tuple(grid) if shape is None else tuple(shape)
    _check_shape(S, shape, chunk_thw)
    code = _dtype_code(q)
    q, k = _aligned_rows(q), _aligned_rows(k)
    weights = _norm_weights((q_weight, k_weight), q)
    lib = _lib.load()
    g = _lib.Grid(*(int(x) for x in grid))
    table = _device_table(lib, D, g, grid, q.device)
    nb = num_blocks(shape, chunk_thw)
    q_out = torch.empty((B, H, S, D), dtype=q.dtype, device=q.device)
    k_out = torch.empty_like(q_out)
    q_blocks = torch.empty((B, H, nb, D), dtype=torch.float32, device=q.device)
    k_blocks = torch.empty_like(q_blocks)
    st = lib.lcv_bsa_prepare_qk(
        q.data_ptr(), k.data_ptr(), code, B, H, S, D, _strides(q), _strides(k),
        _ptr(weights[0]), _ptr(weights[1]), float(eps), g, table.data_ptr(), table.numel(), _geom(shape, chunk_thw),
        q_out.data_ptr(), k_out.data_ptr(), _strides(q_out), _strides(k_out),
        q_blocks.data_ptr(), k_blocks.data_ptr(), _stream(q),
    )
    _lib.check(st, "prepare_qk")
    return q_out, k_out, q_blocks, k_blocks


def prepare_qkv(
    q: torch.Tensor,
    k: torch.Tensor,
    v: Optional[torch.Tensor],
    grid: Sequence[int],
    shape: Sequence[int],
    kv_shape: Sequence[int],
    chunk_thw: Sequence[int],
    *,
    cache: Optional[tuple[torch.Tensor, torch.Tensor]] = None,
    k_norm: Optional[torch.Tensor] = None,
    q_weight: Optional[torch.Tensor] = None,
    k_weight: Optional[torch.Tensor] = None,
    eps: float = RMS_EPS,
):
    """``prepare_qk`` around a KV cache, in one pass (``lcv_bsa_prepare_qkv``).

    ``cache=(k, v)`` holds the normed, un-rotated k and the v of earlier tokens
    (``[B or 1, H, S_c, D]``) that the new ``q, k, v`` ``[B, H, S, D]`` follow;
    ``grid`` is the latent grid of all ``S_c + S`` tokens, ``shape`` / ``kv_shape``
    the BSA geometries of q and of cached + new k.  Without a cache ``v`` may be
    None.  ``k_norm``, if given, receives the new k after its norm and before
    RoPE: what a cache holds.

    Returns ``(q_out, k_out, v_out, q_blocks, k_blocks)`` with k_out and v_out
    over ``S_c + S`` tokens (v_out None when v is).
    """
    _require_device(q, k, *([] if v is None else [v]), *(cache or ()), *([] if k_norm is None else [k_norm]))
    q, k = _bhsd(q, "q"), _bhsd(k, "k")
    v = None if v is None else _bhsd(v, "v")
    B, H, S, D = q.shape
    cached = cache[0].shape[2] if cache is not None else 0
    full = (B, H, cached + S, D)
    for name, t in (("k", k), ("v", v), ("k_norm", k_norm)):
        if t is not None and (t.shape != q.shape or t.dtype != q.dtype):
            raise ValueError(f"{name} must be {tuple(q.shape)} {q.dtype}, got {tuple(t.shape)} {t.dtype}")
    if cache is not None and v is None:
        raise ValueError("a cache needs the new v")
    if k_norm is not None and k_norm.stride(-1) != 1:
        raise ValueError("k_norm must have unit stride in its last dimension")
    old = [None, None]
    for i, c in enumerate(cache or ()):
        if c.dim() != 4 or c.shape[0] not in (1, B) or tuple(c.shape[1:]) != (H, cached, D) or c.dtype != q.dtype:
            raise ValueError(f"cache must hold [{B} or 1, {H}, {cached}, {D}] {q.dtype}, got {tuple(c.shape)} {c.dtype}")
        old[i] = _aligned_rows(_bhsd(c, "cache")).expand(B, H, cached, D)
    _check_shape(S, shape, chunk_thw)
    _check_shape(cached + S, kv_shape, chunk_thw)
    code = _dtype_code(q)
    q, k = _aligned_rows(q), _aligned_rows(k)
    v = None if v is None else _aligned_rows(v)
    weights = _norm_weights((q_weight, k_weight), q)
    lib = _lib.load()
    g = _lib.Grid(*(int(x) for x in grid))
    table = _device_table(lib, D, g, grid, q.device)
    nb, nk = num_blocks(shape, chunk_thw), num_blocks(kv_shape, chunk_thw)
    q_out = torch.empty((B, H, S, D), dtype=q.dtype, device=q.device)
    k_out = torch.empty(full, dtype=q.dtype, device=q.device)
    v_out = None if v is None else torch.empty(full, dtype=q.dtype, device=q.device)
    q_blocks = torch.empty((B, H, nb, D), dtype=torch.float32, device=q.device)
    k_blocks = torch.empty((B, H, nk, D), dtype=torch.float32, device=q.device)
    none = _lib.Strides(0, 0, D)

    def strides(t):
        return none if t is None else _strides(t)

    st = lib.lcv_bsa_prepare_qkv(
        q.data_ptr(), k.data_ptr(), _ptr(v), code, B, H, S, D, _strides(q), _strides(k), strides(v),
        _ptr(old[0]), _ptr(old[1]), cached, strides(old[0]), strides(old[1]), _ptr(weights[0]), _ptr(weights[1]),
        float(eps), g, table.data_ptr(), table.numel(), _geom(shape, chunk_thw), _geom(kv_shape, chunk_thw),
        q_out.data_ptr(), k_out.data_ptr(), _ptr(v_out), _ptr(k_norm), _strides(q_out), _strides(k_out),
        strides(v_out), strides(k_norm), q_blocks.data_ptr(), k_blocks.data_ptr(), _stream(q),
    )
    _lib.check(st, "prepare_qkv")
    return q_out, k_out, v_out, q_blocks, k_blocks
