"""The work that users of this package have it do, as timed cases.

A case is one call of a public entry point:

* ``bsa``: ``bsa_attention`` on head-major q, k, v, as ``_process_attn`` calls
  it (self-attention), or with ``kv_frames`` more frames of keys in front
  (noise queries over conditioning + noise keys);
* ``prefill``: the DiT's self-attention layer over the conditioning frames,
  returning its KV cache;
* ``continue``: the same layer over the noise frames that follow, from such a
  cache;
* ``split``: the same layer over conditioning and noise frames in one call
  (image-to-video);
* ``cross``: the text cross-attention layer, whose text lengths are whatever
  the prompts' token counts are;
* ``block``: one whole DiT block.

Sizes are the refinement pass's latent grids (45 x 80 tokens a frame at 720p,
30 x 52 at 480p, 4096 hidden = 32 heads of 128), the CPU-runnable size of the
reference's own operator test, and smaller grids between them.
"""

from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "longcat-video-mlx_amd"))

from lcv_bsa import bsa_attention  # noqa: E402
from lcv_bsa.dit_block import Attention, LongCatSingleStreamBlock, MultiHeadCrossAttention  # noqa: E402

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
ESZ = {"f16": 2, "bf16": 2, "f32": 4}
KEEP = 0.0625  # the published sparsity, 0.9375


def bsa(name, dtype, B, H, D, T, Hl, Wl, blocks="runs", keep=KEEP, kv_frames=0):
    """``blocks``: runs of 64 tokens, or 4 x 4 x 4 voxels of the grid."""
    return dict(name=name, kind="bsa", dtype=dtype, B=B, H=H, D=D, T=T, Hl=Hl, Wl=Wl, blocks=blocks, keep=keep,
                kv_frames=kv_frames)


def layer(name, kind, dtype, B, H, T, Hl, Wl, cond=0):
    return dict(name=name, kind=kind, dtype=dtype, B=B, H=H, D=128, T=T, Hl=Hl, Wl=Wl, cond=cond, keep=KEEP)


def cross(name, dtype, H, T, Hl, Wl, text):
    """``text``: token counts of the packed prompts, one per batch item."""
    return dict(name=name, kind="cross", dtype=dtype, B=len(text.split(",")), H=H, D=128, T=T, Hl=Hl, Wl=Wl, text=text)


def block(name, dtype, H, T, Hl, Wl, text):
    return dict(name=name, kind="block", dtype=dtype, B=1, H=H, D=128, T=T, Hl=Hl, Wl=Wl, text=text, keep=KEEP)


def listed():
    return [
        # A preview-size latent with the default voxels: a few hundred
        # workgroups at most, so launches and the host's part count.
        bsa("voxel_preview_f16", "f16", 1, 2, 128, 8, 16, 16, "voxels"),
        # The reference's own CPU-runnable operator size, in its fp32.
        bsa("operator_f32", "f32", 1, 2, 64, 1, 64, 64, "runs"),
        # fp32 inputs at 480p over 8 frames (195 blocks: an odd count): a
        # precision check of a whole layer.
        bsa("clip480_f32", "f32", 1, 8, 128, 8, 30, 52, "runs"),
        # Voxels on a grid that they tile: 3 x 7 x 13 = 273 blocks, bf16.
        bsa("voxel_mid_bf16", "bf16", 1, 32, 128, 12, 28, 52, "voxels"),
        # A short 720p clip, 450 blocks.
        bsa("clip720_f16", "f16", 1, 32, 128, 8, 45, 80, "runs"),
        # The 720p refinement pass, 900 blocks: the headline size.
        bsa("refine720_f16", "f16", 1, 32, 128, 16, 45, 80, "runs"),
        # The guidance pair at 720p, twice the blocks kept (lists over 64).
        bsa("guided720_bf16", "bf16", 2, 32, 128, 16, 45, 80, "runs", keep=0.125),
        # Video continuation at 720p: 16 noise frames over 20 of keys.
        bsa("continued720_f16", "f16", 1, 32, 128, 16, 45, 80, "runs", kv_frames=4),
        # Chunked continuation in the layer: the conditioning frames fill the
        # cache once, and each later call decodes noise frames from it.
        layer("layer_prefill_bf16", "prefill", "bf16", 1, 32, 4, 45, 80),
        layer("layer_continue_bf16", "continue", "bf16", 1, 32, 8, 45, 80, cond=4),
        # Text cross-attention of a guidance pair: a long prompt and a short one.
        cross("cross_text_bf16", "bf16", 32, 8, 45, 80, "231,13"),
        # One whole block of the DiT on a short 720p clip.
        block("block720_f16", "f16", 32, 8, 45, 80, "256"),
    ]


def _grid(rng, lo, hi, multiple=64):
    """A latent grid of lo..hi tokens whose count is a multiple of 64."""
    want = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    while True:
        Hl, Wl = rng.randint(8, 48), rng.randint(8, 80)
        T = max(1, round(want / (Hl * Wl)))
        n = T * Hl * Wl
        if T <= 32 and n % multiple == 0 and lo <= n <= hi:
            return T, Hl, Wl


def _voxel_grid(rng, lo, hi):
    want = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    while True:
        Hl, Wl = 4 * rng.randint(2, 12), 4 * rng.randint(2, 20)
        T = 4 * max(1, round(want / (4 * Hl * Wl)))
        if T <= 32 and lo <= T * Hl * Wl <= hi:
            return T, Hl, Wl


def draw(rng):
    kind = rng.choice(["bsa", "bsa", "bsa", "f32", "kv", "prefill", "continue", "split", "cross", "block"])
    half = rng.choice(["f16", "bf16"])
    if kind == "bsa":
        voxels = rng.random() < 0.4
        grid = _voxel_grid(rng, 1024, 57600) if voxels else _grid(rng, 1024, 57600)
        c = bsa("", half, rng.choice([1, 1, 2]), rng.choice([2, 5, 8, 16, 32]), rng.choice([64, 128, 128]), *grid,
                "voxels" if voxels else "runs", rng.choice([0.03125, 0.0625, 0.125]))
    elif kind == "f32":
        c = bsa("", "f32", 1, rng.choice([1, 2, 3, 8]), rng.choice([64, 128]), *_grid(rng, 1024, 12480), "runs",
                rng.choice([0.03125, 0.0625]))
    elif kind == "kv":
        T, Hl, Wl = _grid(rng, 2048, 57600)
        frames = [f for f in range(1, 9) if f * Hl * Wl % 64 == 0 and f * Hl * Wl <= 14400] or [0]
        c = bsa("", half, 1, rng.choice([2, 8, 32]), 128, T, Hl, Wl, "runs", kv_frames=rng.choice(frames))
    elif kind == "cross":
        text = ",".join(str(rng.randint(1, 512)) for _ in range(rng.choice([1, 2])))
        c = cross("", half, rng.choice([8, 16, 32]), *_grid(rng, 1024, 28800), text)
    elif kind == "block":
        c = block("", half, rng.choice([8, 16, 32]), *_grid(rng, 1024, 28800), str(rng.randint(1, 512)))
    else:
        while True:
            T, Hl, Wl = _grid(rng, 2048, 14400 if kind == "prefill" else 28800)
            frames = [0] if kind == "prefill" else [f for f in range(1, T) if f * Hl * Wl % 64 == 0 and f <= 8]
            if frames:
                break
        c = layer("", kind, half, 1 if kind == "split" else rng.choice([1, 1, 2]) if T * Hl * Wl <= 14400 else 1,
                  rng.choice([8, 16, 32]), T, Hl, Wl, rng.choice(frames))
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# Sizes
# ---------------------------------------------------------------------------

def _geometry(c, frames):
    """(shape, chunk) of ``frames`` frames, and their block count."""
    n = frames * c["Hl"] * c["Wl"]
    if c.get("blocks") == "voxels":
        return (frames, c["Hl"], c["Wl"]), (4, 4, 4), n // 64
    return (1, 1, n), (1, 1, 64), n // 64


def _kept(c, nk):
    return max(1, math.ceil(round(c["keep"] * nk, 9)))


def _attention_work(c, nq, nk):
    """Operations of routing nq blocks over nk and attending the kept ones."""
    heads = c["B"] * c["H"]
    return heads * nq * (2 * nk * c["D"] + 4 * _kept(c, nk) * 64 * 64 * c["D"])


def work(c):
    B, H, D, e = c["B"], c["H"], c["D"], ESZ[c["dtype"]]
    C, n = H * D, c["T"] * c["Hl"] * c["Wl"]
    if c["kind"] == "bsa":
        nk = n + c["kv_frames"] * c["Hl"] * c["Wl"]
        return {"bytes": B * C * e * (2 * n + 2 * nk) + 4 * B * H * (n // 64) * _kept(c, nk // 64),
                "flops": _attention_work(c, n // 64, nk // 64)}
    if c["kind"] == "prefill":
        return {"bytes": e * (4 * C * C + B * n * C * 4), "flops": 8 * B * n * C * C + _attention_work(c, n // 64, n // 64)}
    if c["kind"] == "continue":
        cached = c["cond"] * c["Hl"] * c["Wl"]
        return {"bytes": e * (4 * C * C + B * n * C * 2 + B * cached * C * 2),
                "flops": 8 * B * n * C * C + _attention_work(c, n // 64, (n + cached) // 64)}
    if c["kind"] == "split":
        nc = c["cond"] * c["Hl"] * c["Wl"]
        return {"bytes": e * (4 * C * C + B * n * C * 2),
                "flops": 8 * B * n * C * C + _attention_work(c, nc // 64, nc // 64) + _attention_work(c, (n - nc) // 64, n // 64)}
    text = [int(t) for t in c["text"].split(",")]
    cross_flops = sum(4 * n * C * C + 4 * t * C * C + 4 * n * t * C for t in text)
    if c["kind"] == "cross":
        return {"bytes": e * (4 * C * C + B * n * C * 2 + sum(text) * C), "flops": cross_flops}
    F = _ffn_width(C)
    return {"bytes": e * (8 * C * C + 3 * C * F + 6 * C * T_DIM + 2 * n * C + sum(text) * C),
            "flops": 8 * n * C * C + _attention_work(c, n // 64, n // 64) + cross_flops + 6 * n * C * F}


T_DIM = 512  # timestep embedding width


def _ffn_width(C):
    return 256 * ((int(2 * 4 * C / 3) + 255) // 256)


def tolerance(c):
    """About four times what each kind shows against 64 bits.  Block scores within fp32 rounding of each other may be
    ranked either way: at 720p that is about one row of 28,800, whose output then moves by a fifth of its size."""
    if c["dtype"] == "f32":
        return {"rel": 1e-5, "max": 1e-2, "differ": 1e-3}
    f16 = c["dtype"] == "f16"
    rel = {"bsa": (4e-3, 1e-2), "cross": (3e-3, 2e-2), "block": (5e-3, 2e-2)}.get(c["kind"], (2e-2, 3e-2))[0 if f16 else 1]
    return {"rel": rel, "max": 0.9, "differ": 1e-3}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _angles(grid, D, device, dtype):
    """3D RoPE angles [T*H*W, D]: D - 4 (D // 6) dims over frames, then 2 (D // 6) each over rows and columns."""
    parts = []
    for axis, dim in enumerate((D - 4 * (D // 6), 2 * (D // 6), 2 * (D // 6))):
        inv = 10000.0 ** (-torch.arange(0, dim, 2, dtype=dtype, device=device) / dim)
        a = torch.arange(grid[axis], dtype=dtype, device=device)[:, None] * inv.repeat_interleave(2)
        at = [1, 1, 1, dim]
        at[axis] = grid[axis]
        parts.append(a.reshape(at).expand(*grid, dim))
    return torch.cat(parts, -1).reshape(-1, D)


def _rotate(x, angles):
    """x [..., S, D] turned by the angles of its tokens, pairs (2i, 2i + 1)."""
    turned = torch.stack([-x[..., 1::2], x[..., ::2]], -1).reshape(x.shape)
    return x * angles.cos() + turned * angles.sin()


def _voxel_tokens(shape, chunk, device):
    """[blocks, 64]: the tokens of each block."""
    t = torch.arange(shape[0] * shape[1] * shape[2], device=device)
    split = [n for s, c in zip(shape, chunk) for n in (s // c, c)]
    return t.reshape(split).permute(0, 2, 4, 1, 3, 5).reshape(-1, 64)


def _tokens_alike(gen, dev, B, n, width, rank):
    """[B, n, width] unit normals plus, for each run of 64 tokens, an offset in ``rank`` shared directions: tokens near
    each other in a video are alike, which is what routing works on."""
    x = torch.randn(B, n, width, generator=gen, device=dev)
    basis = torch.randn(rank, width, generator=gen, device=dev) / math.sqrt(rank)
    runs = (n + 63) // 64
    offset = torch.randn(B, runs, rank, generator=gen, device=dev) @ basis
    return x.mul_(0.5).add_(offset.repeat_interleave(64, 1)[:, :n], alpha=1.5)


def _fill(module, gen):
    """Weights of the size that keeps activations of order one; norms near one."""
    with torch.no_grad():
        for name, p in module.named_parameters():
            noise = torch.randn(p.shape, generator=gen, device=p.device)
            if "norm" in name and name.endswith("weight"):
                p.copy_(1 + 0.1 * noise)
            elif name.endswith("bias"):
                p.copy_(0.02 * noise)
            else:
                p.copy_(noise / math.sqrt(p.shape[1]))
    return module


def _bsa_on(attn, c, nk):
    attn.enable_bsa, attn.bsa_shape_policy, attn.bsa_cond_noise = True, "contiguous", True
    attn.bsa_top_k = None if c["kind"] == "split" else _kept(c, nk)  # the two parts of a split have their own counts
    return attn


def prepare(c, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    dtype, grid = DTYPES[c["dtype"]], (c["T"], c["Hl"], c["Wl"])
    B, H, D = c["B"], c["H"], c["D"]
    n = grid[0] * grid[1] * grid[2]
    if c["kind"] == "bsa":
        keys = (grid[0] + c["kv_frames"], grid[1], grid[2])
        shape, chunk, _ = _geometry(c, grid[0])
        kv_shape, _, nk = _geometry(c, keys[0])
        basis = torch.linalg.qr(torch.randn(D, 4, generator=gen, device=dev))[0].T
        angles = _angles(keys, D, dev, torch.float32)

        def heads(g, geom, angles):
            """Unit normals, an offset per block, RoPE: what reaches attention from the DiT's projections."""
            tokens = _voxel_tokens(geom, chunk, dev).reshape(-1)
            out = torch.empty(B, H, len(tokens), D, dtype=dtype, device=dev)
            for b in range(B):
                x = torch.randn(H, len(tokens) // 64, 64, D, generator=gen, device=dev)
                x += (0.5 * torch.randn(H, len(tokens) // 64, 1, 4, generator=gen, device=dev)) @ basis
                out[b][:, tokens] = _rotate(x.reshape(H, -1, D), angles[tokens]).to(dtype)
            return out

        q = heads(grid, shape, angles[-n:])
        k = heads(keys, kv_shape, angles)
        v = torch.randn(k.shape, generator=gen, device=dev).to(dtype)
        more = {"kv_shape": kv_shape} if c["kv_frames"] else {}
        return dict(kind="bsa", args=(q, k, v, shape), options=dict(chunk_thw=chunk, top_k=_kept(c, nk), return_indices=True, **more))
    C = H * D
    x = _tokens_alike(gen, dev, B, n, C, 8).to(dtype)
    kw = dict(dtype=dtype, device=dev)
    if c["kind"] == "cross":
        text = [int(t) for t in c["text"].split(",")]
        y = torch.randn(1, sum(text), C, generator=gen, device=dev).to(dtype)
        return dict(kind="cross", module=_fill(MultiHeadCrossAttention(C, H, **kw), gen), x=x, y=y, text=text)
    if c["kind"] == "block":
        text = [int(t) for t in c["text"].split(",")]
        m = _fill(LongCatSingleStreamBlock(C, H, 4, T_DIM, **kw), gen)
        _bsa_on(m.attn, c, n // 64)
        y = torch.randn(1, sum(text), C, generator=gen, device=dev).to(dtype)
        t = torch.randn(B, grid[0], T_DIM, generator=gen, device=dev)
        return dict(kind="block", module=m, x=x, y=y, t=t, text=text, grid=grid)
    cached = c["cond"] * grid[1] * grid[2] if c["kind"] == "continue" else 0
    m = _bsa_on(_fill(Attention(C, H, **kw), gen), c, (n + cached) // 64)
    state = dict(kind=c["kind"], module=m, x=x, grid=grid, cond=c["cond"])
    if c["kind"] == "continue":  # normed, un-rotated keys, and values, of the frames before; one cache for a guidance pair
        w = m.k_norm.weight.detach().float()
        k = _tokens_alike(gen, dev, 1, cached, C, 8).view(1, cached, H, D).transpose(1, 2)
        k = k * torch.rsqrt(k.square().mean(-1, keepdim=True)) * w
        v = torch.randn(1, H, cached, D, generator=gen, device=dev)
        state["cache"] = (k.to(dtype).contiguous(), v.to(dtype))
    return state


def run(s):
    if s["kind"] == "bsa":
        out, idx = bsa_attention(*s["args"], **s["options"])
        return {"out": out, "idx": idx}
    m = s["module"]
    with torch.no_grad():
        if s["kind"] == "cross":
            return {"out": m(s["x"], s["y"], s["text"])}
        if s["kind"] == "block":
            return {"out": m(s["x"], s["y"], s["t"], s["text"], s["grid"])}
        if s["kind"] == "prefill":
            out, (k, v) = m(s["x"], s["grid"], return_kv=True)
            return {"out": out, "k": k, "v": v}
        if s["kind"] == "continue":
            return {"out": m.forward_with_kv_cache(s["x"], s["grid"], s["cond"], s["cache"])}
        return {"out": m(s["x"], s["grid"], s["cond"])}


# ---------------------------------------------------------------------------
# The same in 64 bits, from the definitions
# ---------------------------------------------------------------------------

def _routed(q, k, v, q_tokens, k_tokens, kept, scale):
    """Attention of [B, H, S, D] in 64 bits: each q-block (rows of ``q_tokens``) over its ``kept`` best blocks."""
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for b in range(q.shape[0]):
        for h in range(q.shape[1]):
            Q, K, V = (x[b, h].double()[t] for x, t in ((q, q_tokens), (k, k_tokens), (v, k_tokens)))  # [blocks, 64, D]
            idx = torch.topk(Q.mean(1) @ K.mean(1).T, kept, dim=-1).indices
            step = max(1, (1 << 25) // (kept * 64 * Q.shape[-1]))
            for i in range(0, len(Q), step):
                keys, values = (x[idx[i:i + step]].flatten(1, 2) for x in (K, V))
                p = torch.softmax(torch.matmul(Q[i:i + step], keys.transpose(1, 2).contiguous()) * scale, -1)
                out[b, h][q_tokens[i:i + step]] = torch.matmul(p, values)
    return out


def _linear(m, x):
    """x @ W^T + b in 64 bits, in slices of rows."""
    w = m.weight.double().T.contiguous()
    rows = x.reshape(-1, x.shape[-1])
    out = torch.empty(len(rows), w.shape[1], dtype=torch.float64, device=x.device)
    for i in range(0, len(rows), 8192):
        out[i:i + 8192] = rows[i:i + 8192].double() @ w
    if m.bias is not None:
        out += m.bias.double()
    return out.reshape(*x.shape[:-1], -1)


def _rms(m, x):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + m.eps) * m.weight.double()


def _heads(x, H):
    B, n, C = x.shape
    return x.view(B, n, H, C // H).transpose(1, 2)


def _self_attention(m, x, grid, kept, H, cond=0, cache=None):
    """(out, k before RoPE, v); ``cond``: frames split off (no cache), or held in the cache."""
    n = grid[0] * grid[1] * grid[2]
    runs = lambda a, b: torch.arange(a, b, device=x.device).view(-1, 64)  # noqa: E731
    q, k, v = (_heads(y, H) for y in _linear(m.qkv, x).chunk(3, -1))
    q, k = _rms(m.q_norm, q), _rms(m.k_norm, k)
    scale = q.shape[-1] ** -0.5
    kc, vc = k, v
    if cache is not None:
        k, v = (torch.cat([old.double().expand(len(new), -1, -1, -1), new], 2) for old, new in zip(cache, (k, v)))
    nk = k.shape[2]
    angles = _angles((nk * grid[0] // n,) + grid[1:], q.shape[-1], x.device, torch.float64)
    q, k = _rotate(q, angles[nk - n:]), _rotate(k, angles)
    if cond and cache is None:
        nc = cond * grid[1] * grid[2]
        o = torch.cat([_routed(q[:, :, :nc], k[:, :, :nc], v[:, :, :nc], runs(0, nc), runs(0, nc), kept(nc // 64), scale),
                       _routed(q[:, :, nc:], k, v, runs(0, n - nc), runs(0, n), kept(n // 64), scale)], 2)
    else:
        o = _routed(q, k, v, runs(0, n), runs(0, nk), kept(nk // 64), scale)
    return _linear(m.proj, o.transpose(1, 2).flatten(2)), kc, vc


def _cross_attention(m, x, y, text, H):
    q = _rms(m.q_norm, _heads(_linear(m.q_linear, x), H))
    k, v = (_heads(z, H) for z in _linear(m.kv_linear, y).chunk(2, -1))
    k = _rms(m.k_norm, k)
    out, off = torch.empty_like(q), 0
    for b, t in enumerate(text):
        kt = k[0, :, off:off + t].transpose(1, 2).contiguous()
        for i in range(0, q.shape[2], 4096):
            p = torch.softmax(torch.matmul(q[b, :, i:i + 4096].contiguous(), kt) * m.scale, -1)
            out[b, :, i:i + 4096] = torch.matmul(p, v[0, :, off:off + t].contiguous())
        off += t
    return _linear(m.proj, out.transpose(1, 2).flatten(2))


def _norm(x, eps):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], eps=eps)


def exact(c, seed):
    s = prepare(c, seed)
    with torch.no_grad():
        if c["kind"] == "bsa":
            q, k, v, shape = s["args"]
            o = s["options"]
            tokens = [_voxel_tokens(g, o["chunk_thw"], q.device) for g in (shape, o.get("kv_shape", shape))]
            return {"out": _routed(q, k, v, *tokens, o["top_k"], c["D"] ** -0.5), "idx": None}
        m, H = s["module"], c["H"]
        if c["kind"] == "cross":
            return {"out": _cross_attention(m, s["x"].double(), s["y"].double(), s["text"], H)}
        if c["kind"] in ("prefill", "continue", "split"):
            count = (lambda nk: max(1, int((1.0 - m.bsa_sparsity) * nk))) if c["kind"] == "split" else (lambda nk: _kept(c, nk))
            out, k, v = _self_attention(m, s["x"].double(), s["grid"], count, H, s["cond"], s.get("cache"))
            return {"out": out, "k": k, "v": v} if c["kind"] == "prefill" else {"out": out}
        x, frames = s["x"].double(), c["T"]
        ada = _linear(m.adaLN_modulation[1], torch.nn.functional.silu(s["t"].double()))
        per = [a.repeat_interleave(x.shape[1] // frames, 1) for a in ada.chunk(6, -1)]
        x_m = _norm(x, 1e-6) * (per[1] + 1) + per[0]
        x = x + per[2] * _self_attention(m.attn, x_m, s["grid"], lambda nk: _kept(c, nk), H)[0]
        pre = m.pre_crs_attn_norm
        x = x + _cross_attention(m.cross_attn, _norm(x, 1e-6) * pre.weight.double() + pre.bias.double(), s["y"].double(), s["text"], H)
        x_m = _norm(x, 1e-6) * (per[4] + 1) + per[3]
        f, out = m.ffn, torch.empty_like(x)
        for i in range(0, x.shape[1], 8192):
            part = x_m[:, i:i + 8192]
            out[:, i:i + 8192] = _linear(f.w2, torch.nn.functional.silu(_linear(f.w1, part)) * _linear(f.w3, part))
        return {"out": x + per[5] * out}
