"""prepare_qkv: the pre-BSA pass around a KV cache, against prepare_qk over the
whole sequence (the same arithmetic, so the same bits), and the attention layer
with and without it."""

from __future__ import annotations

import math

import pytest
import torch
from conftest import NORM_CHANGES, changed_norms

from lcv_bsa import mean_pool_blocks_3d, prepare_qk, prepare_qkv
from lcv_bsa.block_ops import head_rms_norm

pytestmark = pytest.mark.gpu

# (cached frames, new frames, H, W, blocks): runs of 64, voxels, a single new
# frame, a cache of one block, no cache.
CASES = [
    (4, 4, 8, 16, "runs"),
    (2, 2, 10, 16, "runs"),     # 320 cached tokens of 640
    (3, 5, 8, 16, "voxel1"),    # (1, 4, 16) voxels: any frame count
    (4, 8, 8, 12, "voxel4"),
    (6, 1, 8, 8, "runs"),
    (1, 64, 2, 32, "runs"),
    (0, 4, 8, 16, "runs"),
]


def _geom(blocks, frames, H, W):
    if blocks == "runs":
        return (1, 1, frames * H * W), (1, 1, 64)
    chunk = (4, 4, 4) if blocks == "voxel4" else (1, 4, 16)
    return (frames, H, W), chunk


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("cached,new,Hl,Wl,blocks", CASES)
def test_cache_matches_whole_sequence(device, dtype, D, cached, new, Hl, Wl, blocks):
    geom = lambda f: _geom(blocks, f, Hl, Wl)  # noqa: E731
    B, H, HW = 2, 3, Hl * Wl
    S, Sc = (cached + new) * HW, cached * HW
    g = torch.Generator(device="cpu").manual_seed(S + D)
    qkv = torch.randn(B, S, 3, H, D, generator=g).to(device, dtype)
    qkv[:, :Sc] = qkv[:1, :Sc]  # one cache for both batch items
    q, k, v = (qkv[:, :, i].transpose(1, 2) for i in range(3))
    wq, wk = ((1 + 0.2 * torch.randn(D, generator=g)).to(device, dtype) for _ in range(2))
    grid = (cached + new, Hl, Wl)
    kshape, chunk = geom(cached + new)
    weights = dict(q_weight=wq, k_weight=wk)
    q_all, k_all, _, kb_all = prepare_qk(q, k, grid, shape=kshape, chunk_thw=chunk, **weights)
    kn_all = head_rms_norm(k, wk)
    cache = (kn_all[:1, :, :Sc], v[:1, :, :Sc]) if cached else None
    kn = torch.full((B, new * HW, H, D), 3.0, dtype=dtype, device=device).transpose(1, 2)
    qo, ko, vo, qb, kb = prepare_qkv(q[:, :, Sc:], k[:, :, Sc:], v[:, :, Sc:], grid, geom(new)[0], kshape, chunk,
                                     cache=cache, k_norm=kn, **weights)
    assert torch.equal(qo, q_all[:, :, Sc:]) and torch.equal(ko, k_all) and torch.equal(vo, v)
    assert torch.equal(kn, kn_all[:, :, Sc:]) and torch.equal(kb, kb_all)
    # fp32 means of the same 64 values in another order: 64 roundings of 2^-24.
    ref = mean_pool_blocks_3d(qo, geom(new)[0], chunk)
    assert (qb - ref).abs().max() <= 64 * 2.0 ** -24 * qo.float().abs().max()


def test_rejects_mismatched_arguments(device):
    q = torch.zeros(1, 2, 128, 64, dtype=torch.float16, device=device)
    c = torch.zeros(1, 2, 64, 64, dtype=torch.float16, device=device)
    runs = lambda n: (1, 1, n)  # noqa: E731
    ok = lambda **kw: prepare_qkv(q, q, kw.pop("v", q), kw.pop("grid", (3, 8, 8)), runs(128), runs(192),  # noqa: E731
                                  (1, 1, 64), **{"cache": (c, c), **kw})
    ok()
    for bad in (dict(cache=(c, c[:, :, :32])), dict(cache=(c.float(), c.float())), dict(v=None), dict(grid=(2, 8, 8)),
                dict(v=q[:, :, :64]), dict(k_norm=torch.empty_like(q[:, :1])), dict(eps=-1.0)):
        with pytest.raises(ValueError):
            ok(**bad)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("policy,ncl", [("contiguous", 2), ("reference", 4)])
def test_layer_cache_with_and_without_gradients(device, calls, dtype, policy, ncl):
    """Without gradients the layer fills and continues its cache through
    prepare_qkv, with them through torch's operations: the same result to the
    order of the row sums, and the cache still differentiable."""
    from lcv_bsa import dit_block
    from lcv_bsa.dit_block import Attention

    kernel = calls(dit_block, "prepare_qkv")
    torch.manual_seed(3)
    C, H, Hl, Wl, T = 256, 2, 8, 16, 4
    a = Attention(C, H, dtype=dtype, device=device)
    a.enable_bsa, a.bsa_cond_noise, a.bsa_shape_policy = True, True, policy
    x = torch.randn(2, (ncl + T) * Hl * Wl, C, dtype=dtype, device=device)
    nc = ncl * Hl * Wl

    def both():
        a.bsa_top_k = ncl * Hl * Wl // 64  # every block: no routing ties
        out, cache = a(x[:, :nc], (ncl, Hl, Wl), return_kv=True)
        a.bsa_top_k = (ncl + T) * Hl * Wl // 64
        return out, *cache, a.forward_with_kv_cache(x[:, nc:], (T, Hl, Wl), ncl, cache)

    slow = both()
    assert slow[1].requires_grad and slow[1].grad_fn is not None and not kernel
    with torch.no_grad():
        fast = both()
    assert len(kernel) == 2
    eps = 2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7
    for f, s in zip(fast, slow):
        assert f.shape == s.shape and f.stride() == s.stride()
        # a unit in the last place here and there, averaged out by the 2-norm
        assert (f.float() - s.float()).norm() <= eps * s.float().norm()
    assert math.isfinite(float(slow[1].detach().float().sum()))


@pytest.mark.parametrize("what", NORM_CHANGES)
def test_layer_runs_its_norms_as_modules(device, what):
    """Around a KV cache, hooks on the norms fire and another norm counts: the same
    bits as with gradients, which torch's sequence gives."""
    from lcv_bsa.dit_block import Attention

    torch.manual_seed(4)
    C, H, Hl, Wl, ncl, T = 256, 2, 8, 16, 2, 4
    a = Attention(C, H, dtype=torch.float16, device=device)
    a.enable_bsa, a.bsa_cond_noise, a.bsa_shape_policy = True, True, "contiguous"
    x = torch.randn(1, (ncl + T) * Hl * Wl, C, dtype=torch.float16, device=device)
    nc = ncl * Hl * Wl

    def both():
        out, cache = a(x[:, :nc], (ncl, Hl, Wl), return_kv=True)
        return out, *cache, a.forward_with_kv_cache(x[:, nc:], (T, Hl, Wl), ncl, cache)

    with changed_norms(what, a):
        want = both()
        with torch.no_grad():
            got = both()
    assert all(torch.equal(g, w) for g, w in zip(got, want))
