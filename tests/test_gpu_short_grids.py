"""Small grids: routing in one kernel and attention without a launch order,
at and around the sizes where the forward switches, against the stages."""

from __future__ import annotations

import math

import pytest
import torch

from lcv_bsa import bsa_attention, bsa_attention_hip, mean_pool_blocks_3d, schedule_block_order, select_block_indices

pytestmark = pytest.mark.gpu


def _qkv(device, dtype, H, nq, nk, D, seed):
    g = torch.Generator(device="cpu").manual_seed(seed)
    return tuple(torch.randn(1, H, 64 * n, D, generator=g).to(device, dtype) for n in (nq, nk, nk))


def _attend(q, k, v, idx, nq, nk, order):
    """The attention stage alone, in the launch order given."""
    from lcv_bsa import _lib
    from lcv_bsa.block_sparse_attention import _dtype_code, _geom, _stream, _strides

    out, (_, H, S, D) = torch.empty_like(q), q.shape
    st = _lib.load().lcv_bsa_attn_fwd_kv(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), _dtype_code(q), 1, H, S, k.shape[2], D, _strides(q), _strides(k),
        _strides(v), idx.data_ptr(), None if order is None else order.data_ptr(), idx.shape[-1], D ** -0.5,
        _geom((1, 1, 64 * nq), (1, 1, 64)), _geom((1, 1, 64 * nk), (1, 1, 64)), out.data_ptr(), _strides(out),
        _stream(q))
    _lib.check(st, "attn_fwd_kv")
    return out


# (H, q-blocks, k-blocks): one block, one key tile and one past it, the widest
# fused rows, the last and first grids of 256 workgroups, 320 / 321 blocks, and
# 6,144 / 6,150 attention workgroups.
GRIDS = [(1, 1, 1), (2, 32, 32), (2, 33, 33), (1, 256, 256), (1, 257, 257), (8, 256, 256), (9, 256, 256),
         (3, 7, 255), (1, 320, 320), (1, 321, 321), (2, 64, 321), (4, 1, 40),
         (24, 256, 256), (25, 246, 246), (8, 224, 224), (2, 225, 225), (9, 224, 224), (10, 224, 224), (8, 3, 224)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("H,nq,nk", GRIDS)
def test_forward_matches_stages(device, dtype, D, H, nq, nk):
    q, k, v = _qkv(device, dtype, H, nq, nk, D, seed=nq + nk)
    shape, kv_shape, chunk = (1, 1, 64 * nq), (1, 1, 64 * nk), (1, 1, 64)
    top_k = max(1, math.ceil(nk / 16))
    means = mean_pool_blocks_3d(q, shape, chunk), mean_pool_blocks_3d(k, kv_shape, chunk)
    idx = select_block_indices(*means, top_k)  # score GEMM + top-k
    assert torch.equal(select_block_indices(*means, top_k, fused=True), idx)
    want = bsa_attention_hip(q, k, v, idx, chunk, shape, kv_shape=kv_shape)
    more = {} if nq == nk else {"kv_shape": kv_shape}
    for kw in ({}, {"block_means": means}):
        out, got = bsa_attention(q, k, v, shape, chunk_thw=chunk, top_k=top_k, return_indices=True, **kw, **more)
        assert torch.equal(got, idx) and torch.equal(out, want)


@pytest.mark.parametrize("D", [16, 32])
def test_other_head_dims_match_stages(device, D):
    q, k, v = _qkv(device, torch.float16, 2, 32, 32, D, seed=D)
    shape, chunk = (1, 1, 2048), (1, 1, 64)
    idx = select_block_indices(*(mean_pool_blocks_3d(t, shape, chunk) for t in (q, k)), 3)
    out, got = bsa_attention(q, k, v, shape, chunk_thw=chunk, top_k=3, return_indices=True)
    assert torch.equal(got, idx) and torch.equal(out, bsa_attention_hip(q, k, v, idx, chunk, shape))


@pytest.mark.parametrize("H,nk", [(2, 319), (2, 320)])
def test_order_is_a_permutation_below_the_line(device, H, nk):
    """The launch order stays available where the forward no longer sorts."""
    q, k, _ = _qkv(device, torch.float16, H, nk, nk, 64, seed=nk)
    idx = select_block_indices(mean_pool_blocks_3d(q, (1, 1, 64 * nk), (1, 1, 64)),
                               mean_pool_blocks_3d(k, (1, 1, 64 * nk), (1, 1, 64)), 20)
    order = schedule_block_order(idx)
    assert torch.equal(order.sort(-1).values, torch.arange(nk, device=device, dtype=torch.int32).expand(1, H, nk))


def test_pool_of_two_grids_in_one_launch(device):
    """q and k of different frame sizes share the pooling launch."""
    g = torch.Generator(device="cpu").manual_seed(5)
    shape, kv_shape, chunk = (4, 8, 8), (8, 12, 16), (4, 4, 4)
    q = torch.randn(1, 3, 256, 64, generator=g).to(device, torch.float16)
    k, v = (torch.randn(1, 3, 1536, 64, generator=g).to(device, torch.float16) for _ in range(2))
    means = mean_pool_blocks_3d(q, shape, chunk), mean_pool_blocks_3d(k, kv_shape, chunk)
    kw = dict(chunk_thw=chunk, top_k=5, kv_shape=kv_shape, return_indices=True)
    out, idx = bsa_attention(q, k, v, shape, **kw)
    want, widx = bsa_attention(q, k, v, shape, block_means=means, **kw)
    assert torch.equal(idx, widx) and torch.equal(out, want)


@pytest.mark.parametrize("H,nq,nk,ordered", [(24, 256, 320, False), (25, 246, 320, True), (24, 200, 321, True)])
def test_order_is_left_out_of_small_grids_only(device, H, nq, nk, ordered):
    """Beyond the line the forward gives the bits of the ordered stages."""
    q, k, v = _qkv(device, torch.bfloat16, H, nq, nk, 64, seed=nk)
    shape, kv_shape, chunk = (1, 1, 64 * nq), (1, 1, 64 * nk), (1, 1, 64)
    out, idx = bsa_attention(q, k, v, shape, chunk_thw=chunk, top_k=20, return_indices=True, kv_shape=kv_shape)
    want = _attend(q, k, v, idx, nq, nk, schedule_block_order(idx, nk) if ordered else None)
    assert torch.equal(out, want)
    other = _attend(q, k, v, idx, nq, nk, None if ordered else schedule_block_order(idx, nk))
    assert not torch.equal(out, other)  # another order of the sums
    assert (out.float() - other.float()).norm() <= 2.0 ** -8 * out.float().norm()
