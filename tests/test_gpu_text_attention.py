"""Text cross-attention kernel (q norm inside, ragged text lengths, any query
count) against fp32 torch on the rounded norms, and the layer's two routes."""

from __future__ import annotations

import math

import pytest
import torch
from conftest import NORM_CHANGES, changed_norms

from lcv_bsa import dit_block
from lcv_bsa.block_ops import head_rms_norm, text_attention
from lcv_bsa.block_sparse_attention import BSADeviceError
from lcv_bsa.dit_block import MultiHeadCrossAttention, RMSNorm_FP32

pytestmark = pytest.mark.gpu

# Batch items' text lengths: one key, edges of the 32-key tiles and of the
# four-slot ring, a full prompt; items of very different lengths; more items
# than one launch holds.
LENGTHS = [(1,), (31, 32), (33,), (63, 64, 65), (96, 7), (127,), (128, 129), (231, 13), (512,), (3,) * 33]


def _inputs(device, dtype, lens, N, H, D, seed, gap=0):
    g = torch.Generator(device="cpu").manual_seed(seed)
    L = sum(lens) + gap
    q = torch.randn(len(lens), N, H, D, generator=g).to(device, dtype)
    kv = torch.randn(L, 2, H, D, generator=g).to(device, dtype)
    w = (1 + 0.2 * torch.randn(D, generator=g)).to(device, dtype)
    return q, kv, w


def _reference(q, k, v, w, lens, scale):
    """[B, N, H, D] fp32 from q rounded as RMSNorm_FP32 rounds it."""
    norm = RMSNorm_FP32(q.shape[-1], 1e-6, dtype=q.dtype, device=q.device)
    with torch.no_grad():
        norm.weight.copy_(w)
        qn = norm(q).float().transpose(1, 2)
    out, off = [], 0
    for b, n in enumerate(lens):
        kb, vb = (t[:, off:off + n].float().contiguous() for t in (k, v))
        p = torch.softmax(torch.matmul(qn[b], kb.transpose(1, 2).contiguous()) * scale, -1)
        out.append(torch.matmul(p, vb).transpose(0, 1))
        off += n
    return torch.stack(out)


def _check(out, ref, dtype):
    # P (relative 2^-11 or 2^-8 each) and the output (the same) rounded once, a
    # normalised q on the other side of a tie here and there: the tolerances
    # that the block-sparse kernel has for outputs of order one.
    err = (out.float() - ref).abs()
    mx, mean = (2e-3, 2e-4) if dtype == torch.float16 else (1.6e-2, 2e-3)
    big = ref.abs().max().clamp(min=1.0)
    assert err.max() <= mx * big and err.mean() <= mean * big, (err.max().item(), err.mean().item())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("lens", LENGTHS)
@pytest.mark.parametrize("N", [1, 127, 128, 200, 576])
def test_matches_reference(device, dtype, D, lens, N):
    H = 3
    q, kv, w = _inputs(device, dtype, lens, N, H, D, seed=N + sum(lens), gap=5)
    k, v = kv[:, 0].transpose(0, 1), kv[:, 1].transpose(0, 1)
    scale = D ** -0.5
    buf = torch.full((len(lens), N + 2, H, D), 7.0, dtype=dtype, device=device)
    text_attention(q.transpose(1, 2), k, v, lens, w, 1e-6, scale, buf[:, 1:-1].transpose(1, 2))
    _check(buf[:, 1:-1], _reference(q, k, v, w, lens, scale), dtype)
    assert (buf[:, 0] == 7).all() and (buf[:, -1] == 7).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_offset_far_below_later_keys(device, dtype):
    """The first 32 keys score far below a later one: the second walk."""
    lens, N, H, D = (100, 40), 200, 2, 128
    q, kv, w = _inputs(device, dtype, lens, N, H, D, seed=3)
    k, v = kv[:, 0].transpose(0, 1).clone(), kv[:, 1].transpose(0, 1)
    k[:, 70] *= 8
    k[:, 139] *= 8
    out = torch.empty_like(q)
    text_attention(q.transpose(1, 2), k, v, lens, w, 1e-6, D ** -0.5, out.transpose(1, 2))
    _check(out, _reference(q, k, v, w, lens, D ** -0.5), dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("lens", [(31,), (32,), (33,), (40, 5), (64, 128)])
def test_zero_scale_gives_the_mean_of_v(device, dtype, D, lens):
    q, kv, w = _inputs(device, dtype, lens, 130, 2, D, seed=7)
    k, v = kv[:, 0].transpose(0, 1), kv[:, 1].transpose(0, 1)
    out = torch.empty_like(q)
    text_attention(q.transpose(1, 2), k, v, lens, w, 1e-6, 0.0, out.transpose(1, 2))
    _check(out, _reference(q, k, v, w, lens, 0.0), dtype)


@pytest.mark.parametrize("lens", [(40,), (32,), (5, 70)])
def test_scores_of_any_finite_size(device, lens):
    """Every score near 1e31 or -1e31 (bf16 reaches it), all alike: the mean of v.
    A row whose scores are all -inf has no softmax: NaN, as torch gives."""
    N, H, D = 64, 1, 64
    q, kv, _ = _inputs(device, torch.bfloat16, lens, N, H, D, seed=8)
    q = torch.ones_like(q)
    w = torch.ones(D, dtype=torch.bfloat16, device=device)
    v = kv[:, 1].transpose(0, 1)
    for value in (-1e30, 1e30, -1e10, float("-inf")):
        k = torch.full_like(kv[:, 0], value).transpose(0, 1)
        out = torch.empty_like(q)
        text_attention(q.transpose(1, 2), k, v, lens, w, 1e-6, D ** -0.5, out.transpose(1, 2))
        if math.isfinite(value):
            _check(out, _reference(q, torch.zeros_like(k), v, w, lens, 1.0), torch.bfloat16)
        else:
            assert out.isnan().all()


def test_non_finite_values(device):
    """Infinite scores and values act as in a softmax, and the text of the next
    item, which the last tile of an item reaches, never does."""
    lens, N, H, D = (40, 5), 64, 1, 128
    q, kv, w = _inputs(device, torch.float16, lens, N, H, D, seed=4)
    k, v = kv[:, 0].transpose(0, 1).clone(), kv[:, 1].transpose(0, 1).clone()
    v[0, 40:] = float("nan")           # item 1 only
    v[0, 39, 3] = float("inf")         # the last key of item 0
    out = torch.empty_like(q)
    text_attention(q.transpose(1, 2), k, v, lens, w, 1e-6, D ** -0.5, out.transpose(1, 2))
    assert torch.isnan(out[1]).all()
    assert (out[0, ..., 3] == float("inf")).all()
    ref = _reference(q, k, v.nan_to_num(0.0, 0.0), w, lens, D ** -0.5)
    rest = [d for d in range(D) if d != 3]
    _check(out[0][..., rest], ref[0][..., rest], torch.float16)


@pytest.mark.parametrize("N", [100, 192])
@pytest.mark.parametrize("text", [(50, 9), (64, 128)])
def test_layer_routes_agree(device, calls, N, text):
    """The layer with the kernel, with torch's operations, and with a gradient
    wanted (which torch's operations give)."""
    kernel = calls(dit_block, "text_attention")
    m = MultiHeadCrossAttention(256, 2, dtype=torch.float16, device=device)
    x = torch.randn(2, N, 256, device=device, dtype=torch.float16)
    y = torch.randn(1, sum(text), 256, device=device, dtype=torch.float16)
    with torch.no_grad():
        fused = m(x, y, text)
        assert len(kernel) == 1
        m.fused = False
        plain = m(x, y, text)
        m.fused = True
    assert len(kernel) == 1
    _check(fused, plain.float(), torch.float16)
    if N % 64 or any(n % 64 for n in text):
        x.requires_grad_()
        out = m(x, y, text)
        assert torch.equal(out, plain)
        out.sum().backward()
        assert x.grad is not None and len(kernel) == 1


@pytest.mark.parametrize("text", [(31, 33), (50, 9), (64, 128)])
@pytest.mark.parametrize("scale", [0.0, -0.1])
def test_layer_takes_any_scale(device, text, scale):
    m = MultiHeadCrossAttention(256, 2, dtype=torch.float16, device=device)
    m.scale = scale
    x = torch.randn(2, 128, 256, device=device, dtype=torch.float16)
    y = torch.randn(1, sum(text), 256, device=device, dtype=torch.float16)
    with torch.no_grad():
        got = m(x, y, text)
        m.fused = False
        _check(got, m(x, y, text).float(), torch.float16)


@pytest.mark.parametrize("part", ["q_linear", "kv_linear"])
@pytest.mark.parametrize("pad", [4, 8])
def test_layer_takes_projections_with_any_row_stride(device, part, pad):
    class Padded(torch.nn.Module):
        def __init__(self, linear):
            super().__init__()
            self.linear = linear

        def forward(self, x):
            return torch.nn.functional.pad(self.linear(x), (0, pad))[..., :-pad]

    m = MultiHeadCrossAttention(256, 2, dtype=torch.float16, device=device)
    setattr(m, part, Padded(getattr(m, part)))
    x = torch.randn(2, 100, 256, device=device, dtype=torch.float16)
    y = torch.randn(1, 59, 256, device=device, dtype=torch.float16)
    with torch.no_grad():
        got = m(x, y, (50, 9))
        m.fused = False
        _check(got, m(x, y, (50, 9)).float(), torch.float16)


@pytest.mark.parametrize("what", NORM_CHANGES)
def test_layer_runs_its_norms_as_modules(device, what):
    """Hooks on the norms fire and another norm counts, as in torch's sequence."""
    m = MultiHeadCrossAttention(256, 2, dtype=torch.float16, device=device)
    x = torch.randn(1, 100, 256, device=device, dtype=torch.float16)
    y = torch.randn(1, 50, 256, device=device, dtype=torch.float16)
    with torch.no_grad(), changed_norms(what, m):
        got = m(x, y, (50,))
        m.fused = False
        assert torch.equal(got, m(x, y, (50,)))


@pytest.mark.parametrize("cond_only", [False, True])
def test_layer_without_queries(device, cond_only):
    """No token, or conditioning tokens alone, over ragged text."""
    m = MultiHeadCrossAttention(256, 2, dtype=torch.float16, device=device)
    x = torch.randn(2, 100 if cond_only else 0, 256, device=device, dtype=torch.float16)
    y = torch.randn(1, 59, 256, device=device, dtype=torch.float16)
    with torch.no_grad():
        out = m(x, y, (50, 9), num_cond_latents=4 if cond_only else None, shape=(4, 5, 5) if cond_only else None)
    assert out.shape == x.shape and (out == 0).all()


def test_refused(device):
    q, kv, w = _inputs(device, torch.float16, (8, 8), 64, 2, 64, seed=1)
    k, v = kv[:, 0].transpose(0, 1), kv[:, 1].transpose(0, 1)
    out = torch.empty_like(q).transpose(1, 2)
    for lens in [(8, 9), (0, 8), (8,), (16, -1)]:
        with pytest.raises(ValueError):
            text_attention(q.transpose(1, 2), k, v, lens, w, 1e-6, 0.125, out)


def test_tensors_on_the_host_are_refused(device):
    q, kv, w = _inputs(device, torch.float16, (8, 8), 64, 2, 64, seed=1)
    k, v = kv[:, 0].transpose(0, 1), kv[:, 1].transpose(0, 1)
    with pytest.raises(BSADeviceError):
        text_attention(q.transpose(1, 2), k, v, (8, 8), w.cpu(), 1e-6, 0.125, torch.empty_like(q).transpose(1, 2))
    for kw in (dict(weight=w.cpu()), dict(weight=w, out=torch.empty(2, 2, 64, 64, dtype=torch.float16))):
        with pytest.raises(BSADeviceError):
            head_rms_norm(q.transpose(1, 2), **kw)
