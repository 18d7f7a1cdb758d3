"""The fp32 attention kernel (split-bf16 MFMA), against 64-bit attention and the
vector-ALU kernel.  Rows that do not start on 16-byte boundaries take the
vector-ALU kernel, so the same values from a buffer one element off give its
result."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from lcv_bsa import bsa_attention_hip
from oracle import bsa_oracle as O

pytestmark = pytest.mark.gpu


def _unaligned(t):
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    out = buf[1:].view(t.shape)
    out.copy_(t)
    return out


def _exact(q, k, v, idx, qtok, ktok, scale):
    """64-bit attention of each q-block over its listed blocks, on the CPU."""
    q, k, v = (t.double().cpu() for t in (q, k, v))
    out = torch.zeros_like(q)
    for b in range(q.shape[0]):
        for h in range(q.shape[1]):
            for n in range(len(qtok)):
                keys = torch.cat([ktok[i] for i in idx[b, h, n].tolist() if 0 <= i < len(ktok)])
                p = torch.softmax(q[b, h, qtok[n]] @ k[b, h, keys].T * scale, -1)
                out[b, h, qtok[n]] = p @ v[b, h, keys]
    return out


def _tokens(shape, chunk):
    blocks = torch.from_numpy(np.asarray(O.build_token_block_indices(shape, chunk)))
    return [torch.nonzero(blocks == n).flatten() for n in range(int(blocks.max()) + 1)]


def _inputs(device, H, D, S, Sk, nq, nk, top_k, seed=0, k_scale=1.0):
    g = torch.Generator(device="cpu").manual_seed(seed)
    q, k, v = (torch.randn(1, H, n, D, generator=g).to(device) for n in (S, Sk, Sk))
    idx = torch.stack([torch.randperm(nk, generator=g)[:top_k].sort().values for _ in range(H * nq)])
    return q, k * k_scale, v, idx.view(1, H, nq, top_k).to(torch.int32).to(device)


# One block, an odd list, a list over 64 entries, voxels whose halves are not
# contiguous (both halves of a block 32 rows apart in every axis), keys on a
# larger grid than the queries.
CASES = [
    ((1, 1, 64), (1, 1, 64), None, 1),
    ((1, 1, 448), (1, 1, 64), None, 5),
    ((1, 1, 4480), (1, 1, 64), None, 67),
    ((4, 8, 12), (4, 4, 4), None, 3),
    ((4, 32, 2), (2, 32, 1), None, 2),
    ((2, 8, 16), (1, 4, 16), (6, 8, 16), 7),
]


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("shape,chunk,kv_shape,top_k", CASES)
def test_error_no_larger_than_the_vector_alu(device, D, shape, chunk, kv_shape, top_k):
    kv = kv_shape or shape
    qtok, ktok = _tokens(shape, chunk), _tokens(kv, chunk)
    S, Sk = int(np.prod(shape)), int(np.prod(kv))
    q, k, v, idx = _inputs(device, 2, D, S, Sk, len(qtok), len(ktok), top_k, seed=D + S, k_scale=2.0)
    kw = dict(chunk_thw=chunk, shape=shape, kv_shape=kv_shape)
    got = bsa_attention_hip(q, k, v, idx, **kw).double().cpu()
    valu = bsa_attention_hip(_unaligned(q), _unaligned(k), _unaligned(v), idx, **kw).double().cpu()
    ref = _exact(q, k, v, idx, qtok, ktok, D ** -0.5)
    err, err_valu = ((x - ref).norm() / ref.norm() for x in (got, valu))
    # Scores up to ~10 in size carry a few fp32 roundings (2^-24 each) into the
    # exponent; the split adds below one more.  A quarter covers small samples.
    assert err <= 2e-6 and err <= 1.25 * err_valu, (float(err), float(err_valu))
    assert torch.equal(got, bsa_attention_hip(q, k, v, idx, **kw).double().cpu())
    assert not torch.equal(got, valu)  # two kernels


def test_strided_rows_negative_scale_and_skipped_entries(device):
    D, S = 128, 640
    q, k, v, idx = _inputs(device, 3, D, S, S, 10, 10, 4, seed=5)
    idx[0, 1, 3] = torch.tensor([-1, 2, 10, 1 << 20], dtype=torch.int32)
    idx[0, 2, 0] = -1  # nothing listed: zeros
    views = [t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v)]
    out = torch.full((1, S, 3, D + 4), 7.0, device=device)
    for scale in (D ** -0.5, -0.2):
        o = out[..., :D].transpose(1, 2)
        bsa_attention_hip(*views, idx, (1, 1, 64), (1, 1, S), scale, out=o)
        ref = bsa_attention_hip(_unaligned(q), _unaligned(k), _unaligned(v), idx, (1, 1, 64), (1, 1, S), scale)
        assert (out[..., D:] == 7.0).all() and (o[0, 2, :64] == 0).all()
        assert (o - ref).norm() <= 2e-6 * ref.norm()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("where,value", [("k", float("inf")), ("k", float("-inf")), ("k", float("nan")),
                                         ("v", float("inf")), ("v", 3.402e38), ("q", float("nan")),
                                         ("q", float("inf")), ("k", 3.402e38)])
def test_values_the_split_cannot_carry(device, D, where, value):
    """Workgroups that meet such a value give what the vector-ALU kernel gives:
    the same non-finite entries, the others to fp32 rounding."""
    S, top_k = 512, 3
    q, k, v, idx = _inputs(device, 1, D, S, S, 8, 8, top_k, seed=9)
    t = {"q": q, "k": k, "v": v}
    t[where][0, 0, 3 * 64 + 17, 5] = value
    got = bsa_attention_hip(q, k, v, idx, (1, 1, 64), (1, 1, S))
    ref = bsa_attention_hip(_unaligned(q), _unaligned(k), _unaligned(v), idx, (1, 1, 64), (1, 1, S))
    fin = torch.isfinite(ref)
    assert not fin.all() or value == 3.402e38
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got[got.isinf()], ref[ref.isinf()])
    assert torch.allclose(got[fin], ref[fin], rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("what", ["small v", "a small column of v", "subnormal v", "small q, large k",
                                  "small k, large q", "small k, large scale", "weights near underflow, large v"])
def test_values_far_from_one(device, D, what):
    """Values whose bf16 pieces reach the subnormal range keep every bit that the
    vector-ALU kernel keeps.  Each small value is made of 24 significant bits."""
    S, top_k = 512, 3
    q, k, v, idx = _inputs(device, 1, D, S, S, 8, 8, top_k, seed=11)
    scale = D ** -0.5
    if what == "small v":
        v = v * 2.0 ** -118
    elif what == "a small column of v":
        v[..., 7] *= 2.0 ** -120
    elif what == "subnormal v":
        v = v * 2.0 ** -100 * 2.0 ** -30
    elif what == "small q, large k":
        q, k = q * 2.0 ** -116, k * 2.0 ** 116
    elif what == "small k, large q":
        q, k = q * 2.0 ** 118, k * 2.0 ** -118
    elif what == "small k, large scale":
        k, scale = k * 2.0 ** -118, scale * 2.0 ** 118
    else:  # exp2 of about -117 against values of 2^115
        q.zero_()
        q[..., 0] = 1.0
        k[..., 0] = torch.where(torch.arange(S, device=device) % 64 == 5, -81.0, 0.0)
        v = v * torch.where(torch.arange(S, device=device) % 64 == 5, 2.0 ** 115, 2.0 ** -6)[:, None]
        scale = 1.0
    kw = dict(chunk_thw=(1, 1, 64), shape=(1, 1, S), sm_scale=scale)
    got = bsa_attention_hip(q, k, v, idx, **kw).double().cpu()
    valu = bsa_attention_hip(_unaligned(q), _unaligned(k), _unaligned(v), idx, **kw).double().cpu()
    tok = _tokens((1, 1, S), (1, 1, 64))
    ref = _exact(q, k, v, idx, tok, tok, scale)
    # Column by column: a small one counts as much as the others.
    err, err_valu = ((x - ref).norm(dim=-2) / ref.norm(dim=-2) for x in (got, valu))
    assert (err <= torch.clamp(1.25 * err_valu, min=2e-6)).all(), ((err / err_valu).max(), err.max())
