"""Row kernels at the row widths where their chunking changes, and the SwiGLU
gate on every half-precision value."""

from __future__ import annotations

import pytest
import torch

from lcv_bsa.block_ops import residual_norm, swiglu

pytestmark = pytest.mark.gpu

HALF_ULP = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("C", [8, 504, 512, 520, 1024, 1032, 2048, 2056, 4096, 4104, 8192])
@pytest.mark.parametrize("mode", ["plain", "add", "gated"])
@pytest.mark.parametrize("norm", ["affine", "modulated", "none"])
def test_residual_norm(device, dtype, C, mode, norm):
    if mode == "plain" and norm == "none":
        pytest.skip("nothing to compute")
    g = torch.Generator(device="cpu").manual_seed(C)
    B, T, per = 2, 3, 3  # 18 rows: a last workgroup of two
    x, a = (torch.randn(B, T * per, C, generator=g).to(device, dtype) for _ in range(2))
    gate, shift, scale = (torch.randn(B, T, C, generator=g).to(device) for _ in range(3))
    w, b = ((1 + torch.randn(C, generator=g)).to(device, dtype) for _ in range(2))
    kw = {"affine": dict(weight=w, bias=b), "modulated": dict(shift=shift, scale=scale), "none": dict(norm=False)}[norm]
    args = {"plain": (), "add": (a,), "gated": (a, gate)}[mode]
    r, n = residual_norm(x, *args, frames=T, eps=1e-6, **kw)
    rows = lambda t: t.repeat_interleave(per, 1)  # noqa: E731
    want = x if mode == "plain" else (x.float() + (rows(gate) * a.float() if mode == "gated" else a.float())).to(dtype)
    assert torch.equal(r, want)
    if norm == "none":
        assert n is None
        return
    d = want.double()
    y = (d - d.mean(-1, keepdim=True)) * torch.rsqrt(d.var(-1, unbiased=False, keepdim=True) + 1e-6)
    mul, add = (w.double(), b.double()) if norm == "affine" else (rows(scale).double() + 1, rows(shift).double())
    ref = y * mul + add
    # One rounding to the dtype; fp32 sums over C values and four fp32 operations
    # before it, below 2^-20 of the terms.
    size = (y * mul).abs() + add.abs() + mul.abs()
    assert ((n.double() - ref).abs() <= 1.001 * HALF_ULP[dtype] * ref.abs() + 2.0 ** -20 * size + 2.0 ** -25).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("reverse", [False, True])
def test_swiglu_on_every_value(device, dtype, reverse):
    """All 65,536 bit patterns (in order and reversed, so that near and far
    values share waves differently): torch's silu, bit for bit."""
    x = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).to(device).view(dtype)
    if reverse:
        x = x.view(256, 256).t().contiguous().view(-1)
    for hidden in (8, 24, 4096):
        rows = -(-len(x) // hidden)
        a = torch.zeros(rows * hidden, dtype=dtype, device=device)
        a[:len(x)] = x
        a = a.view(rows, hidden)
        for gate in (1.0, -2.5):
            b = torch.full_like(a, gate)
            want = torch.nn.functional.silu(a) * b
            got = swiglu(torch.cat([a, b], -1))
            assert torch.equal(got.isnan(), want.isnan())
            assert torch.equal(got.nan_to_num(0.0).view(torch.int16), want.nan_to_num(0.0).view(torch.int16))
