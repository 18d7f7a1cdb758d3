"""AdaLN modulation kernel against 64 bits, and the block's two routes to it."""

from __future__ import annotations

import pytest
import torch

from lcv_bsa import dit_block
from lcv_bsa.block_ops import adaln_modulation
from lcv_bsa.dit_block import LongCatSingleStreamBlock

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K", [8, 504, 512, 520, 1024])
@pytest.mark.parametrize("B,T,C,chunks", [(1, 1, 8, 1), (1, 7, 64, 6), (2, 4, 136, 6), (1, 9, 256, 2), (3, 11, 4096, 6)])
def test_matches_64_bits(device, dtype, K, B, T, C, chunks):
    g = torch.Generator(device="cpu").manual_seed(K + C)
    t = (2 * torch.randn(B, T, K, generator=g)).to(device)
    w = torch.randn(chunks * C, K, generator=g).to(device, dtype)
    b = torch.randn(chunks * C, generator=g).to(device, dtype)
    out = adaln_modulation(t, w, b, chunks)
    s = torch.nn.functional.silu(t.double()).reshape(-1, K)
    want = s @ w.double().T + b.double()
    size = s.abs() @ w.double().abs().T + b.double().abs()
    shape = (B * T, chunks, C)
    err = (out.reshape(chunks, B * T, C).transpose(0, 1).double() - want.reshape(shape)).abs()
    # A sum passes at most 16 + 7 additions and silu 4 roundings, each 2^-24 of
    # the summed magnitudes: below 2e-6 of them.
    assert (err <= 2e-6 * size.reshape(shape)).all(), (err / size.reshape(shape)).max().item()


@pytest.mark.parametrize("K", [64, 512, 36])
def test_block_modulation_routes_agree(device, calls, K):
    """Kernel and torch (K = 36 takes torch's on both sides)."""
    kernel = calls(dit_block, "adaln_modulation")
    blk = LongCatSingleStreamBlock(256, 2, 4, K, dtype=torch.float16, device=device)
    t = torch.randn(2, 5, K, device=device)
    with torch.no_grad():
        for got, want in zip(blk._modulation(t, True), blk._modulation(t, False), strict=True):
            assert got.shape == want.shape == (2, 5, 1, 256) and got.dtype == torch.float32
            assert torch.allclose(got, want, rtol=1e-5, atol=2e-6)
    assert len(kernel) == (K != 36)


def test_a_weight_that_stands_for_others(device):
    """A tensor subclass says itself what its values are: only torch asks it."""
    class Doubled(torch.Tensor):
        def float(self):
            return 2 * self.as_subclass(torch.Tensor).float()

    blk = LongCatSingleStreamBlock(256, 2, 4, 64, dtype=torch.float16, device=device)
    lin = blk.adaLN_modulation[1]
    t = torch.randn(2, 5, 64, device=device)
    with torch.no_grad():
        for name in ("weight", "bias"):
            doubled = getattr(lin, name).detach().as_subclass(Doubled)
            delattr(lin, name)
            setattr(lin, name, doubled)
            for got, want in zip(blk._modulation(t, True), blk._modulation(t, False), strict=True):
                assert torch.allclose(got, want, rtol=1e-5, atol=2e-6)


@pytest.mark.parametrize("B,T,K", [(1, 8 * 65535 + 1, 8), (2, 0, 64), (0, 3, 64), (1, 2, 0)])
def test_sizes_beyond_the_kernel_go_through_torch(device, B, T, K):
    blk = LongCatSingleStreamBlock(8, 1, 4, K, dtype=torch.float16, device=device)
    t = torch.randn(B, T, K, device=device)
    with torch.no_grad():
        for got, want in zip(blk._modulation(t, True), blk._modulation(t, False), strict=True):
            assert got.shape == (B, T, 1, 8) and torch.equal(got, want)
