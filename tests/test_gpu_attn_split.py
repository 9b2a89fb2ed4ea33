"""fp32 attention with the keys split over four waves (attn_split_kernel) at the edges of its tiles, chunks and rule."""

from __future__ import annotations

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Lq,Lk,H,hd,mask", [(1, 1, 1, 1, 64, 1), (2, 1, 480, 4, 64, 0), (1, 33, 33, 2, 32, 1),
                                               (3, 17, 129, 2, 64, 2), (2, 32, 31, 3, 64, 0), (1, 480, 480, 4, 64, 1),
                                               (20, 481, 481, 8, 32, 1), (70, 193, 193, 4, 64, 1), (1, 5, 700, 2, 32, 2),
                                               (9, 130, 257, 4, 32, 2)])
@pytest.mark.parametrize("scale", [None, -0.2])
def test_split_attention_vs_float64(dev, B, Lq, Lk, H, hd, mask, scale):
    from montlok import _C

    g = torch.Generator().manual_seed(B + Lq + Lk + hd)
    q, k = torch.randn(B, Lq, H, hd, generator=g).to(dev), torch.randn(B, Lk, H, hd, generator=g).to(dev)
    kv = torch.randn(B, Lk, H, hd + 16, generator=g).to(dev)
    v = kv[..., 16:]
    scale = hd ** -0.5 if scale is None else scale
    out = _C.attention(q, k, v, mask, scale)
    s = torch.einsum("bihd,bjhd->bhij", q.double().cpu(), k.double().cpu()) * scale
    i, j = torch.arange(Lq)[:, None], torch.arange(Lk)[None]
    allowed = {0: torch.ones(Lq, Lk, dtype=torch.bool), 1: j <= i, 2: j <= i + Lk - Lq}[mask]
    p = torch.softmax(s.masked_fill(~allowed, -math.inf), -1)
    ref = torch.einsum("bhij,bjhd->bihd", p, v.double().cpu())
    # Scores of |q| |k| sqrt(hd) eps, so weights relative to that; sums of Lk products of weights that add up to one.
    bound = 2.0 ** -24 * (8 * abs(scale) * math.sqrt(hd) * 6 * 6 + Lk / 16 + 16) * v.abs().max().item()
    assert (out.cpu().double() - ref).abs().max().item() <= bound


def test_split_attention_special_values(dev):
    """A score of +-inf and a NaN key: as softmax has them, in the rows that see the key and in no others."""
    from montlok import _C

    q = torch.ones(1, 200, 2, 64, device=dev)
    k = torch.zeros(1, 200, 2, 64, device=dev)
    v = torch.randn(1, 200, 2, 64, generator=torch.Generator().manual_seed(1)).to(dev)
    k[0, 70, 0, 3] = -float("inf")
    k[0, 150, 1, 3] = float("nan")
    out = _C.attention(q, k, v, _C.MASK_CAUSAL_TOP_LEFT, 0.125)
    assert torch.isfinite(out[:, :, 0]).all() and torch.isfinite(out[:, :150, 1]).all()
    assert torch.isnan(out[:, 150:, 1]).all()
    keep = [j for j in range(200) if j != 70]
    assert torch.allclose(out[0, 199, 0], v[0, keep, 0].mean(0), atol=1e-6)
