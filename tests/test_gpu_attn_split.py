"""fp32 attention with the keys split over four waves (attn_split_kernel) at the edges of its tiles, chunks and rule,
and the one-launch MLA beyond 256 rows."""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch

import bf16_emu as emu
from helpers import BF16_TOL, assert_close, assert_emulated
from test_gpu_mla import _mla_params, _oracle_mla, _t, rope_tables

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
    """A score of -inf (no weight), of +inf (inf - inf: NaN) and a NaN key: as softmax has them, in the rows that see
    the key and in no others."""
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
    k[0, 90, 0, 5] = float("inf")
    out = _C.attention(q, k, v, _C.MASK_CAUSAL_TOP_LEFT, 0.125)
    assert torch.isfinite(out[:, :90, 0]).all() and torch.isnan(out[:, 90:, 0]).all()


@pytest.mark.parametrize("B,L,bias", [(4, 257, True), (5, 480, False), (8, 512, True), (4, 320, True)])
def test_one_launch_mla_beyond_256_rows(dev, oracle, B, L, bias):
    from montlok import _C

    H, hd, nope, kvr = 4, 64, 32, 64
    d = H * hd
    rng = np.random.default_rng(B + L)
    x = rng.standard_normal((B, L, d)).astype(np.float32)
    p = _mla_params(rng, d, H, hd, nope, kvr, True)
    if not bias:
        p["ln_b"] = np.zeros_like(p["ln_b"])
    cos, sin = rope_tables(L, hd - nope)
    bw = lambda a: _t(a, dev).to(torch.bfloat16)  # noqa: E731
    in_w = np.concatenate([p["q"], p["kv_down"], p["k_rope"]])
    args = (_t(x, dev), bw(in_w), torch.empty(0, device=dev), _t(p["ln_w"], dev), _t(p["ln_b"], dev) if bias else None, 1e-5,
            bw(p["kv_up"]), bw(p["o"]), _t(cos, dev), _t(sin, dev), H, hd, nope, kvr, L, True, hd ** -0.5)
    out = _C._mla_forward(*args, allow_fused=True)
    assert _C.mla_forward_launches() == ["mla_forward"]
    emulated = emu.mla_forward(x, p["q"], p["kv_down"], p["k_rope"], p["ln_w"], p["ln_b"], 1e-5, p["kv_up"], p["o"],
                               cos, sin, H, hd, nope, hd ** -0.5)
    assert_emulated(out, emulated, name=f"one-launch MLA {B}x{L} vs the bf16 emulation")
    assert_close(out, _oracle_mla(oracle, x, p, H, hd, nope, kvr, L, True, hd ** -0.5, cos, sin), tol=BF16_TOL, name="vs oracle")
    _C._mla_forward(args[0][:3], *args[1:], allow_fused=True)
    assert _C.mla_forward_launches() == ["separate"], "few long windows run the separate operators"
