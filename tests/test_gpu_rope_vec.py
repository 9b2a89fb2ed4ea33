"""RoPE and key assembly four lanes at a time: the one-lane kernel bit for bit (which unaligned operands still take)."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,L,Lq,H,hd,nope", [(2, 33, 33, 4, 64, 32), (3, 7, 1, 2, 32, 16), (1, 1, 1, 1, 8, 0), (2, 50, 9, 3, 48, 40),
                                              (5, 129, 129, 8, 32, 16)])
def test_vector_rope_equals_scalar(dev, B, L, Lq, H, hd, nope):
    from montlok import _C

    g = torch.Generator().manual_seed(B * L + hd)
    rope = hd - nope
    q = torch.randn(B, Lq, H, hd, generator=g).to(dev)
    kv = torch.randn(B, L, H, nope + hd, generator=g).to(dev)
    wide = torch.randn(B, L, rope + 8, generator=g).to(dev)
    wide1 = torch.empty(B * L * (rope + 8) + 1, device=dev)[1:].view(B, L, rope + 8).copy_(wide)  # 4 bytes off
    cos, sin = torch.randn(2, L, rope, generator=g).to(dev)
    qv, qs = q.clone(), q.clone()
    kv_vec = _C.mla_rope_qk(qv, kv, wide[..., 4:4 + rope], cos, sin, nope)
    kv_one = _C.mla_rope_qk(qs, kv, wide1[..., 4:4 + rope], cos, sin, nope)
    assert torch.equal(kv_vec, kv_one) and torch.equal(qv, qs)
    assert not torch.equal(qv, q)
