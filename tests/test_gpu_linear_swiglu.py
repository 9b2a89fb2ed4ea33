"""linear -> swiglu in one launch: against float64 at the edges of its 64-row, 32-column blocks, and the same
values of the linear as the two operators."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,hidden,bias", [(480, 256, 512, False), (1921, 256, 353, True), (2500, 136, 97, True),
                                             (64, 1032, 5000, False), (30000, 256, 1, True), (129, 256, 3104, True), (7680, 256, 512, True), (8100, 292, 505, False)])
def test_linear_swiglu_vs_float64(dev, M, K, hidden, bias):
    from montlok import _C

    g = torch.Generator(device="cpu").manual_seed(M + K + hidden)
    x = torch.randn(M, K, generator=g).to(dev)
    w = (torch.randn(2 * hidden, K, generator=g) / K ** 0.5).to(dev)
    b = torch.randn(2 * hidden, generator=g).to(dev) if bias else None
    out = _C._ops().linear_swiglu(x, w, b)
    assert out is not None, "the shape has the fused form"
    wide = _C.linear(x, w, b)
    assert (wide[:, :hidden].double() - x.double() @ w[:hidden].double().t() - (b[:hidden].double() if bias else 0)).abs().max() < 1e-5
    gate, up = wide.double().chunk(2, dim=-1)
    ref = gate * torch.sigmoid(gate) * up
    # One rounding of the fp64 product, and the last bits of exp and of the quotient in fp64.
    assert bool(((out.double() - ref).abs() <= 2.0 ** -24 * (1 + 1e-6) * ref.abs() + 1e-45).all())


@pytest.mark.parametrize("M,hidden", [(2000, 700), (600, 350), (7680, 512)])
def test_linear_swiglu_infinities(dev, M, hidden):
    """In 64 x 64 blocks, with two waves a tile, and in 128 x 128 blocks."""
    from montlok import _C

    x = torch.randn(M, 256, generator=torch.Generator().manual_seed(3)).to(dev)
    w = torch.randn(2 * hidden, 256, generator=torch.Generator().manual_seed(4)).to(dev)
    x[70, 3], x[M // 2 - 100, 7], x[M - 1] = float("inf"), float("nan"), 1e-37
    w[hidden + 3] *= 2.0 ** 30
    out = _C._ops().linear_swiglu(x, w, None)
    expect = _C.swiglu(_C.linear(x, w))
    assert torch.equal(torch.isnan(out), torch.isnan(expect)) and torch.equal(torch.isinf(out), torch.isinf(expect))
    assert torch.equal(out[~torch.isnan(out)], expect[~torch.isnan(expect)])


def test_other_shapes_run_the_two_operators(dev):
    from montlok import _C

    x, w = torch.randn(100, 64, device=dev), torch.randn(48, 64, device=dev)
    assert _C._ops().linear_swiglu(x, w, None) is None
    down = torch.randn(8, 24, device=dev)
    assert torch.equal(_C.swiglu_mlp(x, w, None, down), _C.linear(_C.swiglu(_C.linear(x, w)), down))
    with pytest.raises(RuntimeError, match="must end in an even dimension"):
        _C.swiglu_mlp(x, w[:47], None, down)
