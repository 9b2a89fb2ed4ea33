"""The fp32-weight linear on three bf16 planes (linear_split.hip) and the four-waves-per-tile form for few tiles
(linear_small_split_kernel): edges of their tiles and of the rules that choose them, against float64."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _operands(dev, M, K, N, seed, wdt="f32", pad=0):
    g = torch.Generator(device="cpu").manual_seed(seed)
    x = torch.randn(M, K + pad, generator=g).to(dev)[:, :K]
    w = (torch.randn(N, K, generator=g) / K ** 0.5).to(dev)
    b, r = torch.randn(N, generator=g).to(dev), torch.randn(M, N, generator=g).to(dev)
    return x, w.bfloat16() if wdt == "bf16" else w, b, r


def _assert_bound(got, x, w, terms, extra=0.0):
    """|y - x W^T| <= c 2^-24 sum |x| |w|: c counts the fp32 roundings a sum meets (one per `terms` products and
    the few that join partial sums, bias and residual) and, for the three planes, the dropped 2^-26 terms."""
    xd, wd = x.double(), w.double()
    K = x.shape[1]
    slack = (K / terms + 8) * 2.0 ** -24 * (xd.abs() @ wd.abs().t() + extra) + 2.0 ** -148  # (subnormal results)
    off = (got.double() - xd @ wd.t()).abs() - slack
    assert bool((off <= 0).all()), f"{off.max().item():.3e} over the bound"


# (rows, K, N, x row padding): one past a block, K not a multiple of the 32-wide step or of 8, ragged and tiny N, the
# first shapes past the one-wave rule's 1536 tiles, K just above 128, one row against many columns; then calls that
# fill rounds of 128 x 128 blocks, with ragged last rows and columns, K not a multiple of the step, one and two steps;
# then 256 blocks of 64 x 64, the last of two waves a tile, and one row more; K = 128 on both
# sides of its 3072 blocks; K from 64 to 127 that is no multiple of 8, which has no one-wave form, on few rows.
SPLIT = [(1921, 256, 352, 0), (2049, 136, 200, 4), (1600, 132, 257, 0), (30000, 256, 1, 8), (64, 2048, 5200, 0),
         (1, 256, 24592, 0), (12304, 160, 30, 0), (1537, 256, 256, 12),
         (15360, 512, 256, 0), (16371, 260, 255, 4), (3840, 136, 1024, 0), (32700, 132, 256, 0), (65536, 544, 120, 0),
         (4096, 148, 256, 0), (4097, 148, 256, 0), (6001, 128, 667, 4), (65537, 128, 130, 0), (1, 68, 30, 0), (16, 100, 257, 0), (130, 124, 64, 8)]


@pytest.mark.parametrize("M,K,N,pad", SPLIT)
def test_split_linear_vs_float64(dev, M, K, N, pad):
    from montlok import _C

    x, w, b, r = _operands(dev, M, K, N, M + K + N, pad=pad)
    y = _C.linear(x, w)
    _assert_bound(y, x, w, 16)
    assert torch.equal(_C.linear(x, w, b), y + b)
    assert torch.equal(_C.linear_residual(x, w, b, r), r + (y + b))


@pytest.mark.parametrize("M,K,N", [(1, 264, 16), (480, 512, 256), (77, 1000, 33), (1280 * 16, 520, 9), (17, 1024, 300)])
@pytest.mark.parametrize("wdt", ["f32", "bf16"])
def test_four_waves_per_tile_vs_float64(dev, M, K, N, wdt):
    from montlok import _C

    x, w, b, r = _operands(dev, M, K, N, M + K + N, wdt)
    y = _C.linear(x, w)
    _assert_bound(y, x.bfloat16() if wdt == "bf16" else x, w, 2)
    assert torch.equal(_C.linear(x, w, b), y + b)
    assert torch.equal(_C.linear_residual(x, w, b, r), r + (y + b))


@pytest.mark.parametrize("M,K,N,groups", [(1921, 256, 352, 32), (1921, 256, 352, 16), (2500, 256, 300, 8),
                                          (3001, 256, 270, 4), (2100, 160, 260, 20), (1930, 192, 350, 3), (3300, 256, 300, 16),
                                          (7000, 128, 300, 16), (33000, 128, 24, 8), (65536, 128, 200, 4),
                                          (16384, 128, 256, 16), (16371, 128, 255, 8)])
def test_rms_norm_split_linear_equals_the_two_operators(dev, M, K, N, groups):
    """One launch, and the two operators bit for bit, also where linear takes 128 x 128 blocks (the last two shapes) and
    the norm's form 64 x 64 ones."""
    from montlok import _C
    from montlok._C import _load

    x, w, b, _ = _operands(dev, M, K, N, M + groups)
    x = 3 * x
    nw = torch.rand(K, generator=torch.Generator().manual_seed(1)).to(dev) + 0.5
    out = torch.empty(M, N, device=dev)
    status = _load().mlk_rms_norm_linear(x.data_ptr(), M, K, K, nw.data_ptr(), 1e-5, groups, w.data_ptr(), 0,
                                         b.data_ptr(), N, out.data_ptr(), N, torch.cuda.current_stream().cuda_stream)
    assert status == 0
    assert torch.equal(out, _C.linear(_C.rms_norm(x, nw, 1e-5, groups), w, b))


def test_split_linear_special_values(dev):
    """Infinities, NaN, values whose bf16 rounding is infinite: as the fp32 sum has them; subnormals to its bound."""
    from montlok import _C

    x, w, _, _ = _operands(dev, 2000, 256, 300, 7)
    x[3, 5], x[64, 9], x[70, 11], x[200, 200] = float("inf"), float("nan"), 3.4e38, float("-inf")
    x[300] = 1e-39
    w[7, 200], w[9, 3], w[11] = float("inf"), 0.0, 0.0
    w[11, 11] = 0.5
    y, ref = _C.linear(x, w), (x.double() @ w.double().t()).float()
    assert torch.equal(torch.isnan(y), torch.isnan(ref)) and torch.equal(torch.isinf(y), torch.isinf(ref))
    assert torch.equal(y[torch.isinf(y)], ref[torch.isinf(ref)])
    assert abs(y[70, 11].item() / 1.7e38 - 1) < 1e-6
    plain = [i for i in range(2000) if i not in (3, 64, 70, 200)]
    cols = [j for j in range(300) if j != 7]
    _assert_bound(y[plain][:, cols], x[plain], w[cols], 16)


# One shape for each form: two waves a tile, 64 x 64 blocks with a ragged step, 128 x 128 blocks.
FORMS = [(2000, 256, 300), (4000, 260, 350), (16371, 260, 255)]


@pytest.mark.parametrize("M,K,N", FORMS)
def test_split_linear_infinities_in_every_form(dev, M, K, N):
    """Results that the planes cannot form (infinite operands, operands that round to bf16 infinity) are formed again;
    the other results of their tiles, and rows with a NaN, stay as they are."""
    from montlok import _C

    x, w, b, _ = _operands(dev, M, K, N, M)
    clean = _C.linear(x, w, b)
    last = M - 1
    x[3, 5], x[40, 7], x[64, K - 1], x[70], x[last, 0] = float("inf"), float("nan"), float("-inf"), 3.4e38 / K ** 0.5, 3.4e38
    w[11], w[N - 2] = 0.0, 0.0
    w[11, 0], w[N - 2, 0] = 0.5, -0.25
    y, ref = _C.linear(x, w, b), (x.double() @ w.double().t() + b.double()).float()
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    assert torch.equal(y[torch.isinf(ref)], ref[torch.isinf(ref)])
    assert torch.isnan(y[40]).all() and torch.isinf(y[3]).any()
    assert abs(y[last, 11].item() / 1.7e38 - 1) < 1e-6 and abs(y[last, N - 2].item() / -0.85e38 - 1) < 1e-6
    rows = [i for i in range(M) if i not in (3, 40, 64, 70, last)]
    cols = [j for j in range(N) if j not in (11, N - 2)]
    assert torch.equal(y[rows][:, cols], clean[rows][:, cols])


@pytest.mark.parametrize("M,K,N", FORMS)
def test_split_linear_over_the_whole_range(dev, M, K, N):
    """Rows of x and of W from the smallest subnormals to near the largest float: the same bound, at any size whose
    absolute sum is finite. The planes of a value below 2^-110 as it stands have no exact bf16 form."""
    from montlok import _C

    x, w, _, _ = _operands(dev, M, K, N, M + 1)
    sizes = [1e-30, 1e-33, 1e-34, 1e-36, 1e-38, 1e-39, 1e-42, 1e-44, 1e10, 1e20, 1e25, 1e30, 1e34, 1e37]
    for i, size in enumerate(sizes):
        x[5 + 37 * i] *= size
        w[3 + 17 * i] *= size
    x[1500] = (1 + 2.0 ** -8 + 2.0 ** -9) * 2.0 ** 60  # rounds up to bf16: the sum of first planes is above the sum
    w[250] = 3.4e38 / K / x[1500, 0] * (1 - 2.0 ** -11)
    y, total = _C.linear(x, w), x.double().abs() @ w.double().abs().t()
    ref = x.double() @ w.double().t()
    assert 3.39e38 < ref[1500, 250] < 3.4e38
    # Operands of 2^104 or results of 2^80 take the fp32 products, two to a rounding.
    plain = (x.abs().amax(1) >= 2.0 ** 104)[:, None] | (w.abs().amax(1) >= 2.0 ** 104)[None] | (total >= 2.0 ** 80)
    slack = torch.where(plain, K / 2 + 8.0, K / 16 + 8.0).double() * 2.0 ** -24 * total + 2.0 ** -148
    held = total <= 3.4e38
    assert bool(torch.isfinite(y[held]).all()), "a finite sum became infinite"
    off = torch.where(held, (y.double() - ref).abs() - slack, torch.zeros_like(ref))
    assert bool((off <= 0).all()), f"{(off / total).max().item():.3e} of the absolute sum over the bound"


def test_norm_split_linear_infinities(dev):
    """The norm's prologue in front of results that are formed again: as the two operators."""
    from montlok import _C

    x, w, b, _ = _operands(dev, 3300, 256, 300, 5)
    nw = torch.rand(256, generator=torch.Generator().manual_seed(2)).to(dev) + 0.5
    w[5, 100], w[6, 30] = float("inf"), 3.4e38
    x[9, 4], x[100, 7] = float("nan"), float("inf")
    for groups in (4, 32):
        normed = _C.rms_norm(x, nw, 1e-5, groups)
        two, ref = _C.linear(normed, w, b), (normed.double() @ w.double().t() + b.double()).float()
        one = _C.rms_norm_linear(x, nw, 1e-5, groups, w, b)
        assert torch.equal(one[~torch.isnan(two)], two[~torch.isnan(two)]) and torch.equal(torch.isnan(one), torch.isnan(two))
        assert torch.equal(torch.isfinite(two), torch.isfinite(ref)) and torch.isfinite(two[:, 6]).sum() > 2000


def _us(fn, calls=20):
    fn()
    times = []
    for _ in range(5):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(calls):
            fn()
        b.record()
        b.synchronize()
        times.append(a.elapsed_time(b) * 1e3 / calls)
    return min(times)


@pytest.mark.parametrize("M,K,N", [(7680, 512, 256), (15360, 512, 256), (3840, 1024, 256), (15360, 256, 1192)])
@pytest.mark.parametrize("value", ["nan", "inf"])
def test_rows_of_missing_values_do_not_slow_the_call(dev, M, K, N, value):
    """One row with a NaN or an infinity, and all of them, in the time of a few calls (formed one sum after another in
    a lane they took 7 to 120 times a call's; 1.0 to 2.0 measured for NaN, up to 3.3 for infinities)."""
    from montlok import _C

    x, w, _, _ = _operands(dev, M, K, N, 1)
    plain = _us(lambda: _C.linear(x, w))
    x[M // 2, 3] = float(value)
    one = _us(lambda: _C.linear(x, w))
    x[:, 3] = float(value)
    every = _us(lambda: _C.linear(x, w))
    assert one < 5 * plain and every < 8 * plain, (plain, one, every)


@pytest.mark.parametrize("K", [100, 128, 196, 260, 1028])
def test_rows_too_far_apart_for_the_planes(dev, K):
    """A row stride of 2^23 floats and more (the last position of very long windows) takes the fp32 forms."""
    from montlok import _C

    x, w, b, r = _operands(dev, 3, K, 300, K)
    far = torch.empty(3 * 2 ** 23, device=dev).view(3, 2 ** 23)[:, :K]
    far.copy_(x)
    y = _C.linear(far, w)
    _assert_bound(y, x, w, 2)
    assert torch.equal(_C.linear(far, w, b), y + b) and torch.equal(_C.linear_residual(far, w, b, r), r + (y + b))


@pytest.mark.parametrize("M,K,N", [(100, 256, 4000), (3, 64, 40)])
def test_norm_linear_of_rows_far_apart_equals_the_two_operators(dev, M, K, N):
    """The norm leaves dense rows, so linear's form may differ from the one that x's stride would ask for."""
    from montlok import _C

    x, w, b, _ = _operands(dev, M, K, N, K)
    nw = torch.rand(K, generator=torch.Generator().manual_seed(1)).to(dev) + 0.5
    far = torch.empty(M * 2 ** 23, device=dev).view(M, 2 ** 23)[:, :K]
    far.copy_(x)
    assert torch.equal(_C.rms_norm_linear(far, nw, 1e-5, 4, w, b), _C.linear(_C.rms_norm(far, nw, 1e-5, 4), w, b))
