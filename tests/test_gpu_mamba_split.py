"""The Mamba-3 scan with its chunks in parallel (few window x head pairs): the unfused prep -> rotate -> chunked
recurrence bit for bit, at the edges of the rule that chooses it, of a chunk and of the layouts."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import assert_bitwise, assert_close
from test_gpu_mamba import _random_layer, _t

pytestmark = pytest.mark.gpu

_KEYS = ("b_bias", "c_bias", "b_norm_w", "c_norm_w", "dt_bias", "skip")


def _case(dev, B, L, N, G, H, D, R):
    proj, p = _random_layer(np.random.default_rng(B + L + N + D), B, L, N, G, H, D, R)
    return _t(proj, dev), [_t(p[k], dev) for k in _KEYS], (N, G, H, D, R, 1e-5, 1e-5, 1e-4)


@pytest.mark.parametrize("B,L,N,G,H,D,R", [(1, 97, 64, 1, 8, 64, 16), (16, 128, 64, 1, 8, 64, 17), (2, 129, 32, 2, 4, 32, 0),
                                           (3, 480, 16, 1, 4, 32, 4), (1, 500, 64, 1, 1, 64, 32), (7, 161, 16, 3, 6, 64, 8),
                                           (24, 353, 64, 1, 8, 64, 16), (5, 255, 32, 1, 5, 64, 9), (4, 130, 64, 1, 2, 32, 16)])
def test_chunk_parallel_scan_equals_unfused(dev, monkeypatch, B, L, N, G, H, D, R):
    from montlok import _C

    proj, params, geo = _case(dev, B, L, N, G, H, D, R)
    wide = torch.randn(B, L, proj.shape[-1] + 12, device=dev)
    wide[..., :proj.shape[-1]] = proj
    z = proj[..., :H * D].double()
    gate = (z * torch.sigmoid(z)).float()
    got = _C.mamba3_siso_forward(proj, None, *params, *geo)
    strided = _C.mamba3_siso_forward(wide[..., :proj.shape[-1]], None, *params, *geo)
    gated = _C.mamba3_siso_forward(proj, gate, *params, *geo)
    monkeypatch.setenv("MLK_MAMBA3_SCAN", "unfused")
    expect = _C.mamba3_siso_forward(proj, None, *params, *geo).cpu().numpy()
    assert_bitwise(got, expect, "chunk-parallel vs unfused")
    assert_bitwise(strided, expect, "strided rows")
    assert_bitwise(gated, _C.mamba3_siso_forward(proj, gate, *params, *geo).cpu().numpy(), "explicit gate")


@pytest.mark.parametrize("B,L,G,H,D,R", [(24, 161, 1, 8, 64, 16), (33, 200, 2, 8, 64, 32), (200, 192, 1, 1, 32, 0),
                                         (65, 225, 1, 3, 64, 9), (48, 170, 1, 4, 32, 17)])
def test_scan_with_token_launch_equals_unfused(dev, monkeypatch, B, L, G, H, D, R):
    """d_state 64 over six chunks and more with many pairs: coefficients and tanh(angle) from a launch of their own."""
    from montlok import _C

    proj, params, geo = _case(dev, B, L, 64, G, H, D, R)
    got = _C.mamba3_siso_forward(proj, None, *params, *geo)
    monkeypatch.setenv("MLK_MAMBA3_SCAN", "unfused")
    assert_bitwise(got, _C.mamba3_siso_forward(proj, None, *params, *geo).cpu().numpy(), "token launch vs unfused")


@pytest.mark.parametrize("B,L,N,G,H,R", [(2, 200, 64, 1, 4, 16), (1, 97, 16, 2, 4, 8)])
def test_chunk_parallel_scan_headdim16(dev, oracle, monkeypatch, B, L, N, G, H, R):
    from montlok import _C

    proj, params, geo = _case(dev, B, L, N, G, H, 16, R)
    got = _C.mamba3_siso_forward(proj, None, *params, *geo)
    monkeypatch.setenv("MLK_MAMBA3_SCAN", "sequential")
    assert_close(got, _C.mamba3_siso_forward(proj, None, *params, *geo), tol=1e-6, name="vs sequential")


@pytest.mark.parametrize("B,L,N,G,H,D,R", [(1, 2048, 16, 1, 3, 32, 8), (1, 2049, 16, 1, 3, 32, 8), (2, 2600, 64, 1, 2, 64, 32),
                                           (3, 2100, 32, 2, 4, 16, 5), (1, 2200, 16, 1, 1, 64, 0)])
def test_long_windows_equal_unfused(dev, monkeypatch, B, L, N, G, H, D, R):
    """On both sides of 64 chunks, past which the angle sums before each chunk come from a launch of their own."""
    from montlok import _C

    proj, params, geo = _case(dev, B, L, N, G, H, D, R)
    got = _C.mamba3_siso_forward(proj, None, *params, *geo)
    if D == 16:
        monkeypatch.setenv("MLK_MAMBA3_SCAN", "sequential")
        assert_close(got, _C.mamba3_siso_forward(proj, None, *params, *geo), tol=1e-6, name="vs sequential")
        return
    monkeypatch.setenv("MLK_MAMBA3_SCAN", "unfused")
    assert_bitwise(got, _C.mamba3_siso_forward(proj, None, *params, *geo).cpu().numpy(), "chunk-parallel vs unfused")


def test_time_grows_with_the_window_not_its_square(dev):
    """64 pairs at four times the length: 4.1 times the time (5.9 where each chunk adds up all before it)."""
    from montlok import _C

    us = []
    _, params, geo = _case(dev, 8, 8, 16, 1, 8, 32, 4)
    for L in (8000, 32000):
        proj = torch.randn(8, L, 2 * 8 * 32 + 2 * 16 + 3 * 8 + 4, device=dev)
        times = []
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            _C.mamba3_siso_forward(proj, None, *params, *geo)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b) * 1e3)
        us.append(min(times))
    assert us[1] < 5.0 * us[0], us


def test_smaller_workspace_takes_the_fused_scan(dev):
    """A caller that holds only the unfused kernels' slab is served as before, with the same result."""
    from montlok import _C

    B, L, N, G, H, D, R = 2, 300, 64, 1, 8, 64, 16
    proj, params, geo = _case(dev, B, L, N, G, H, D, R)
    expect = _C.mamba3_siso_forward(proj, None, *params, *geo)
    lib = _C.library()
    slab = 4 * (2 * B * L * H * N + 3 * B * L * H + B * L * H * R)
    assert lib.mlk_mamba3_workspace_bytes(B, L, H, N, R) > slab
    ws = torch.empty(slab, dtype=torch.uint8, device=dev)
    out = torch.full((B, L, H * D), float("nan"), device=dev)
    status = lib.mlk_mamba3_siso_forward(proj.data_ptr(), B, L, proj.shape[-1], proj.stride(0), proj.stride(1), None, 0, 0,
                                         *(t.data_ptr() for t in params), N, G, H, D, R, 1e-5, 1e-5, 1e-4, out.data_ptr(),
                                         ws.data_ptr(), slab, torch.cuda.current_stream().cuda_stream)
    assert status == 0
    assert torch.equal(out, expect)
