"""The operators' argument checks (csrc/torch_ops.cpp) where no GPU is needed: what is refused, with which text."""

from __future__ import annotations

import sys
import threading

import numpy as np
import pytest
import torch


@pytest.mark.parametrize("call,text", [
    (lambda c, x: c.rms_norm(x, x[0], 1e-5, 1), "x must be on the GPU"),
    (lambda c, x: c.rms_norm(None, x[0], 1e-5, 1), "x must be defined"),
    (lambda c, x: c.add_rms_norm(x, None, x[0], 1e-5, 1), "left must be on the GPU"),
    (lambda c, x: c.layer_norm(x, x[0], None, 1e-5), "x must be on the GPU"),
    (lambda c, x: c.swiglu(x), "x must be on the GPU"),
    (lambda c, x: c.linear(x, x), "input must be on the GPU"),
    (lambda c, x: c.linear_residual(x, x, None, x), "input must be on the GPU"),
    (lambda c, x: c.rms_norm_linear(x, x[0], 1e-5, 1, x), "x must be on the GPU"),
    (lambda c, x: c.mhc_prepare(x, *[None] * 9, 20), None),
    (lambda c, x: c.mhc_combine(x, x, x, x), "streams must be on the GPU"),
    (lambda c, x: c.mamba3_siso_forward(x, None, *[x] * 6, 16, 1, 2, 32, 4, 1e-5, 1e-5, 1e-4), "projected must be on the GPU"),
    (lambda c, x: c.mla_rope_qk(x, x, x, x, x, 2), "q must be on the GPU"),
    (lambda c, x: c.attention(x, x, x, 0, 1.0), "q must be on the GPU"),
    (lambda c, x: c.attention(x, x, x, 0, 1.0, torch.float16), "precision must be float32 or bfloat16"),
])
def test_refusals_without_a_gpu(call, text):
    from montlok import _C

    x = torch.ones(4, 4)
    with pytest.raises((RuntimeError, TypeError) if text is None else RuntimeError, match=text):
        call(_C, x)


def test_missing_library_is_refused(tmp_path):
    from montlok import _C

    with pytest.raises(RuntimeError):
        _C._ops().bind(str(tmp_path / "absent.so"))


@pytest.mark.parametrize("one", [1, 1.0, torch.tensor(1), np.float32(1), np.int64(1)])
@pytest.mark.parametrize("eps", [1e-5, "1e-5", torch.tensor(1e-5), np.float32(1e-5)])
def test_numbers_as_int_and_float_take_them(one, eps):
    """Whole numbers of any type for groups, iterations, streams and mask; anything float() takes for eps and scale."""
    from montlok import _C

    x, n = torch.ones(4, 4), (None,)
    for call in (lambda: _C.rms_norm(x, x, eps, one), lambda: _C.add_rms_norm(x, x, x, eps, one),
                 lambda: _C.rms_norm_linear(x, x, eps, one, x), lambda: _C.layer_norm(x, x, None, eps),
                 lambda: _C.mhc_prepare(x, x, eps, *n * 7, one, one, None, eps),
                 lambda: _C.mhc_combine_prepare(x, x, x, x, x, eps, *n * 7, one, None, eps),
                 lambda: _C.mamba3_siso_forward(x, None, *n * 6, 16, 1, 2, 32, 4, eps, eps, eps),
                 lambda: _C.rms_norm_mamba3_forward(x, x, eps, one, x, *n * 6, 16, 1, 2, 32, 4, eps, eps, eps),
                 lambda: _C.attention(x, x, x, one, eps)):
        with pytest.raises(RuntimeError, match="must be on the GPU"):
            call()


@pytest.mark.parametrize("groups,eps", [(1.5, 1e-5), ("1", 1e-5), (None, 1e-5), (2.0 ** 70, 1e-5), (float("nan"), 1e-5),
                                        (1, None), (1, "small"), (1, 1j)])
def test_what_is_no_number_is_refused(groups, eps):
    from montlok import _C

    x = torch.ones(4, 4)
    with pytest.raises(TypeError):
        _C.rms_norm(x, x, eps, groups)


_N = (None,)
_OPERATORS = [
    lambda c, x: c.rms_norm(x, x, 1e-5, 1),
    lambda c, x: c.add_rms_norm(x, x, x, 1e-5, 1),
    lambda c, x: c.layer_norm(x, x, None, 1e-5),
    lambda c, x: c.swiglu(x),
    lambda c, x: c.linear(x, x),
    lambda c, x: c.linear_residual(x, x, None, x),
    lambda c, x: c.rms_norm_linear(x, x, 1e-5, 1, x),
    lambda c, x: c.swiglu_mlp(x, x, None, x),
    lambda c, x: c.mhc_prepare(x, x, 1e-5, *_N * 7, 20),
    lambda c, x: c.mhc_combine(x, x, x, x),
    lambda c, x: c.mhc_combine_collapse(x, x, x, x),
    lambda c, x: c.mhc_combine_prepare(x, x, x, x, x, 1e-5, *_N * 7, 20),
    lambda c, x: c.mamba3_siso_forward(x, None, *_N * 6, 16, 1, 2, 32, 4, 1e-5, 1e-5, 1e-4),
    lambda c, x: c.mamba3_siso_step(x, dict(ssm=x, k=x, v=x, angle=x), *_N * 6, 16, 1, 2, 32, 4, 1e-5, 1e-5, 1e-4),
    lambda c, x: c.rms_norm_mamba3_forward(x, x, 1e-5, 1, x, *_N * 6, 16, 1, 2, 32, 4, 1e-5, 1e-5, 1e-4),
    lambda c, x: c.mla_rope_qk(x, x, x, x, x, 2),
    lambda c, x: c.attention(x, x, x, 0, 1.0),
]


@pytest.mark.parametrize("call", _OPERATORS)
def test_operators_let_other_threads_run(call):
    """The checks, the allocation and the launch run without the interpreter's lock. With the switch interval out of
    reach, a thread that waits for the lock gets it only where a call gives it up."""
    from montlok import _C

    _C._ops()
    x, ran, gate = torch.ones(4, 4), threading.Event(), threading.Lock()

    def other():
        with gate:
            ran.set()

    before = sys.getswitchinterval()
    sys.setswitchinterval(1000.0)
    try:
        gate.acquire()
        thread = threading.Thread(target=other, daemon=True)
        thread.start()
        gate.release()
        for _ in range(20000):
            try:
                call(_C, x)
            except RuntimeError:
                pass
            if ran.is_set():
                break
        passed = ran.is_set()
    finally:
        sys.setswitchinterval(before)
    thread.join(10.0)
    assert passed
