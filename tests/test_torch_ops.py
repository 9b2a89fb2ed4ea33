"""The operators' argument checks (csrc/torch_ops.cpp) where no GPU is needed: what is refused, with which text."""

from __future__ import annotations

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
