"""GPU operators of the RDT4quant fused forward, under the names of ``montlok._C``.

The reference exposes these operators from a pybind11 CPU extension
(rdt4quant_cpu/montlok.cpp, op table at montlok.cpp:1457-1499). This module
keeps their names, positional/keyword order, return tuples and error texts,
and runs them on the ROCm device through the C ABI of ``libmlk_hip.so``
(``include/mlk_hip.h``). Inputs must be float32 tensors on the GPU; outputs
are allocated here with the caching allocator and filled on the current
stream. There is no CPU fallback: a missing library raises.
"""

from __future__ import annotations

import ctypes as C
import json
import os
import weakref
from pathlib import Path

import torch

LIB_PATH = Path(__file__).resolve().parent / "rdt" / "lib" / "libmlk_hip.so"

_vp = C.c_void_p
_i64 = C.c_int64
_dbl = C.c_double
_lib = None


def _load():
    global _lib
    if _lib is not None:
        return _lib
    path = Path(os.environ.get("MLK_HIP_LIB", LIB_PATH))
    if not path.exists():
        raise RuntimeError(f"{path} is not built: run __graft_entry__.build() (make -C montlok.cpp_amd)")
    lib = C.CDLL(str(path))
    lib.mlk_last_error.restype = C.c_char_p
    lib.mlk_abi_version.restype = C.c_int
    lib.mlk_build_info.argtypes = [C.c_char_p, C.c_size_t]
    lib.mlk_empty_kernel.argtypes = [_i64, _i64, C.c_size_t, _vp]
    lib.mlk_empty_kernel.restype = C.c_int
    sigs = {
        "mlk_rms_norm": [_vp, _i64, _i64, _i64, _vp, _dbl, _i64, _vp, _vp],
        "mlk_add_rms_norm": [_vp, _vp, _i64, _i64, _vp, _dbl, _i64, _vp, _vp, _vp],
        "mlk_layer_norm": [_vp, _i64, _i64, _i64, _vp, _vp, _dbl, _vp, _vp],
        "mlk_swiglu": [_vp, _i64, _i64, _i64, _vp, _vp],
        "mlk_linear": [_vp, _i64, _i64, _i64, _vp, C.c_int32, _vp, _i64, _vp, _i64, _vp],
        "mlk_linear_residual": [_vp, _i64, _i64, _i64, _vp, C.c_int32, _vp, _i64, _vp, _i64, _vp, _i64, _vp],
        "mlk_rms_norm_linear": [_vp, _i64, _i64, _i64, _vp, _dbl, _i64, _vp, C.c_int32, _vp, _i64, _vp, _i64, _vp],
        "mlk_linear_swiglu": [_vp, _i64, _i64, _i64, _vp, C.c_int32, _vp, _i64, _vp, _i64, _vp],
        "mlk_layer_norm_bf16": [_vp, _i64, _i64, _i64, _vp, _vp, _dbl, _vp, _vp],
        "mlk_mla_attend_normed": [_vp, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _vp, _vp, _vp, _vp, _dbl,
                                  _vp, _vp],
        "mlk_mla_rope_qk": [_vp, _i64, _i64, _vp, _vp, _i64, _vp, _vp, _i64, _i64, _i64, _i64, _i64, _vp, _vp],
        "mlk_mla_forward": [_vp, _i64, _i64, _i64, _i64, _i64, _vp, _vp, _vp, _dbl, _vp, _vp, _vp, _vp, _i64, _i64,
                            _i64, _i64, C.c_int32, _dbl, _vp, _vp],
        "mlk_mla_pack_weights": [_vp, _vp, _vp, _i64, _i64, _i64, _i64, _i64, C.c_int32, _vp, _vp],
        "mlk_mla_forward_packed": [_vp, _i64, _i64, _i64, _i64, _i64, _vp, _vp, _vp, _dbl, _vp, _vp, _i64, _i64, _i64,
                                   _i64, _dbl, _vp, _vp],
        "mlk_mla_attend": [_vp, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _vp, _vp, _dbl, _vp, _vp,
                           _vp, _dbl, _vp, _vp],
        "mlk_attention": [_vp, _i64, _i64, _vp, _i64, _i64, _vp, _i64, _i64, _i64, _i64, _i64, _i64, _i64, C.c_int32,
                          _dbl, C.c_int32, _vp, _vp],
        "mlk_mhc_prepare": [_vp, _i64, _i64, _i64, _i64, _i64, _vp, _dbl, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i64,
                            _vp, _dbl, _vp, _vp, _vp, _vp, _vp],
        "mlk_mhc_combine": [_vp, _i64, _i64, _i64, _i64, _i64, _vp, _vp, _vp, _vp, _vp, _vp],
        "mlk_math_check": [_vp, _i64, _vp, _vp],
        "mlk_mamba3_siso_recurrent": [_vp, _vp] * 7 + [_vp] + [_i64] * 5 + [_vp, _vp, C.c_size_t, _vp],
        "mlk_mamba3_siso_recurrent_noalloc": [_vp, _vp] * 7 + [_vp] + [_i64] * 5 + [_vp, _vp],
        "mlk_rms_norm_mamba3_forward": [_vp, _i64, _i64, _i64, _i64, _i64, _vp, _dbl, _i64, _vp, C.c_int32] +
                                       [_vp] * 6 + [_i64] * 5 + [_dbl, _dbl, _dbl, _vp, _vp],
        "mlk_mamba3_siso_forward": [_vp, _i64, _i64, _i64, _i64, _i64, _vp, _i64, _i64] + [_vp] * 6 + [_i64] * 5 +
                                   [_dbl, _dbl, _dbl, _vp, _vp, C.c_size_t, _vp],
        "mlk_mamba3_siso_step": [_vp, _i64, _i64] + [_vp] * 6 + [_i64] * 5 + [_dbl, _dbl, _dbl] + [_vp] * 4 +
                                [C.c_int, _vp, _vp],
        "mlk_mhc_combine_prepare": [_vp, _i64, _i64, _i64, _i64, _i64, _vp, _vp, _vp, _vp, _dbl, _vp, _vp, _vp, _vp,
                                    _vp, _vp, _vp, _i64, _vp, _dbl, _vp, _vp, _vp, _vp, _vp, _vp],
    }
    for name, args in sigs.items():
        fn = getattr(lib, name)
        fn.argtypes = args
        fn.restype = C.c_int
    lib.mlk_mamba3_workspace_bytes.argtypes = [_i64] * 5
    lib.mlk_mamba3_workspace_bytes.restype = C.c_size_t
    lib.mlk_mla_packed_elems.argtypes = [_i64] * 5
    lib.mlk_mla_packed_elems.restype = C.c_int64
    _lib = lib
    return lib


_native = None


def _ops():
    """The operators that make one launch each, from tensors to the C ABI (csrc/torch_ops.cpp), bound to the
    library that ``_load`` opened."""
    global _native
    if _native is None:
        import importlib.machinery
        import importlib.util

        _load()
        path = LIB_PATH.with_name("_torch_ops.so")
        if not path.exists():
            raise RuntimeError(f"{path} is not built: run __graft_entry__.build() (make -C montlok.cpp_amd)")
        loader = importlib.machinery.ExtensionFileLoader("_torch_ops", str(path))
        module = importlib.util.module_from_spec(importlib.util.spec_from_loader("_torch_ops", loader))
        loader.exec_module(module)
        module.bind(os.environ.get("MLK_HIP_LIB", str(LIB_PATH)))
        _native = module
    return _native


def library():
    """The loaded ``libmlk_hip.so`` (ctypes.CDLL)."""
    return _load()


def _call(name: str, *args) -> None:
    lib = _load()
    status = getattr(lib, name)(*args)
    if status != 0:
        raise RuntimeError(lib.mlk_last_error().decode())


def _stream() -> int:
    return (_native or _ops()).current_stream()


def _ptr(t: torch.Tensor | None) -> int | None:
    return None if t is None else t.data_ptr()


def _check(cond: bool, msg: str) -> None:
    if not cond:
        raise RuntimeError(msg)


# Validation mirrors montlok.cpp:43-65 with "on the GPU" in place of "on CPU".
def _require_f32_gpu(t: torch.Tensor | None, name: str) -> None:
    _check(t is not None, f"{name} must be defined")
    _check(t.device.type == "cuda", f"{name} must be on the GPU")
    _check(t.dtype == torch.float32, f"{name} must be float32")


def _dense_parameter(t: torch.Tensor, numel: int, name: str) -> torch.Tensor:
    _require_f32_gpu(t, name)
    _check(t.numel() == numel, f"{name} must have {numel} elements, got {t.numel()}")
    return t.contiguous()


def _rows(x: torch.Tensor, dim: int) -> tuple[torch.Tensor, int, int]:
    """[..., dim] -> (2-D view, rows, row stride), like x.reshape(-1, dim) (montlok.cpp:921-924)."""
    rows = x.reshape(-1, dim)
    if rows.stride(1) != 1 and dim != 1:
        rows = rows.contiguous()
    stride = rows.stride(0) if rows.size(0) > 1 else dim
    return rows, rows.size(0), stride


# ------------------------------------------------------------------ norms


def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float, groups: int) -> torch.Tensor:
    """montlok.cpp:915-938."""
    return (_native or _ops()).rms_norm(x, weight, eps, groups)


def add_rms_norm(left: torch.Tensor, right: torch.Tensor, weight: torch.Tensor, eps: float,
                 groups: int) -> tuple[torch.Tensor, torch.Tensor]:
    """montlok.cpp:978-1007: (left + right, rms_norm(left + right))."""
    return (_native or _ops()).add_rms_norm(left, right, weight, eps, groups)


def layer_norm(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None, eps: float) -> torch.Tensor:
    """montlok.cpp:1057-1082 (bias may be None or empty)."""
    return (_native or _ops()).layer_norm(x, weight, bias, eps)


def swiglu(x: torch.Tensor) -> torch.Tensor:
    """montlok.cpp:942-963: x [..., 2*hidden] = [gate | up] -> silu(gate) * up."""
    return (_native or _ops()).swiglu(x)


# ------------------------------------------------------------------ linear

_WEIGHT_DTYPES = {torch.float32: 0, torch.bfloat16: 1}


def _weight(weight: torch.Tensor, name: str = "weight") -> torch.Tensor:
    _check(weight is not None, f"{name} must be defined")
    _check(weight.device.type == "cuda", f"{name} must be on the GPU")
    _check(weight.dtype in _WEIGHT_DTYPES, f"{name} must be float32 or bfloat16")
    _check(weight.dim() == 2, f"{name} must be [out_features, in_features]")
    return weight.contiguous()


def _linear_into(rows: torch.Tensor, count: int, stride: int, weight: torch.Tensor, bias, out: torch.Tensor,
                 out_stride: int) -> None:
    n, k = weight.shape
    _call("mlk_linear", _ptr(rows), count, k, stride, _ptr(weight), _WEIGHT_DTYPES[weight.dtype], _ptr(bias), n,
          _ptr(out), out_stride, _stream())


def linear(input: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None = None) -> torch.Tensor:
    """linear_dispatch (montlok.cpp:67-91): input [..., K] @ weight[N, K]^T + bias -> [..., N].

    weight may be float32 or bfloat16 (bf16 matrix cores, fp32 accumulate)."""
    return (_native or _ops()).linear(input, weight, bias)


def linear_residual(input: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None,
                    residual: torch.Tensor) -> torch.Tensor:
    """residual + linear(input, weight, bias) in one launch, bit-identical to the two steps (the
    x = x + f(x) update of python/montlok/rdt/reference/Model/blocks.py:66-75)."""
    return (_native or _ops()).linear_residual(input, weight, bias, residual)


def rms_norm_linear(x: torch.Tensor, norm_weight: torch.Tensor, eps: float, groups: int, weight: torch.Tensor,
                    bias: torch.Tensor | None = None) -> torch.Tensor:
    """linear(rms_norm(x, norm_weight, eps, groups), weight, bias), one launch where the fused form is
    built (few rows, or K = 128 with fp32 weights), else the two operators; the results are identical either way."""
    out = (_native or _ops()).rms_norm_linear(x, norm_weight, eps, groups, weight, bias)
    if out is None:  # no fused form for this shape
        return linear(rms_norm(x, norm_weight, eps, groups), weight, bias)
    return out


def swiglu_mlp(input, in_weight, in_bias=None, out_weight=None, out_bias=None):
    """montlok.cpp:967-976: linear -> swiglu -> linear, the first two in one launch where that is built (fp32
    weights with K from 64 on, more than a few hundred rows)."""
    hidden = (_native or _ops()).linear_swiglu(input, in_weight, in_bias)
    if hidden is None:
        hidden = swiglu(linear(input, in_weight, in_bias))
    return linear(hidden, out_weight, out_bias)


# ------------------------------------------------------------------ mHC


def mhc_prepare(streams, norm_w, eps, proj_w, pre_bias, post_bias, res_bias, pre_alpha, post_alpha, res_alpha,
                sinkhorn_iters, n_streams=0, agg_norm_w=None, agg_norm_eps=0.0):
    """montlok.cpp:659-691 -> (agg [B,L,d], pre [B,L,n], post [B,L,n], res [B,L,n,n])."""
    return (_native or _ops()).mhc_prepare(streams, norm_w, eps, proj_w, pre_bias, post_bias, res_bias, pre_alpha, post_alpha,
                                           res_alpha, sinkhorn_iters, n_streams, agg_norm_w, agg_norm_eps)


def mhc_combine(streams, res, post, out):
    """montlok.cpp:726-739 -> new streams [B,L,n,d]."""
    return (_native or _ops()).mhc_combine(streams, res, post, out, False)


def mhc_combine_collapse(streams, res, post, out):
    """montlok.cpp:743-758 -> mean over the new streams [B,L,d]; streams never materialised."""
    return (_native or _ops()).mhc_combine(streams, res, post, out, True)


def mhc_combine_prepare(streams, res, post, out, norm_w, eps, proj_w, pre_bias, post_bias, res_bias, pre_alpha,
                        post_alpha, res_alpha, sinkhorn_iters, agg_norm_w=None, agg_norm_eps=0.0):
    """montlok.cpp:763-802 -> (new_streams, agg, pre, post, res) of the next residual."""
    return _mhc_combine_prepare(streams, res, post, out, norm_w, eps, proj_w, pre_bias, post_bias, res_bias,
                                pre_alpha, post_alpha, res_alpha, sinkhorn_iters, agg_norm_w, agg_norm_eps)


def _mhc_combine_prepare(streams, res, post, out, norm_w, eps, proj_w, pre_bias, post_bias, res_bias, pre_alpha,
                         post_alpha, res_alpha, sinkhorn_iters, agg_norm_w=None, agg_norm_eps=0.0, *,
                         reuse_streams=False, into=None):
    """mhc_combine_prepare with the buffers of montlok.cpp:807-852, 853-912 (mhc_combine_prepare_inplace,
    mhc_combine_prepare_reuse): reuse_streams writes the new streams over `streams` (contiguous
    [B, L, n, d], n <= 8); `into` = (agg, pre, post, res) buffers the next residual's coefficients are
    written into (they may be the `res` and `post` this call reads). Values are those of the plain call."""
    return (_native or _ops()).mhc_combine_prepare(streams, res, post, out, norm_w, eps, proj_w, pre_bias, post_bias, res_bias,
                                                   pre_alpha, post_alpha, res_alpha, sinkhorn_iters, agg_norm_w,
                                                   agg_norm_eps, reuse_streams, into)


# ------------------------------------------------------------------ Mamba-3


def _strides3(t: torch.Tensor):
    arr = (C.c_int64 * 3)(t.stride(0), t.stride(1), t.stride(2))
    return arr


def _require_inner_dense(t: torch.Tensor, name: str) -> None:
    """montlok.cpp:52-55."""
    _check(t.dim() >= 1 and (t.stride(-1) == 1 or t.size(-1) == 1),
           f"{name} must be contiguous along its last dimension")


def _workspace(nbytes: int, device) -> torch.Tensor:
    return torch.empty(max(int(nbytes), 4), dtype=torch.uint8, device=device)


def mamba3_siso_recurrent(q, k, v, gate, adt, dt, trap_logit, skip):
    """montlok.cpp:245-325: gated SSM output [B, L, H, D] (gate = z * sigmoid(z))."""
    return _siso_recurrent(q, k, v, gate, adt, dt, trap_logit, skip, noalloc=False)


def mamba3_siso_recurrent_noalloc(q, k, v, gate, adt, dt, trap_logit, skip):
    """mamba3_siso_recurrent through the entry point that allocates no device memory: the coefficients live
    in the library's static per-GPU scratch (B * L * H at most 699,050). Same result bit for bit. The library
    orders the calls that share a GPU's scratch across streams with an event; under graph capture only the
    graph orders them, and the first call on a device must be eager. No counterpart in the reference."""
    return _siso_recurrent(q, k, v, gate, adt, dt, trap_logit, skip, noalloc=True)


def _siso_recurrent(q, k, v, gate, adt, dt, trap_logit, skip, noalloc: bool):
    for t, name in ((q, "q"), (k, "k"), (v, "v"), (gate, "gate"), (adt, "adt"), (dt, "dt"),
                    (trap_logit, "trap_logit")):
        _require_f32_gpu(t, name)
    _check(q.dim() == 4 and k.shape == q.shape, "q/k must be [B,L,H,N]")
    _check(v.dim() == 4 and gate.shape == v.shape, "v/gate must be [B,L,H,D]")
    B, L, H, N = q.shape
    D = v.size(3)
    _check(v.size(0) == B and v.size(1) == L and v.size(2) == H, "v shape mismatch")
    _check(tuple(adt.shape) == (B, L, H), "adt must be [B,L,H]")
    _check(dt.shape == adt.shape and trap_logit.shape == adt.shape, "dt/trap_logit shape mismatch")
    for t, name in ((q, "q"), (k, "k"), (v, "v"), (gate, "gate")):
        _require_inner_dense(t, name)
    sk = _dense_parameter(skip, H, "skip")
    out = torch.empty((B, L, H, D), dtype=torch.float32, device=q.device)
    args = (_ptr(q), _strides3(q), _ptr(k), _strides3(k), _ptr(v), _strides3(v), _ptr(gate), _strides3(gate),
            _ptr(adt), _strides3(adt), _ptr(dt), _strides3(dt), _ptr(trap_logit), _strides3(trap_logit), _ptr(sk),
            B, L, H, N, D, _ptr(out))
    if noalloc:
        _call("mlk_mamba3_siso_recurrent_noalloc", *args, _stream())
    else:
        ws = _workspace(4 * 3 * B * L * H, q.device)
        _call("mlk_mamba3_siso_recurrent", *args, _ptr(ws), ws.numel(), _stream())
    return out


def mamba3_siso_forward(projected, gate, b_bias, c_bias, b_norm_w, c_norm_w, dt_bias, skip, d_state, ngroups,
                        nheads, headdim, num_rope_angles, b_eps, c_eps, a_floor):
    """montlok.cpp:333-492: in_proj output [B, L, W] -> out_proj input [B, L, d_inner].

    An empty ``gate`` evaluates silu of the z lanes of ``projected`` in the kernel."""
    return (_native or _ops()).mamba3_siso_forward(projected, gate, b_bias, c_bias, b_norm_w, c_norm_w, dt_bias, skip, d_state,
                                                   ngroups, nheads, headdim, num_rope_angles, b_eps, c_eps, a_floor)


def mamba3_siso_step(projected, state, b_bias, c_bias, b_norm_w, c_norm_w, dt_bias, skip, d_state, ngroups,
                     nheads, headdim, num_rope_angles, b_eps, c_eps, a_floor):
    """One token for S streams with carried state (no reference operator).

    projected: [S, W]; state: dict with ssm [S,H,N,D], k [S,H,N], v [S,H,D]
    (float32), angle [S,H,max(R,1)] (float64) updated in place, and
    ``started`` (False before the first token of a zero state; set True here).
    Returns [S, H*D]."""
    out = (_native or _ops()).mamba3_siso_step(projected, state["ssm"], state["k"], state["v"], state["angle"],
                                               bool(state.get("started", False)), b_bias, c_bias, b_norm_w, c_norm_w, dt_bias,
                                               skip, d_state, ngroups, nheads, headdim, num_rope_angles, b_eps, c_eps, a_floor)
    state["started"] = True
    return out


def mamba3_siso_layer(inputs, in_weight, out_weight, b_bias, c_bias, b_norm_w, c_norm_w, dt_bias, skip, d_state,
                      ngroups, nheads, headdim, num_rope_angles, b_eps, c_eps, a_floor):
    """montlok.cpp:496-519: in_proj -> mamba3_siso_forward (in-kernel gate) -> out_proj."""
    projected = linear(inputs, in_weight)
    output = mamba3_siso_forward(projected, None, b_bias, c_bias, b_norm_w, c_norm_w, dt_bias, skip, d_state, ngroups,
                                 nheads, headdim, num_rope_angles, b_eps, c_eps, a_floor)
    return linear(output, out_weight)


_BLOCK_PATH = {"last": None}


def rms_norm_mamba3_forward(inputs, norm_weight, norm_eps, norm_groups, in_weight, b_bias, c_bias, b_norm_w,
                            c_norm_w, dt_bias, skip, d_state, ngroups, nheads, headdim, num_rope_angles, b_eps, c_eps,
                            a_floor):
    """mamba3_siso_forward(linear(rms_norm(inputs, norm_weight, norm_eps, norm_groups), in_weight)) with the
    in-kernel gate: [B, L, d_model] -> [B, L, d_inner]. One launch where the fused kernel is built for the
    geometry (the in_proj rows stay in LDS), else rms_norm_linear then mamba3_siso_forward; the same result
    bit for bit where rms_norm_linear takes its one-wave-per-tile form. No single counterpart in the
    reference's op table (montlok.cpp:915-938, 333-492)."""
    out = (_native or _ops()).rms_norm_mamba3_forward(inputs, norm_weight, norm_eps, norm_groups, in_weight, b_bias, c_bias,
                                                      b_norm_w, c_norm_w, dt_bias, skip, d_state, ngroups, nheads, headdim,
                                                      num_rope_angles, b_eps, c_eps, a_floor)
    if out is not None:
        _BLOCK_PATH["mixer"] = ["rms_norm_mamba3_forward"]
        return out
    projected = rms_norm_linear(inputs, norm_weight, norm_eps, norm_groups, in_weight)
    _BLOCK_PATH["mixer"] = ["rms_norm_linear", "mamba3_siso_forward"]
    return mamba3_siso_forward(projected, None, b_bias, c_bias, b_norm_w, c_norm_w, dt_bias, skip, d_state, ngroups,
                               nheads, headdim, num_rope_angles, b_eps, c_eps, a_floor)


def mamba3_block(inputs, norm_weight, norm_eps, norm_groups, in_weight, out_weight, b_bias, c_bias, b_norm_w,
                 c_norm_w, dt_bias, skip, d_state, ngroups, nheads, headdim, num_rope_angles, b_eps, c_eps, a_floor):
    """The RMSNorm -> Mamba-3 residual block, x + mamba3_siso_layer(GroupedRMSNorm(x)) (the Mamba3Layer
    forward of python/montlok/rdt/reference/Model/layers/mamba3_layer.py:488-498 on the official backend;
    montlok.cpp:496-519 for the layer). No single counterpart in the reference's op table.

    rms_norm_mamba3_forward (one launch where built), then out_proj with the residual added in its
    epilogue: equal to rms_norm -> mamba3_siso_layer -> x + y bit for bit where the linears take their
    one-wave-per-tile forms."""
    _require_f32_gpu(inputs, "inputs")
    _check(inputs.dim() == 3, "inputs must be [B,L,d_model]")
    w_out = _weight(out_weight)
    _check(tuple(w_out.shape) == (inputs.size(-1), nheads * headdim),
           f"out_proj weight must be [{inputs.size(-1)}, {nheads * headdim}]")
    y = rms_norm_mamba3_forward(inputs, norm_weight, norm_eps, norm_groups, in_weight, b_bias, c_bias, b_norm_w,
                                c_norm_w, dt_bias, skip, d_state, ngroups, nheads, headdim, num_rope_angles, b_eps,
                                c_eps, a_floor)
    _BLOCK_PATH["last"] = _BLOCK_PATH["mixer"] + ["linear_residual"]
    return linear_residual(y, out_weight, None, inputs)


def mamba3_block_launches() -> list[str] | None:
    """The kernel launches the last ``mamba3_block`` call made, in order."""
    return _BLOCK_PATH["last"]


def mamba3_block_step(inputs, state, norm_weight, norm_eps, norm_groups, in_weight, out_weight, b_bias, c_bias,
                      b_norm_w, c_norm_w, dt_bias, skip, d_state, ngroups, nheads, headdim, num_rope_angles, b_eps,
                      c_eps, a_floor):
    """One token of ``mamba3_block`` for S streams with carried state: inputs [S, d_model] ->
    x + out_proj(mamba3_siso_step(in_proj(GroupedRMSNorm(x)))). ``state`` as for mamba3_siso_step, updated
    in place. Stepping T tokens from a zero state gives mamba3_block over those T tokens."""
    _require_f32_gpu(inputs, "inputs")
    _check(inputs.dim() == 2, "inputs must be [S,d_model]")
    projected = rms_norm_linear(inputs, norm_weight, norm_eps, norm_groups, in_weight)
    y = mamba3_siso_step(projected, state, b_bias, c_bias, b_norm_w, c_norm_w, dt_bias, skip, d_state, ngroups,
                         nheads, headdim, num_rope_angles, b_eps, c_eps, a_floor)
    return linear_residual(y, out_weight, None, inputs)


def stage1_forward(inputs, layers, mamba_norm_eps, mamba_norm_groups, ffn_norm_eps, d_state, ngroups, nheads, headdim,
                   num_rope_angles, b_eps, c_eps, a_floor):
    """montlok.cpp:1011-1053. Each layer pack holds 14 tensors: outer norm, Mamba in/out, B/C bias and norm,
    dt bias, D, FFN norm, FFN in weight/bias, FFN out weight/bias (empty tensor = no bias)."""
    _check(len(layers) > 0, "stage1 layers must not be empty")
    for layer in layers:
        _check(len(layer) == 14, "each stage1 tensor pack must contain 14 tensors")
    hidden = inputs
    mamba_input = rms_norm(hidden, layers[0][0], mamba_norm_eps, mamba_norm_groups)
    for index, layer in enumerate(layers):
        mamba_output = mamba3_siso_layer(mamba_input, *layer[1:9], d_state, ngroups, nheads, headdim,
                                         num_rope_angles, b_eps, c_eps, a_floor)
        hidden, normalized = add_rms_norm(hidden, mamba_output, layer[9], ffn_norm_eps, 1)
        in_bias = layer[11] if layer[11].numel() else None
        out_bias = layer[13] if layer[13].numel() else None
        ffn_output = swiglu_mlp(normalized, layer[10], in_bias, layer[12], out_bias)
        if index + 1 == len(layers):
            hidden = hidden + ffn_output
        else:
            hidden, mamba_input = add_rms_norm(hidden, ffn_output, layers[index + 1][0], mamba_norm_eps,
                                               mamba_norm_groups)
    return hidden


def stage2_tail_forward(backbone, depth, n_streams, attn_hc, attn_hc_eps, attn_sinkhorn_iters, attn_norm_weight,
                        attn_norm_eps, mla, kv_norm_eps, n_heads, head_dim, nope_dim, kv_lora_rank, attn_scale, ffn_hc,
                        ffn_hc_eps, ffn_sinkhorn_iters, ffn_norm_weight, ffn_norm_eps, ffn):
    """montlok.cpp:1217-1359: the recurrent stage-2 mHC tail, `depth` applications of one layer.

    The backbone [B, L, d] is expanded to n_streams as a broadcast view; each step runs MLA on the
    aggregated input, writes the attention residual fused with the FFN residual's coefficients, runs the
    SwiGLU MLP and writes that residual fused with the next attention residual's coefficients. The last
    step evaluates only the final query and returns the collapsed hidden state [B, 1, d].

    Packs (as model.py:160-232 builds them): each mHC pack holds dyn-norm weight, fp64 projection block,
    pre/post/res bias and pre/post/res alpha; the MLA pack holds the full and tail in_proj weights, q weight,
    kv-norm weight and bias (empty = none), kv_up weight, o_proj weight, cos and sin; the FFN pack holds the
    in weight and bias and the out weight and bias (empty = none).

    Buffers, as montlok.cpp:1291-1295 chooses them (values are the same either way): with
    MONTLOK_STAGE2_INPLACE unset or not "0" and n_streams <= 8, each residual write after the first goes
    over the materialised streams in place; with MONTLOK_STAGE2_REUSE_COEFF unset or not "0", the next
    residual's agg/pre/post/res are written over the current ones."""
    _check(depth > 0, "depth must be positive")
    _check(n_streams > 0, "n_streams must be positive")
    _check(len(attn_hc) == 8 and len(ffn_hc) == 8, "each mHC tensor pack must contain dyn/proj/biases/alphas")
    _check(len(mla) == 9, "MLA tensor pack must contain full/tail/q/norm/kv/out/rope tensors")
    _check(len(ffn) == 4, "FFN tensor pack must contain in/out weights and biases")

    def prepare(streams, hc, eps, iters, broadcast, norm_weight, norm_eps):
        return mhc_prepare(streams, hc[0], eps, hc[1], hc[2], hc[3], hc[4], hc[5], hc[6], hc[7], iters, broadcast,
                           norm_weight, norm_eps)

    def combine_prepare(streams, res, post, out, hc, eps, iters, norm_weight, norm_eps):
        return mhc_combine_prepare(streams, res, post, out, hc[0], eps, hc[1], hc[2], hc[3], hc[4], hc[5], hc[6],
                                   hc[7], iters, norm_weight, norm_eps)

    def run_mla(inputs, n_last):
        projection = mla[0] if n_last == inputs.size(1) else mla[1]
        return mla_forward(inputs, projection, mla[2], mla[3], mla[4], kv_norm_eps, mla[5], mla[6], mla[7], mla[8],
                           n_heads, head_dim, nope_dim, kv_lora_rank, n_last, True, attn_scale)

    def ffn_mlp(inputs):
        return swiglu_mlp(inputs, ffn[0], ffn[1] if ffn[1].numel() else None, ffn[2],
                          ffn[3] if ffn[3].numel() else None)

    agg, pre, post, res = prepare(backbone, attn_hc, attn_hc_eps, attn_sinkhorn_iters, n_streams,
                                  attn_norm_weight, attn_norm_eps)
    streams = backbone
    use_inplace = n_streams <= 8 and os.environ.get("MONTLOK_STAGE2_INPLACE") != "0"
    reuse_coefficients = os.environ.get("MONTLOK_STAGE2_REUSE_COEFF") != "0"

    def combine_prepare_reuse(streams, agg, pre, post, res, out, hc, eps, iters, norm_weight, norm_eps, in_place):
        return _mhc_combine_prepare(streams, res, post, out, hc[0], eps, hc[1], hc[2], hc[3], hc[4], hc[5], hc[6],
                                    hc[7], iters, norm_weight, norm_eps, reuse_streams=in_place,
                                    into=(agg, pre, post, res))

    def combine_prepare_inplace(streams, res, post, out, hc, eps, iters, norm_weight, norm_eps):
        return _mhc_combine_prepare(streams, res, post, out, hc[0], eps, hc[1], hc[2], hc[3], hc[4], hc[5], hc[6],
                                    hc[7], iters, norm_weight, norm_eps, reuse_streams=True)

    for step in range(depth):
        if step + 1 == depth:
            attn_out = run_mla(agg, 1)
            last = streams.size(1) - 1
            tail_streams = streams.narrow(1, last, 1).contiguous()
            written = mhc_combine(tail_streams, res.narrow(1, last, 1).contiguous(),
                                  post.narrow(1, last, 1).contiguous(), attn_out)
            f_agg, _, f_post, f_res = prepare(written, ffn_hc, ffn_hc_eps, ffn_sinkhorn_iters, 0, ffn_norm_weight,
                                              ffn_norm_eps)
            return mhc_combine_collapse(written, f_res, f_post, ffn_mlp(f_agg))
        attn_out = run_mla(agg, agg.size(1))
        if reuse_coefficients:
            streams = combine_prepare_reuse(streams, agg, pre, post, res, attn_out, ffn_hc, ffn_hc_eps,
                                            ffn_sinkhorn_iters, ffn_norm_weight, ffn_norm_eps,
                                            use_inplace and streams.dim() == 4)[0]
            ffn_out = ffn_mlp(agg)
            streams = combine_prepare_reuse(streams, agg, pre, post, res, ffn_out, attn_hc, attn_hc_eps,
                                            attn_sinkhorn_iters, attn_norm_weight, attn_norm_eps, use_inplace)[0]
            continue
        if use_inplace and streams.dim() == 4:
            streams, f_agg, _, f_post, f_res = combine_prepare_inplace(streams, res, post, attn_out, ffn_hc,
                                                                       ffn_hc_eps, ffn_sinkhorn_iters,
                                                                       ffn_norm_weight, ffn_norm_eps)
        else:
            streams, f_agg, _, f_post, f_res = combine_prepare(streams, res, post, attn_out, ffn_hc, ffn_hc_eps,
                                                               ffn_sinkhorn_iters, ffn_norm_weight, ffn_norm_eps)
        ffn_out = ffn_mlp(f_agg)
        if use_inplace:
            streams, agg, pre, post, res = combine_prepare_inplace(streams, f_res, f_post, ffn_out, attn_hc,
                                                                   attn_hc_eps, attn_sinkhorn_iters,
                                                                   attn_norm_weight, attn_norm_eps)
        else:
            streams, agg, pre, post, res = combine_prepare(streams, f_res, f_post, ffn_out, attn_hc, attn_hc_eps,
                                                           attn_sinkhorn_iters, attn_norm_weight, attn_norm_eps)
    raise AssertionError("unreachable stage-2 loop")


def new_mamba3_state(streams: int, nheads: int, d_state: int, headdim: int, num_rope_angles: int, device) -> dict:
    """Zero carried state for mamba3_siso_step."""
    return {"ssm": torch.zeros(streams, nheads, d_state, headdim, device=device),
            "k": torch.zeros(streams, nheads, d_state, device=device),
            "v": torch.zeros(streams, nheads, headdim, device=device),
            "angle": torch.zeros(streams, nheads, max(num_rope_angles, 1), dtype=torch.float64, device=device),
            "started": False}


# ------------------------------------------------------------------ MLA

MASK_NONE, MASK_CAUSAL_TOP_LEFT, MASK_CAUSAL_BOTTOM_RIGHT = 0, 1, 2


def mla_rope_qk(q: torch.Tensor, kv: torch.Tensor, k_rope: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor,
                nope_dim: int) -> torch.Tensor:
    """montlok.cpp:1093-1154: rotates q's rope lanes IN PLACE and returns k = cat(k_nope, rope(k_rope))."""
    return (_native or _ops()).mla_rope_qk(q, kv, k_rope, cos, sin, nope_dim)


def attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, mask: int, scale: float,
              precision: torch.dtype = torch.float32) -> torch.Tensor:
    """softmax(q k^T * scale) v over [B, L, H, hd] views -> [B, Lq, H, hd] (montlok.cpp:1205-1208).

    mask: MASK_NONE, MASK_CAUSAL_TOP_LEFT (is_causal) or MASK_CAUSAL_BOTTOM_RIGHT (trailing queries).
    precision: torch.bfloat16 runs QK^T and PV on bf16 matrix cores, torch.float32 stays fp32."""
    _check(precision in (torch.float32, torch.bfloat16), "precision must be float32 or bfloat16")
    return (_native or _ops()).attention(q, k, v, mask, scale, precision == torch.bfloat16)


def mla_forward(x, in_proj_weight, q_weight, kv_norm_weight, kv_norm_bias, kv_norm_eps, kv_up_weight, out_weight,
                cosine, sine, n_heads, head_dim, nope_dim, kv_lora_rank, n_last, causal, scale):
    """montlok.cpp:1159-1211: projection, latent LayerNorm, kv_up, RoPE, attention and output projection.

    Weights may be float32 or bfloat16; with bf16 weights the attention contractions run on bf16 matrix
    cores as well (fp32 softmax and accumulation), and for the full causal sequence the part between the
    two projections runs as one fused kernel (same result, bit for bit)."""
    return _mla_forward(x, in_proj_weight, q_weight, kv_norm_weight, kv_norm_bias, kv_norm_eps, kv_up_weight,
                        out_weight, cosine, sine, n_heads, head_dim, nope_dim, kv_lora_rank, n_last, causal, scale,
                        allow_fused=True)


def _fused_attend(projected, batch, length, q_width, n_heads, head_dim, nope_dim, kv_lora_rank, kv_norm_weight,
                  kv_norm_bias, kv_norm_eps, kv_up_weight, cosine, sine, scale):
    """The fused LayerNorm/kv_up/RoPE/attention kernel, or None where it is not built for the geometry."""
    rope = head_dim - nope_dim
    geometry = (head_dim, nope_dim, kv_lora_rank) in ((32, 16, 64), (64, 32, 64)) and \
        length <= (128 if head_dim == 32 else 256)
    if not geometry or kv_up_weight.dtype != torch.bfloat16 or projected.stride(-1) != 1:
        return None
    w = _dense_parameter(kv_norm_weight, kv_lora_rank, "kv_norm.weight")
    b = None if kv_norm_bias is None or kv_norm_bias.numel() == 0 else _dense_parameter(kv_norm_bias, kv_lora_rank,
                                                                                       "kv_norm.bias")
    up = _weight(kv_up_weight, "kv_up_weight")
    _check(tuple(cosine.shape) == (length, rope) and cosine.is_contiguous(), "cos must be contiguous [L,rope_dim]")
    _check(sine.shape == cosine.shape and sine.is_contiguous(), "sin must be contiguous [L,rope_dim]")
    out = torch.empty((batch, length, n_heads, head_dim), dtype=torch.float32, device=projected.device)
    ts = projected.stride(1) if length > 1 else projected.size(-1)
    lib = _load()
    status = lib.mlk_mla_attend(_ptr(projected), batch, length, ts, 0, q_width, q_width + kv_lora_rank, n_heads,
                                head_dim, nope_dim, kv_lora_rank, _ptr(w), _ptr(b), float(kv_norm_eps), _ptr(up),
                                _ptr(cosine), _ptr(sine), float(scale), _ptr(out), _stream())
    if status == 3:  # MLK_ERR_UNSUPPORTED
        return None
    if status != 0:
        raise RuntimeError(lib.mlk_last_error().decode())
    return out


def _latent_normed(projected: torch.Tensor, q_width: int, kv_lora_rank: int, kv_norm_weight, kv_norm_bias,
                   kv_norm_eps: float):
    """LayerNorm of the latent columns of the in_proj rows [count, W], once per row, rounded to bf16
    (the form the fused attention takes); None where the rows have no vector form."""
    count, n = projected.shape
    lw = _dense_parameter(kv_norm_weight, kv_lora_rank, "kv_norm.weight")
    lb = None if kv_norm_bias is None or kv_norm_bias.numel() == 0 else _dense_parameter(kv_norm_bias, kv_lora_rank,
                                                                                        "kv_norm.bias")
    latent = torch.empty((count, kv_lora_rank), dtype=torch.bfloat16, device=projected.device)
    lib = _load()
    status = lib.mlk_layer_norm_bf16(_ptr(projected) + 4 * q_width, count, kv_lora_rank, n, _ptr(lw), _ptr(lb),
                                     float(kv_norm_eps), _ptr(latent), _stream())
    if status == 3:  # MLK_ERR_UNSUPPORTED
        return None
    if status != 0:
        raise RuntimeError(lib.mlk_last_error().decode())
    return latent


def _attend_normed(projected: torch.Tensor, latent: torch.Tensor, batch, length, q_width, n_heads, head_dim,
                   nope_dim, kv_lora_rank, kv_up_weight, cosine, sine, scale):
    """The fused attention reading the normalised bf16 latent; None where it is not built."""
    rope = head_dim - nope_dim
    up = _weight(kv_up_weight, "kv_up_weight")
    _check(tuple(cosine.shape) == (length, rope) and cosine.is_contiguous(), "cos must be contiguous [L,rope_dim]")
    _check(sine.shape == cosine.shape and sine.is_contiguous(), "sin must be contiguous [L,rope_dim]")
    n = projected.size(-1)
    out = torch.empty((batch, length, n_heads, head_dim), dtype=torch.float32, device=projected.device)
    lib = _load()
    status = lib.mlk_mla_attend_normed(_ptr(projected), batch, length, n, 0, q_width + kv_lora_rank, n_heads,
                                       head_dim, nope_dim, kv_lora_rank, _ptr(latent), _ptr(up), _ptr(cosine),
                                       _ptr(sine), float(scale), _ptr(out), _stream())
    if status == 3:
        return None
    if status != 0:
        raise RuntimeError(lib.mlk_last_error().decode())
    return out


def _fused_attend_ln(x, in_proj_weight, batch, length, q_width, n_heads, head_dim, nope_dim, kv_lora_rank,
                     kv_norm_weight, kv_norm_bias, kv_norm_eps, kv_up_weight, cosine, sine, scale):
    """in_proj, the latent LayerNorm once per row into bf16, then the fused attention reading the
    normalised latent (rather than normalising it again in every head's block): bit-identical to linear
    followed by _fused_attend. None where a kernel is not built for the geometry."""
    geometry = (head_dim, nope_dim, kv_lora_rank) in ((32, 16, 64), (64, 32, 64)) and \
        length <= (128 if head_dim == 32 else 256)
    if not geometry or kv_up_weight.dtype != torch.bfloat16:
        return None
    w = _weight(in_proj_weight, "in_proj_weight")
    n, k = w.shape
    _check(x.size(-1) == k, f"input must end in in_features={k}")
    rows, count, stride = _rows(x, k)
    projected = torch.empty((count, n), dtype=torch.float32, device=x.device)
    _linear_into(rows, count, stride, w, None, projected, n)
    latent = _latent_normed(projected, q_width, kv_lora_rank, kv_norm_weight, kv_norm_bias, kv_norm_eps)
    if latent is None:
        return None
    return _attend_normed(projected, latent, batch, length, q_width, n_heads, head_dim, nope_dim, kv_lora_rank,
                          kv_up_weight, cosine, sine, scale)


_MLA_PATH = {"last": None}


def mla_forward_launches() -> list[str] | None:
    """The kernel launches the last ``mla_forward`` call made, in order."""
    return _MLA_PATH["last"]


# Packed copies of the per-window kernel's weights (mlk_mla_pack_weights), one per (in_proj, kv_up, out)
# weight triple. An entry holds the three tensors only through weak references (a deleted model's weights
# and its entry go together) and is used only while each weight is the same live object with the same
# data_ptr() and _version, the key the reference's own weight caches use; an in-place update through the
# tensor or a `.data = new` swap makes a new copy. Like the reference's caches it cannot see an in-place
# change made through `w.data` (that leaves both data_ptr and _version as they were). A pack made while a
# stream is being captured is used for that call and not cached (its pack kernel runs only at replay).
# A few entries at most, oldest dropped first.
_MLA_PACKS: list = []
_MLA_PACKS_MAX = 4


def _weight_key(w):
    return (w.data_ptr(), w._version)


def _mla_packed(in_proj_weight, kv_up_weight, out_weight, n_heads, head_dim, nope_dim, kv_lora_rank):
    """The packed weights of mlk_mla_forward_packed, from the cache or made now; None where the geometry
    has no packed form."""
    ws = (in_proj_weight, kv_up_weight, out_weight)
    keys = tuple(_weight_key(w) for w in ws)
    stream = torch.cuda.current_stream(in_proj_weight.device)
    _MLA_PACKS[:] = [e for e in _MLA_PACKS if all(r() is not None for r in e[0])]
    for refs, ekeys, packed, made_on in _MLA_PACKS:
        if all(r() is w for r, w in zip(refs, ws)) and ekeys == keys:
            if stream != made_on:
                packed.record_stream(stream)
            return packed
    packed = mla_pack_weights(in_proj_weight, kv_up_weight, out_weight, n_heads, head_dim, nope_dim, kv_lora_rank)
    if packed is None or torch.cuda.is_current_stream_capturing():
        return packed
    _MLA_PACKS.insert(0, (tuple(weakref.ref(w) for w in ws), keys, packed, stream))
    del _MLA_PACKS[_MLA_PACKS_MAX:]
    return packed


def mla_pack_weights(in_proj_weight, kv_up_weight, out_weight, n_heads, head_dim, nope_dim, kv_lora_rank):
    """The three bf16 weights of the one-launch MLA kernel in its fragment order (mlk_mla_pack_weights), or
    None where no such kernel is built for the geometry."""
    for name, w in (("in_proj_weight", in_proj_weight), ("kv_up_weight", kv_up_weight), ("out_weight", out_weight)):
        _check(w.is_cuda and w.dtype == torch.bfloat16 and w.is_contiguous(), f"{name} must be contiguous bf16 on GPU")
    d_model = n_heads * head_dim
    lib = _load()
    elems = lib.mlk_mla_packed_elems(d_model, n_heads, head_dim, nope_dim, kv_lora_rank)
    if elems <= 0:
        return None
    packed = torch.empty(elems, dtype=torch.bfloat16, device=in_proj_weight.device)
    _call("mlk_mla_pack_weights", _ptr(in_proj_weight), _ptr(kv_up_weight), _ptr(out_weight), d_model, n_heads,
          head_dim, nope_dim, kv_lora_rank, _WEIGHT_DTYPES[torch.bfloat16], _ptr(packed), _stream())
    return packed


def _mla_window(x, in_proj_weight, kv_norm_weight, kv_norm_bias, kv_norm_eps, kv_up_weight, out_weight, cosine,
                sine, n_heads, head_dim, nope_dim, kv_lora_rank, scale):
    """The whole forward for every causal query in one launch, on the weights packed in the kernel's fragment
    order (bf16 weights, kv rank 64, a positive scale; 8 heads of 32 with rope 16 and L <= 128: one block per
    window; 4 heads of 64 with rope 32 and L <= 512: one block per window and 64 query rows); None where no
    such kernel is built for the call."""
    batch, length, d_model = x.shape
    ws = [in_proj_weight, kv_up_weight, out_weight]
    if any(w.dtype != torch.bfloat16 or not w.is_contiguous() for w in ws) or x.stride(-1) != 1:
        return None
    rope = head_dim - nope_dim
    if tuple(cosine.shape) != (length, rope) or not cosine.is_contiguous() or sine.shape != cosine.shape or \
            not sine.is_contiguous():
        return None
    _check(tuple(in_proj_weight.shape) == (d_model + kv_lora_rank + rope, d_model),
           "in_proj_weight must be [d_model + kv_lora_rank + rope_dim, d_model]")
    _check(tuple(kv_up_weight.shape) == (n_heads * (nope_dim + head_dim), kv_lora_rank),
           "kv_up_weight must be [n_heads * (nope_dim + head_dim), kv_lora_rank]")
    _check(tuple(out_weight.shape) == (d_model, d_model), "out_weight must be [d_model, d_model]")
    w = _dense_parameter(kv_norm_weight, kv_lora_rank, "kv_norm.weight")
    b = None if kv_norm_bias is None or kv_norm_bias.numel() == 0 else _dense_parameter(kv_norm_bias, kv_lora_rank,
                                                                                       "kv_norm.bias")
    out = torch.empty((batch, length, d_model), dtype=torch.float32, device=x.device)
    lib = _load()
    packed = _mla_packed(in_proj_weight, kv_up_weight, out_weight, n_heads, head_dim, nope_dim, kv_lora_rank)
    if packed is not None:
        status = lib.mlk_mla_forward_packed(_ptr(x), batch, length, d_model, x.stride(0), x.stride(1), _ptr(packed),
                                            _ptr(w), _ptr(b), float(kv_norm_eps), _ptr(cosine), _ptr(sine), n_heads,
                                            head_dim, nope_dim, kv_lora_rank, float(scale), _ptr(out), _stream())
    else:
        status = lib.mlk_mla_forward(_ptr(x), batch, length, d_model, x.stride(0), x.stride(1),
                                     _ptr(in_proj_weight), _ptr(w), _ptr(b), float(kv_norm_eps), _ptr(kv_up_weight),
                                     _ptr(out_weight), _ptr(cosine), _ptr(sine), n_heads, head_dim, nope_dim,
                                     kv_lora_rank, _WEIGHT_DTYPES[torch.bfloat16], float(scale), _ptr(out), _stream())
    if status == 3:  # MLK_ERR_UNSUPPORTED
        return None
    if status != 0:
        raise RuntimeError(lib.mlk_last_error().decode())
    return out


def _mla_forward(x, in_proj_weight, q_weight, kv_norm_weight, kv_norm_bias, kv_norm_eps, kv_up_weight, out_weight,
                 cosine, sine, n_heads, head_dim, nope_dim, kv_lora_rank, n_last, causal, scale, allow_fused,
                 allow_window=True):
    _require_f32_gpu(x, "x")
    _check(x.dim() == 3, "x must be [B,L,d_model]")
    batch, length, d_model = x.shape
    _check(n_heads > 0 and head_dim > 0 and d_model == n_heads * head_dim, "invalid MLA head geometry")
    _check(0 <= nope_dim < head_dim and kv_lora_rank > 0, "invalid MLA latent geometry")
    _check(n_last == 1 or n_last == length, "native MLA supports the final query or the full sequence")
    precision = torch.bfloat16 if _weight(in_proj_weight, "in_proj_weight").dtype == torch.bfloat16 else torch.float32
    full = n_last == length
    # Beyond 256 rows a block of the one-launch kernel walks up to eight key tiles: 35 us at 257 rows and 53 at 512
    # however few windows there are, against 33 and 48 us for one window, 39 and 59 for three, 41 and 65 for four in
    # separate operators (ten lengths from 257 to 512, from four windows on 1.17 to 2.1 times as fast at each).
    if allow_fused and allow_window and full and causal and precision == torch.bfloat16 and \
            (length <= 256 or batch >= 4):
        out = _mla_window(x, in_proj_weight, kv_norm_weight, kv_norm_bias, kv_norm_eps, kv_up_weight, out_weight,
                          cosine, sine, n_heads, head_dim, nope_dim, kv_lora_rank, scale)
        if out is not None:
            _MLA_PATH["last"] = ["mla_forward"]
            return out
    if allow_fused and full and causal and precision == torch.bfloat16:
        attended = _fused_attend_ln(x, in_proj_weight, batch, length, d_model, n_heads, head_dim, nope_dim,
                                    kv_lora_rank, kv_norm_weight, kv_norm_bias, kv_norm_eps, kv_up_weight, cosine,
                                    sine, scale)
        if attended is not None:
            _MLA_PATH["last"] = ["linear", "layer_norm_bf16", "mla_attend_normed", "linear"]
            return linear(attended.view(batch, length, d_model), out_weight)
    projected = linear(x, in_proj_weight)
    if allow_fused and full and causal and precision == torch.bfloat16:
        attended = _fused_attend(projected, batch, length, d_model, n_heads, head_dim, nope_dim, kv_lora_rank,
                                 kv_norm_weight, kv_norm_bias, kv_norm_eps, kv_up_weight, cosine, sine, scale)
        if attended is not None:
            _MLA_PATH["last"] = ["linear", "mla_attend", "linear"]
            return linear(attended.view(batch, length, d_model), out_weight)
    _MLA_PATH["last"] = ["separate"]
    q_width = d_model if full else 0
    if full:
        q = projected[..., :q_width]
    else:
        _check(q_weight.numel() == d_model * d_model, "q_weight must be [d_model,d_model] for a tail query")
        q = linear(x[:, length - 1:], q_weight)
    q = q.view(batch, n_last, n_heads, head_dim) if q.is_contiguous() else q.unflatten(-1, (n_heads, head_dim))
    kv_latent = projected[..., q_width:q_width + kv_lora_rank]
    k_rope = projected[..., q_width + kv_lora_rank:]
    kv_normalized = layer_norm(kv_latent, kv_norm_weight, kv_norm_bias, kv_norm_eps)
    kv = linear(kv_normalized, kv_up_weight).view(batch, length, n_heads, nope_dim + head_dim)
    k = mla_rope_qk(q, kv, k_rope, cosine, sine, nope_dim)
    v = kv[..., nope_dim:]
    mask = MASK_CAUSAL_TOP_LEFT if (full and causal) else MASK_NONE
    attended = attention(q, k, v, mask, scale, precision)
    return linear(attended.view(batch, n_last, d_model), out_weight)


# ------------------------------------------------------------------ introspection


def build_info() -> dict:
    """Kernel variant and device of this library (replaces montlok.cpp:1417-1455)."""
    lib = _load()
    buf = C.create_string_buffer(1024)
    _call("mlk_build_info", buf, len(buf))
    info = json.loads(buf.value.decode())
    info["library"] = str(LIB_PATH)
    return info


def cpu_features() -> dict:
    """Instruction-set features of the host CPU, with the reference's keys (montlok.cpp:1361-1378), read
    from /proc/cpuinfo (empty brand and all flags false where that file is absent)."""
    import platform

    brand, flags = "", set()
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                key, _, value = line.partition(":")
                key = key.strip()
                if key == "model name" and not brand:
                    brand = value.strip()
                elif key in ("flags", "Features") and not flags:
                    flags = set(value.split())
    except OSError:
        pass
    machine = platform.machine().lower()
    info = {"brand": brand,
            "arch": "x86-64" if machine in ("x86_64", "amd64") else ("arm64" if machine in ("aarch64", "arm64")
                                                                     else "other")}
    for key, flag in (("sse2", "sse2"), ("sse4_2", "sse4_2"), ("avx", "avx"), ("fma", "fma"), ("avx2", "avx2"),
                      ("avx512f", "avx512f"), ("avx512dq", "avx512dq"), ("avx512bw", "avx512bw"),
                      ("avx512vl", "avx512vl")):
        info[key] = flag in flags
    # The OS saves the wide registers when it exposes the features (xsave state enabled).
    info["os_avx"] = info["avx"] and "osxsave" in flags
    info["os_avx512"] = info["os_avx"] and info["avx512f"]
    return info


def isa_variants() -> list[dict]:
    """One kernel variant (gfx950); the reference lists its x86 ISA variants here."""
    return [{"name": "gfx950", "supported": True, "fma": True}]


def active_isa() -> str:
    return "gfx950"


def set_isa(name: str, force: bool = False) -> str:
    if name not in ("gfx950", "auto"):
        raise RuntimeError(f"unknown kernel variant {name!r}: this library has gfx950 only")
    return "gfx950"


def exported_symbols() -> list[str]:
    """Names of the C ABI entry points this module binds."""
    return ["mlk_last_error", "mlk_abi_version", "mlk_build_info", "mlk_empty_kernel", "mlk_rms_norm", "mlk_add_rms_norm",
            "mlk_layer_norm", "mlk_swiglu", "mlk_mhc_prepare", "mlk_mhc_combine", "mlk_mhc_combine_prepare",
            "mlk_math_check", "mlk_mamba3_workspace_bytes", "mlk_mamba3_siso_recurrent",
            "mlk_mamba3_siso_recurrent_noalloc", "mlk_mamba3_siso_forward", "mlk_rms_norm_mamba3_forward",
            "mlk_mamba3_siso_step", "mlk_linear", "mlk_linear_residual", "mlk_rms_norm_linear", "mlk_linear_swiglu",
            "mlk_layer_norm_bf16", "mlk_mla_rope_qk", "mlk_attention", "mlk_mla_attend", "mlk_mla_attend_normed",
            "mlk_mla_forward", "mlk_mla_packed_elems", "mlk_mla_pack_weights", "mlk_mla_forward_packed"]


def empty_kernel(blocks: int, threads: int, dynamic_lds_bytes: int = 0) -> None:
    """One launch of a kernel that does nothing, in the given launch shape, on the current stream (graph
    nodes of it time a launch's floor). No counterpart in the reference."""
    _call("mlk_empty_kernel", blocks, threads, dynamic_lds_bytes, _stream())


def math_check(x: torch.Tensor) -> dict:
    """Device exp / tanh / sigmoid / reciprocal (float64) of x, for error bounds."""
    _check(x.device.type == "cuda" and x.dtype == torch.float64, "x must be a float64 GPU tensor")
    x = x.contiguous().reshape(-1)
    out = torch.empty(4 * x.numel(), dtype=torch.float64, device=x.device)
    _call("mlk_math_check", _ptr(x), x.numel(), _ptr(out), _stream())
    e, t, s, r = out.view(4, -1)
    return {"exp": e, "tanh": t, "sigmoid": s, "recip": r}
