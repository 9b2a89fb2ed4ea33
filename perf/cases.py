"""The forward passes whose speed this package answers for.

Each case is one call that a program makes on the public modules of
``montlok.rdt`` with inputs on the GPU: a single layer or block with weights of
its own, or a whole model. ``listed()`` names fixed ones, ``draw(rng)`` gives
further ones of the same ranges, ``prepare`` builds what the program holds
before the call, ``run`` is the call, ``exact`` the same values in float64 from
plain tensor operations, ``work`` the bytes and operations the call cannot do
without and ``tolerance`` how far two correct implementations may differ.

Geometries are those of the package's own configurations: the RDT4quant model
reads windows of 480 bars of 57 features at d_model 256 (Mamba-3 with 8 heads
of 64 and d_state 64, MLA with 4 heads of 64, 32 of them rotary, kv rank 64, 4
mHC streams); the stack reads 256 bars of 40 features with bf16 weights; the
decode stack steps d_model 128 layers; the short block is d_model 64.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path
from types import SimpleNamespace

import torch
from torch.nn import functional as F

_PACKAGE = str(Path("montlok.cpp_amd").resolve())  # the working folder is the repository's root
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import montlok.rdt as rdt  # noqa: E402
from montlok.rdt.stack import HybridStackHIP  # noqa: E402

DEV = "cuda"
_BF16 = torch.bfloat16

# Mamba-3 block of the short windows, of the decode layers, of the model; MLA with 8 heads of 32 or 4 of 64.
_SHORT = dict(d_model=64, d_state=16, headdim=32)
_DECODE = dict(d_model=128, d_state=64, headdim=64)
_MODEL = dict(d_model=256, d_state=64, headdim=64)
_MLA = {8: dict(head_dim=32, rope=16), 4: dict(head_dim=64, rope=32)}
_KV_RANK = 64
_FFN_HIDDEN = 512
_FEATURES, _STACK_FEATURES = 57, 40


def listed():
    return [
        # The short-window block in fp32: ten microseconds of device work, so launches and the host count.
        dict(name="block_64x32", kind="block", windows=64, length=32),
        # One residual of four streams around a norm, at the width of the stand-alone mHC configuration.
        dict(name="mhc_8192", kind="mhc", windows=32, length=256, d_model=128),
        # The row norms at the stack's activation size: as much memory traffic as a call can have.
        dict(name="norms_262144", kind="norms", rows=262144, d_model=256),
        # The model's feed-forward over 16 windows of 480 bars, fp32 weights.
        dict(name="ffn_16x480", kind="ffn", windows=16, length=480, weights="f32"),
        # Attention over short windows, bf16 weights.
        dict(name="mla_256x128", kind="mla", windows=256, length=128, heads=8, weights="bf16"),
        # Attention over the model's full window, bf16 weights (serving) and fp32 weights (a checkpoint as it is).
        dict(name="mla_64x480", kind="mla", windows=64, length=480, heads=4, weights="bf16"),
        dict(name="mla_16x480_f32", kind="mla", windows=16, length=480, heads=4, weights="f32"),
        # The model's Mamba-3 layer over a batch of windows, fp32 weights.
        dict(name="mixer_16x480", kind="mixer", windows=16, length=480, weights="f32"),
        # One bar for 16384 instruments with carried state: the state is read and written once.
        dict(name="decode_16384", kind="decode", streams=16384),
        # The bf16 stack over a batch: every operator, fused as a server runs it.
        dict(name="stack_256x256", kind="stack", windows=256, length=256),
        # The whole model: one window as it arrives, and a batch of them as in a backtest.
        dict(name="model_1x480", kind="model", windows=1, length=480, depth=4),
        dict(name="model_32x480", kind="model", windows=32, length=480, depth=4),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["block", "mhc", "norms", "ffn", "mla", "mixer", "decode", "stack", "model"])
    weights = rng.choice(["f32", "bf16"])
    if kind == "block":
        return dict(kind=kind, windows=_log_int(rng, 1, 1024), length=rng.randint(4, 100))
    if kind == "norms":
        return dict(kind=kind, rows=_log_int(rng, 64, 262144), d_model=rng.choice([64, 128, 256]))
    if kind == "decode":
        return dict(kind=kind, streams=_log_int(rng, 16, 16384))
    length = rng.choice([rng.randint(16, 128), rng.randint(129, 256), rng.randint(257, 480)])
    if kind == "mhc":
        return dict(kind=kind, windows=_log_int(rng, 1, 64), length=length, d_model=rng.choice([64, 128, 256]))
    if kind == "ffn":
        return dict(kind=kind, windows=_log_int(rng, 1, 64), length=length, weights=weights)
    if kind == "mla":
        return dict(kind=kind, windows=_log_int(rng, 1, 64), length=length, heads=rng.choice([4, 8]), weights=weights)
    if kind == "mixer":
        return dict(kind=kind, windows=_log_int(rng, 1, 64), length=length, weights=weights)
    if kind == "stack":
        return dict(kind=kind, windows=_log_int(rng, 1, 128), length=length)
    return dict(kind=kind, windows=_log_int(rng, 1, 16), length=length, depth=rng.randint(1, 4))


# --------------------------------------------------------------- modules and inputs


def _mla_config(heads):
    g = _MLA[heads]
    return SimpleNamespace(d_model=heads * g["head_dim"], n_heads=heads, head_dim=g["head_dim"],
                           nope_head_dim=g["head_dim"] - g["rope"], rope_head_dim=g["rope"], kv_lora_rank=_KV_RANK,
                           q_lora_rank=0, rope_theta=10000.0, dropout=0.0)


def _model_config():
    model = dict(d_model=256, n_heads=4, head_dim=64, rope_head_dim=32, nope_head_dim=32, kv_lora_rank=_KV_RANK,
                 ffn_hidden=_FFN_HIDDEN, n_prelude=0, n_coda=0, core_type="two_stage", stage1_mamba_layers=5,
                 stage2_attn_layers=1, recurrent_steps=4, recurrent_drift_mode="mhc", mhc_n_streams=4,
                 mhc_sinkhorn_iters=20, mamba_d_state=64, mamba_headdim=64, mamba_expand=2, use_official_mamba=True,
                 use_morphological_rope=False, max_seq_len=480)
    return {"model": model, "horizons_minutes": [15, 60, 240]}


class _Residual(torch.nn.Module):
    """One hyper-connection around a norm, as the mHC sub-layers call it."""

    def __init__(self, d_model):
        super().__init__()
        self.hc = rdt.ManifoldHyperConnectionHIP(d_model, 4, 20)
        self.norm = rdt.RMSNormHIP(d_model)

    def forward(self, streams):
        return self.hc(streams, self.norm)


class _Norms(torch.nn.Module):
    def __init__(self, d_model):
        super().__init__()
        self.rms = rdt.RMSNormHIP(d_model)
        self.layer = rdt.LayerNormHIP(d_model)

    def forward(self, x):
        return self.rms(x), self.layer(x)


def _module(case):
    kind = case["kind"]
    if kind == "block":
        return rdt.Mamba3BlockHIP(**_SHORT)
    if kind == "mhc":
        return _Residual(case["d_model"])
    if kind == "norms":
        return _Norms(case["d_model"])
    if kind == "ffn":
        return rdt.SwiGLUHIP(256, _FFN_HIDDEN)
    if kind == "mla":
        return rdt.MLAHIP(_mla_config(case["heads"]))
    if kind == "mixer":
        return rdt.Mamba3HIP(**_MODEL)
    if kind == "decode":
        return rdt.DecodeStackHIP(n_layers=2, **_DECODE)
    if kind == "stack":
        return HybridStackHIP(_STACK_FEATURES)
    return rdt.RDT4QuantHIP(_FEATURES, _model_config())


def _as_trained(module, generator):
    """Norm weights off one, data-dependent mHC mixing, biases off zero: what a trained checkpoint has."""
    for name, p in module.named_parameters():
        if "norm" in name.lower() and p.dim() == 1 or name.endswith(("rms.weight", "layer.weight", "layer.bias")):
            p.add_(0.1 * torch.randn(p.shape, generator=generator))
        elif name.endswith(("pre_alpha", "post_alpha", "res_alpha")):
            p.fill_(0.7)
        elif name.endswith(("pre_proj.weight", "post_proj.weight", "res_proj.weight")):
            p.normal_(0.0, p.shape[1] ** -0.5, generator=generator)
        elif name.endswith(("res_bias", "pre_bias", "post_bias")):
            p.add_(0.5 * torch.randn(p.shape, generator=generator))
        elif name.endswith(("B_bias", "C_bias", ".D")):
            p.add_(0.2 * torch.randn(p.shape, generator=generator))


def _built(case, seed):
    with torch.random.fork_rng(devices=[]), torch.no_grad():
        torch.manual_seed(seed)
        generator = torch.Generator().manual_seed(seed)
        module = _module(case).eval()
        _as_trained(module, generator)
        linears = [m for m in module.modules() if isinstance(m, torch.nn.Linear)]
        if case["kind"] == "stack":  # bf16 GEMM weights N(0, 0.02); the hyper-connections' projections stay fp32
            linears = [m for m in linears if any(m.weight is w for w in module.linear_weights())]
            for m in linears:
                m.weight.normal_(0.0, 0.02, generator=generator)
        if case["kind"] == "stack" or case.get("weights") == "bf16":
            for m in linears:
                m.weight.data = m.weight.data.to(_BF16)
        return module.to(DEV)


def prepare(case, seed):
    kind = case["kind"]
    module = _built(case, seed)
    generator = torch.Generator(DEV).manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, device=DEV, generator=generator)

    state = dict(kind=kind, module=module)
    if kind == "block":
        state["x"] = normal(case["windows"], case["length"], 64)
    elif kind == "mhc":
        state["x"] = normal(case["windows"], case["length"], 4, case["d_model"])
    elif kind == "norms":
        state["x"] = normal(case["rows"], case["d_model"])
    elif kind in ("ffn", "mla", "mixer"):
        state["x"] = normal(case["windows"], case["length"], 256)
    elif kind == "decode":
        state["x"] = normal(case["streams"], _DECODE["d_model"])
        state["states"] = module.new_state(case["streams"], DEV)
        for s in state["states"]:  # a stream that has been running
            for key in ("ssm", "k", "v"):
                s[key].normal_(0.0, 0.1, generator=generator)
            s["angle"].uniform_(0.0, 2 * math.pi, generator=generator)
            s["started"] = True
    elif kind == "stack":
        state["x"] = normal(case["windows"], case["length"], _STACK_FEATURES).clamp_(-8.0, 8.0)
    else:
        state["x"] = normal(case["windows"], case["length"], _FEATURES).clamp_(-8.0, 8.0)
        state["depth"] = case["depth"]
    return state


def run(state):
    module, x = state["module"], state["x"]
    with torch.no_grad():
        if state["kind"] == "decode":
            out = module.step(x, state["states"])
            return {"out": out, "states": [[s["ssm"], s["k"], s["v"], s["angle"]] for s in state["states"]]}
        if state["kind"] == "model":
            return module(x, state["depth"])
        return module(x)


# --------------------------------------------------------------- the same in float64


def _lin(x, layer):
    y = x @ layer.weight.double().t()
    return y if layer.bias is None else y + layer.bias.double()


def _rms64(x, norm, groups=1):
    g = x.reshape(*x.shape[:-1], groups, -1)
    g = g * torch.rsqrt(g.square().mean(-1, keepdim=True) + norm.eps)
    return g.reshape(x.shape) * norm.weight.double()


def _ln64(x, norm):
    return F.layer_norm(x, x.shape[-1:], norm.weight.double(), norm.bias.double(), norm.eps)


def _swiglu64(x, m):
    gate, up = _lin(x, m.w_in).chunk(2, dim=-1)
    return _lin(F.silu(gate) * up, m.w_down)


def _mixer64(m, x, carried=None):
    """The Mamba-3 layer token by token; ``carried`` (ssm, k, v, angle) continues running streams."""
    B, L, _ = x.shape
    H, N, D, R = m.nheads, m.d_state, m.headdim, m.num_rope_angles
    z, v, b, c, dt, a, trap, ang = torch.split(_lin(x, m.in_proj), [m.d_inner, m.d_inner, N, N, H, H, H, R], dim=-1)
    k = _rms64(b, m.B_norm).unsqueeze(2) + m.B_bias.double().view(H, N)
    q = _rms64(c, m.C_norm).unsqueeze(2) + m.C_bias.double().view(H, N)
    dt = F.softplus(dt + m.dt_bias.double())
    alpha = torch.exp(-(a.clamp_min(0) + 1 / (1 - a.clamp_max(0))).clamp_min(m.A_floor) * dt)
    trap = torch.sigmoid(trap)
    beta, gamma = (1 - trap) * dt * alpha, trap * dt
    phase = torch.cumsum(torch.tanh(ang).unsqueeze(2) * math.pi * dt.unsqueeze(-1), dim=1)
    if carried is not None:
        phase = phase + carried[3].unsqueeze(1)
    cos, sin = torch.cos(phase), torch.sin(phase)

    def rotate(t):
        pairs = t[..., :2 * R].unflatten(-1, (R, 2))
        left, right = pairs[..., 0], pairs[..., 1]
        turned = torch.stack((left * cos - right * sin, left * sin + right * cos), -1).flatten(-2)
        return torch.cat((turned, t[..., 2 * R:]), -1)

    q, k = rotate(q), rotate(k)
    v = v.reshape(B, L, H, D)
    if carried is None:
        s, k_prev, v_prev = x.new_zeros(B, H, N, D), x.new_zeros(B, H, N), x.new_zeros(B, H, D)
    else:
        s, k_prev, v_prev = (t.double() for t in carried[:3])
    y = torch.empty(B, L, H, D, dtype=torch.float64, device=x.device)
    for t in range(L):
        s = s * alpha[:, t, :, None, None]
        s += k_prev.unsqueeze(-1) * (beta[:, t].unsqueeze(-1) * v_prev).unsqueeze(-2)
        s += k[:, t].unsqueeze(-1) * (gamma[:, t].unsqueeze(-1) * v[:, t]).unsqueeze(-2)
        k_prev, v_prev = k[:, t], v[:, t]
        y[:, t] = (q[:, t].unsqueeze(-1) * s).sum(-2)
    y = (y + m.D.double().view(H, 1) * v).reshape(B, L, m.d_inner) * F.silu(z)
    return _lin(y, m.out_proj), [s, k_prev, v_prev, phase[:, -1]]


def _mla64(m, x):
    B, L, _ = x.shape
    H, hd, nope, rope = m.n_heads, m.head_dim, m.nope_dim, m.rope_dim
    freqs = 1.0 / (m.rope.theta ** (torch.arange(0, rope, 2, dtype=torch.float64, device=x.device) / rope))
    angles = torch.arange(L, dtype=torch.float64, device=x.device).unsqueeze(-1) * freqs
    cos, sin = torch.cat([angles, angles], -1).cos(), torch.cat([angles, angles], -1).sin()

    def turned(t):
        first, second = t.chunk(2, dim=-1)
        return t * cos + torch.cat((-second, first), -1) * sin

    q = _lin(x, m.q_proj).view(B, L, H, hd).transpose(1, 2)
    kv = _lin(_ln64(_lin(x, m.kv_down), m.kv_norm), m.kv_up).view(B, L, H, nope + hd).transpose(1, 2)
    k_rope = turned(_lin(x, m.k_rope_proj).unsqueeze(1)).expand(B, H, L, rope)
    q = torch.cat([q[..., :nope], turned(q[..., nope:])], -1)
    k = torch.cat([kv[..., :nope], k_rope], -1)
    v = kv[..., nope:].contiguous()
    hidden = torch.ones(L, L, dtype=torch.bool, device=x.device).triu(1)
    scores = torch.matmul(q.contiguous(), k.transpose(-1, -2).contiguous()) * m.scale
    out = torch.matmul(torch.softmax(scores.masked_fill_(hidden, -math.inf), -1), v)
    return _lin(out.transpose(1, 2).reshape(B, L, H * hd), m.o_proj)


def _mhc64(hc, streams, fn):
    n = hc.n_streams
    ref = _rms64(streams.mean(-2), hc.dyn_norm)
    pre = torch.sigmoid(hc.pre_bias.double() + hc.pre_alpha.double() * torch.tanh(_lin(ref, hc.pre_proj)))
    post = 2 * torch.sigmoid(hc.post_bias.double() + hc.post_alpha.double() * torch.tanh(_lin(ref, hc.post_proj)))
    dynamic = torch.tanh(_lin(ref, hc.res_proj)).view(*ref.shape[:-1], n, n)
    res = hc.res_bias.double() + hc.res_alpha.double() * dynamic
    for _ in range(max(hc.sinkhorn_iters, 1)):
        res = res - torch.logsumexp(res, -1, keepdim=True)
        res = res - torch.logsumexp(res, -2, keepdim=True)
    out = fn((pre.unsqueeze(-1) * streams).sum(-2))
    return torch.matmul(torch.exp(res), streams) + post.unsqueeze(-1) * out.unsqueeze(-2)


def _expand64(x, n):
    return x.unsqueeze(-2).expand(-1, -1, n, -1)


def _model64(m, x, depth):
    x = _ln64(_lin(x, m.projection), m.input_norm)
    for layer in m.recurrent.stage1:
        x = x + _mixer64(layer.mamba.mamba, _rms64(x, layer.mamba.norm, layer.mamba.norm.num_groups))[0]
        x = x + _swiglu64(_rms64(x, layer.ffn_norm), layer.ffn)
    streams = _expand64(x, m.recurrent.n_streams)
    layer = m.recurrent.stage2[0]
    for _ in range(depth):
        streams = _mhc64(layer.attn_hc, streams, lambda a: _mla64(layer.attn, _rms64(a, layer.attn_norm)))
        streams = _mhc64(layer.ffn_hc, streams, lambda a: _swiglu64(_rms64(a, layer.ffn_norm), layer.ffn))
    hidden = streams.mean(-2)[:, -1]
    raw = _lin(_rms64(hidden, m.final_norm), m.head).reshape(-1, m.n_horizons, 3)
    center = raw[..., 0]
    out = torch.stack((center - F.softplus(raw[..., 1]), center, center + F.softplus(raw[..., 2])), -1)
    return out, hidden.square().mean().sqrt()


def exact(case, seed):
    state = prepare(case, seed)
    kind, m, x = case["kind"], state["module"], state["x"].double()
    with torch.no_grad():
        if kind == "block":
            return x + _mixer64(m.mamba, _rms64(x, m.norm, m.norm.num_groups))[0]
        if kind == "mhc":
            return _mhc64(m.hc, x, lambda a: _rms64(a, m.norm))
        if kind == "norms":
            return _rms64(x, m.rms), _ln64(x, m.layer)
        if kind == "ffn":
            return _swiglu64(x, m)
        if kind == "mla":
            return _mla64(m, x)
        if kind == "mixer":
            return _mixer64(m, x)[0]
        if kind == "decode":
            states = []
            for layer, s in zip(m.layers, state["states"]):
                y, after = _mixer64(layer.mamba, _rms64(x, layer.norm, layer.norm.num_groups).unsqueeze(1),
                                    [s["ssm"], s["k"], s["v"], s["angle"]])
                x = x + y[:, 0]
                states.append(after)
            return {"out": _lin(_rms64(x, m.final_norm), m.head), "states": states}
        if kind == "stack":
            streams = _expand64(_lin(x, m.feature_proj), m.n_streams)
            for i, (hc, norm, mixer) in enumerate(zip(m.hcs, m.norms, m.mixers)):
                streams = _mhc64(hc, streams, lambda a: (_mla64(mixer, _rms64(a, norm)) if i % 2 else
                                                         _mixer64(mixer, _rms64(a, norm))[0]))
            return streams.mean(-2)
        return _model64(m, x, case["depth"])


# --------------------------------------------------------------- work and tolerance


def _scan_flops(tokens, heads, n, d):
    return tokens * heads * n * d * 7  # decay, two rank-1 updates and the read-out of the state


def _mixer_work(tokens, d_model, d_state, headdim, weight_bytes):
    inner = 2 * d_model
    heads = inner // headdim
    params = (2 * inner + 2 * d_state + 3 * heads + d_state // 4) * d_model + inner * d_model
    return params * weight_bytes, 2.0 * tokens * params + _scan_flops(tokens, heads, d_state, headdim)


def _mla_work(tokens, length, heads, weight_bytes):
    g = _MLA[heads]
    d, hd, rope = heads * g["head_dim"], g["head_dim"], g["rope"]
    params = (d + _KV_RANK + rope) * d + heads * (2 * hd - rope) * _KV_RANK + d * d
    return params * weight_bytes, 2.0 * tokens * params + 2.0 * tokens * (length + 1) * heads * hd


def _ffn_work(tokens, weight_bytes):
    params = 3 * 256 * _FFN_HIDDEN
    return params * weight_bytes, 2.0 * tokens * params


def _mhc_flops(tokens, d, n=4, iters=20):
    return tokens * (2.0 * d * (2 * n + n * n) + 2.0 * n * n * d + 6.0 * n * d + iters * 4 * n * n)


def work(case):
    kind = case["kind"]
    wb = 2 if case.get("weights") == "bf16" or kind == "stack" else 4
    if kind == "norms":
        values = case["rows"] * case["d_model"]
        return {"bytes": 12 * values, "flops": 11 * values}  # one read, two written
    if kind == "decode":
        s, d, n, heads = case["streams"], 128, 64, 4
        per_state = 4 * (heads * n * 64 + heads * n + heads * 64) + 8 * heads * 16
        weights, flops = _mixer_work(s, d, n, 64, 4)
        return {"bytes": 2 * (2 * s * per_state + weights) + 4 * s * (d + 1), "flops": 2 * flops + 2 * s * d}
    tokens = case["windows"] * case["length"]
    if kind == "block":
        weights, flops = _mixer_work(tokens, 64, 16, 32, 4)
        return {"bytes": weights + 8 * tokens * 64, "flops": flops}
    if kind == "mhc":
        d = case["d_model"]
        return {"bytes": 8 * tokens * 4 * d + 8 * 24 * d, "flops": _mhc_flops(tokens, d)}
    if kind == "ffn":
        weights, flops = _ffn_work(tokens, wb)
        return {"bytes": weights + 8 * tokens * 256, "flops": flops}
    if kind == "mla":
        weights, flops = _mla_work(tokens, case["length"], case["heads"], wb)
        return {"bytes": weights + 8 * tokens * 256, "flops": flops}
    mixer_w, mixer_f = _mixer_work(tokens, 256, 64, 64, wb)
    if kind == "mixer":
        return {"bytes": mixer_w + 8 * tokens * 256, "flops": mixer_f}
    mla_w, mla_f = _mla_work(tokens, case["length"], 4, wb)
    if kind == "stack":
        proj = 256 * _STACK_FEATURES
        return {"bytes": 2 * (mixer_w + mla_w) + wb * proj + 4 * tokens * (_STACK_FEATURES + 256),
                "flops": 2 * (mixer_f + mla_f) + 4 * _mhc_flops(tokens, 256) + 2.0 * tokens * proj}
    ffn_w, ffn_f = _ffn_work(tokens, wb)
    # The last step evaluates the final position alone (its keys and values need every position).
    steps = case["depth"] - 1
    keys = 2.0 * tokens * ((_KV_RANK + 32) * 256 + 4 * 96 * _KV_RANK)
    flops = (2.0 * tokens * 256 * _FEATURES + 5 * (mixer_f + ffn_f) + steps * (mla_f + ffn_f) + keys
             + (2 * steps + 1) * _mhc_flops(tokens, 256))
    return {"bytes": 5 * (mixer_w + ffn_w) + mla_w + ffn_w + 4 * tokens * _FEATURES, "flops": flops}


def tolerance(case):
    """About four times the distance from float64 (2-norm; a few times that for the worst value): 3e-3 where bf16
    weights round the activations to bf16, 6e-7 where fp32 sums run over 256 products and more, 4e-8 where the
    sums are in float64 and only the results are rounded."""
    if case["kind"] == "stack" or case.get("weights") == "bf16":
        return {"rel": 1e-2, "max": 0.1}
    if case["kind"] in ("mhc", "norms"):
        return {"rel": 1e-6, "max": 1e-5}
    if case["kind"] == "model":
        return {"rel": 1e-5, "max": 2e-4}
    return {"rel": 5e-6, "max": 1e-4}
