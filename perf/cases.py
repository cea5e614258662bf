"""Workloads of the decider forward: what a user of this package has it compute.

Each case is one call (or one model forward) through the package's public entry
points, over the sizes a decision service meets: requests of a few hundred to
8192 tokens, alone, in padded batches or packed with ``cu_seqlens``; the
decider-2b shape (16 linear heads of 128, 16/4 attention heads of 128, hidden
2048) and the reference launcher's 8/2 heads of 256.

    listed()              the fixed cases
    draw(rng)             one more case of the same ranges
    prepare(case, seed)   inputs, weights and engines a program holds before the call
    run(state)            one pass; returns its outputs
    work(case)            bytes and flops the pass cannot do without
    tolerance(case)       how far another correct implementation may be
    exact(case, seed)     the outputs in 64 bits, by plain torch
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

DEV = "cuda"
EPS = 1e-6
LETTERS = 10


def listed():
    return [
        # one short request's attention (a one-question prompt): the smallest call, launch-bound
        {"name": "gqa_short", "kind": "gqa", "batch": 1, "lens": "", "T": 190, "hq": 16, "hkv": 4, "d": 128, "gated": False},
        # the attention layer's call at the service's standard bucket, output gate applied in the store
        {"name": "gqa_2048_gated", "kind": "gqa", "batch": 1, "lens": "", "T": 2048, "hq": 16, "hkv": 4, "d": 128, "gated": True},
        # four requests of unequal length packed into one row, as the batcher forms them
        {"name": "gqa_packed", "kind": "gqa", "batch": 1, "lens": "4177,611,8002,301", "T": 13091, "hq": 16, "hkv": 4, "d": 128, "gated": True},
        # the reference launcher's own geometry: two requests, 8/2 heads of 256
        {"name": "gqa_d256", "kind": "gqa", "batch": 2, "lens": "", "T": 2048, "hq": 8, "hkv": 2, "d": 256, "gated": False},
        # the delta rule of a linear-attention layer with its gated norm, standard bucket
        {"name": "delta_2048", "kind": "delta", "batch": 1, "lens": "", "T": 2048, "hk": 16, "hv": 16, "norm": True, "state": False},
        # the same over packed requests
        {"name": "delta_packed", "kind": "delta", "batch": 1, "lens": "4177,611,8002,301", "T": 13091, "hk": 16, "hv": 16, "norm": True, "state": False},
        # a padded batch continued from and into fp32 states, q/k normalised by the caller,
        # two value heads per key head, fp32 beta: transformers' own signature
        {"name": "delta_states", "kind": "delta", "batch": 4, "lens": "", "T": 500, "hk": 8, "hv": 16, "norm": False, "state": True},
        # conv + SiLU into q/k/v and the gate projection of one layer, read in place from the wide projection
        {"name": "conv_gates_2048", "kind": "conv", "batch": 1, "lens": "", "T": 2048},
        # the same over packed requests (windows restart at every request)
        {"name": "conv_gates_packed", "kind": "conv", "batch": 1, "lens": "4177,611,8002,301", "T": 13091},
        # residual add + RMSNorm of a padded batch of four
        {"name": "add_rmsnorm", "kind": "norm", "batch": 4, "T": 2048, "width": 2048},
        # two short requests packed through the model layer by layer, no graph (a shape seen once)
        {"name": "forward_short", "kind": "forward", "layers": 4, "vocab": 4096, "lens": "301,97", "T": 398, "graph": False},
        # the whole decider forward at the standard bucket, replayed from the engine's graph
        {"name": "forward_2048", "kind": "forward", "layers": 28, "vocab": 65536, "lens": "", "T": 2048, "graph": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gqa", "gqa", "delta", "delta", "conv", "norm", "forward"])
    if kind == "norm":
        return {"kind": "norm", "batch": rng.randint(1, 6), "T": _log_int(rng, 40, 2048),
                "width": rng.choice([1024, 2048, 2048, 2560, 4096])}
    if kind == "forward":
        T = _log_int(rng, 100, 2048)
        cut = rng.randint(1, T - 1)
        return {"kind": "forward", "layers": 4, "vocab": 4096, "lens": rng.choice(["", f"{cut},{T - cut}"]), "T": T,
                "graph": False}
    packed = rng.random() < 0.4
    batch, lens, T = 1, "", 0
    if packed:
        parts = [_log_int(rng, 16, 4096) for _ in range(rng.randint(2, 6))]
        lens, T = ",".join(map(str, parts)), sum(parts)
    else:
        T = _log_int(rng, 33, 8192)
        batch = rng.randint(1, max(1, min(6, 8192 // T)))
    if kind == "gqa":
        hq, hkv, d = rng.choice([(16, 4, 128), (16, 4, 128), (8, 2, 256), (16, 4, 64), (8, 8, 128)])
        return {"kind": "gqa", "batch": batch, "lens": lens, "T": T, "hq": hq, "hkv": hkv, "d": d,
                "gated": rng.random() < 0.5}
    if kind == "delta":
        hk, hv = rng.choice([(16, 16), (16, 16), (8, 16), (4, 8)])
        return {"kind": "delta", "batch": batch, "lens": lens, "T": T, "hk": hk, "hv": hv,
                "norm": rng.random() < 0.5, "state": rng.random() < 0.5}
    return {"kind": "conv", "batch": batch, "lens": lens, "T": T}


# ---------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(gen, *shape, std=1.0, dtype=torch.bfloat16):
    return (torch.randn(shape, generator=gen, device=DEV) * std).to(dtype)


def _lens(case):
    return [int(s) for s in case["lens"].split(",")] if case.get("lens") else []


def _cu(case):
    lens = _lens(case)
    if not lens:
        return None, 0
    ends = [0]
    for n in lens:
        ends.append(ends[-1] + n)
    return torch.tensor(ends, dtype=torch.int32, device=DEV), max(lens)


def _spans(case):
    """(row, start, end) of every request."""
    lens = _lens(case)
    if not lens:
        return [(b, 0, case["T"]) for b in range(case.get("batch", 1))]
    out, at = [], 0
    for n in lens:
        out.append((0, at, at + n))
        at += n
    return out


def _decay_params(gen, heads):
    """A_log and dt_bias as such layers are initialised: A in U(1, 16), steps log-uniform in [0.001, 0.1]."""
    a = torch.empty(heads, device=DEV).uniform_(1.0, 16.0, generator=gen)
    dt = torch.exp(torch.empty(heads, device=DEV).uniform_(math.log(1e-3), math.log(1e-1), generator=gen))
    return torch.log(a), dt + torch.log(-torch.expm1(-dt))


def _gqa_inputs(case, seed):
    gen = _gen(seed)
    B, T, hq, hkv, d = case["batch"], case["T"], case["hq"], case["hkv"], case["d"]
    q = _normal(gen, B, T, hq, d).transpose(1, 2)          # token-major, as the prologue leaves them
    k = _normal(gen, B, T, hkv, d).transpose(1, 2)
    # v and the gate are views of the layer's combined projection output
    proj = _normal(gen, B, T, hq * 2 * d + 2 * hkv * d)
    v = proj[..., hq * 2 * d + hkv * d:].unflatten(-1, (hkv, d)).transpose(1, 2)
    gate = proj[..., :hq * 2 * d].unflatten(-1, (hq, 2 * d))[..., d:].transpose(1, 2) if case["gated"] else None
    return q, k, v, gate


def _delta_inputs(case, seed):
    gen = _gen(seed)
    B, T, hk, hv = case["batch"], case["T"], case["hk"], case["hv"]
    q, k = (F.silu(_normal(gen, B, T, hk, 128, dtype=torch.float32)) for _ in range(2))
    if not case["norm"]:
        q, k = (t * torch.rsqrt((t * t).sum(-1, keepdim=True) + EPS) for t in (q, k))
    q, k = q.to(torch.bfloat16), k.to(torch.bfloat16)
    v = F.silu(_normal(gen, B, T, hv, 128, dtype=torch.float32)).to(torch.bfloat16)
    a_log, dt_bias = _decay_params(gen, hv)
    g = -torch.exp(a_log) * F.softplus(_normal(gen, B, T, hv, dtype=torch.float32) + dt_bias)
    beta = torch.sigmoid(_normal(gen, B, T, hv, dtype=torch.float32))
    beta = beta.to(torch.float32 if case["state"] else torch.bfloat16)
    z = w = s0 = None
    if case["norm"]:
        proj = _normal(gen, B, T, (2 * hk + 2 * hv) * 128)   # q|k|v|z of the layer; z is read in place
        z = proj[..., (2 * hk + hv) * 128:].unflatten(-1, (hv, 128))
        w = 1.0 + _normal(gen, 128, std=0.02)
    if case["state"]:
        n = len(_lens(case)) or B
        s0 = _normal(gen, n, hv, 128, 128, std=0.1, dtype=torch.float32)
    return q, k, v, g, beta, z, w, s0


def _conv_inputs(case, seed):
    gen = _gen(seed)
    B, T = case["batch"], case["T"]
    proj = _normal(gen, B, T, 8192, std=0.9)                 # q|k|v|z: the conv reads the first 6144
    weight = _normal(gen, 6144, 1, 4, std=0.25)
    hidden = _normal(gen, B, T, 2048)
    gate_weight = _normal(gen, 32, 2048, std=0.02)
    a_log, dt_bias = (t.to(torch.bfloat16) for t in _decay_params(gen, 16))
    return proj, weight, hidden, gate_weight, a_log, dt_bias


def _norm_inputs(case, seed):
    gen = _gen(seed)
    B, T, W = case["batch"], case["T"], case["width"]
    return _normal(gen, B, T, W), _normal(gen, B, T, W, std=2.0), _normal(gen, W, std=0.02)


def _forward_weights(case, seed):
    """A decider's parameters by name: N(0, 0.02) matrices, gains near one, decays as above."""
    gen = _gen(seed)
    H, I = 2048, 6144
    w = {"letters": (LETTERS, H), "core.embed_tokens.weight": (case["vocab"], H), "core.norm.weight": (H,)}
    for i in range(case["layers"]):
        p = f"core.layers.{i}."
        w.update({p + "input_layernorm.weight": (H,), p + "post_attention_layernorm.weight": (H,),
                  p + "mlp.gate_proj.weight": (I, H), p + "mlp.up_proj.weight": (I, H), p + "mlp.down_proj.weight": (H, I)})
        if i % 4 == 3:
            p += "self_attn."
            w.update({p + "q_proj.weight": (4096, H), p + "k_proj.weight": (512, H), p + "v_proj.weight": (512, H),
                      p + "o_proj.weight": (H, 2048), p + "q_norm.weight": (128,), p + "k_norm.weight": (128,)})
        else:
            p += "linear_attn."
            w.update({p + "in_proj_qkv.weight": (6144, H), p + "in_proj_z.weight": (2048, H),
                      p + "in_proj_b.weight": (16, H), p + "in_proj_a.weight": (16, H),
                      p + "conv1d.weight": (6144, 1, 4), p + "norm.weight": (128,), p + "out_proj.weight": (H, 2048)})
    out = {}
    for name, shape in w.items():
        out[name] = _normal(gen, *shape, std=0.25 if "conv1d" in name else 0.02)
        if name.endswith("linear_attn.norm.weight"):
            out[name] = 1.0 + out[name]
    for i in range(case["layers"]):
        if i % 4 != 3:
            p = f"core.layers.{i}.linear_attn."
            out[p + "A_log"], out[p + "dt_bias"] = (t.to(torch.bfloat16) for t in _decay_params(gen, 16))
    ids = torch.randint(0, case["vocab"], (1, case["T"]), generator=gen, device=DEV)
    return out, ids


# ---------------------------------------------------------------- the calls

def prepare(case, seed):
    kind = case["kind"]
    cu, longest = _cu(case) if kind in ("gqa", "delta", "conv", "forward") else (None, 0)
    s = {"kind": kind, "cu": cu, "longest": longest}
    if kind == "gqa":
        s["in"] = _gqa_inputs(case, seed)
    elif kind == "delta":
        s["in"] = _delta_inputs(case, seed)
        s["state"] = case["state"]
    elif kind == "conv":
        s["in"] = _conv_inputs(case, seed)
    elif kind == "norm":
        s["in"] = _norm_inputs(case, seed)
    else:
        from dataclasses import replace
        from fastdecisions_amd.engine import Engine
        from fastdecisions_amd.model import DECIDER_2B_SHAPED, build_decider, install_hip_kernels
        shape = replace(DECIDER_2B_SHAPED, num_hidden_layers=case["layers"], vocab_size=case["vocab"])
        weights, ids = _forward_weights(case, seed)
        model = build_decider(shape, seed=0, device=DEV)
        with torch.no_grad():
            params = dict(model.named_parameters())
            assert set(params) == set(weights)
            for name, p in params.items():
                p.copy_(weights[name])
        install_hip_kernels(model)
        s["model"], s["ids"], s["graph"] = model, ids, case["graph"]
        s["segments"] = [(a, b) for _, a, b in _spans(case)]
        if case["graph"]:
            s["engine"] = Engine(model)
            s["engine"].logits_all(ids)                     # captures the graph of this shape
    return s


def run(s):
    kind = s["kind"]
    if kind == "gqa":
        from fastdecisions_amd.native_gqa_kernel import native_gqa_attention
        q, k, v, gate = s["in"]
        if s["cu"] is None:
            return native_gqa_attention(q, k, v, gate=gate)
        return native_gqa_attention(q, k, v, gate=gate, cu_seqlens=s["cu"], max_seqlen=s["longest"])
    if kind == "delta":
        from fastdecisions_amd.gated_delta_kernel import chunk_gated_delta_rule
        q, k, v, g, beta, z, w, s0 = s["in"]
        out, final = chunk_gated_delta_rule(q, k, v, g, beta, initial_state=s0, output_final_state=s["state"],
                                            use_qk_l2norm_in_kernel=z is not None, cu_seqlens=s["cu"],
                                            norm=None if z is None else (z, w, EPS))
        return (out, final) if s["state"] else out
    if kind == "conv":
        from fastdecisions_amd.packed_conv_kernel import prep_qkv_gates
        proj, weight, hidden, gate_weight, a_log, dt_bias = s["in"]
        return prep_qkv_gates(proj[..., :6144], weight, hidden, gate_weight, a_log, dt_bias, cu_seqlens=s["cu"])
    if kind == "norm":
        from fastdecisions_amd.persistent_residual_rms_kernel import fused_add_rms_norm
        x, residual, weight = s["in"]
        return fused_add_rms_norm(x, residual, weight, EPS)
    if s["graph"]:
        return s["engine"].logits_all(s["ids"])
    with torch.no_grad():
        if s["cu"] is None:
            return s["model"](s["ids"])
        return s["model"](s["ids"], cu_seqlens=s["cu"], segments=s["segments"], max_seqlen=s["longest"])


# ---------------------------------------------------------------- the least work

def _gqa_flops(spans, hq, d):
    return sum(4.0 * hq * d * (e - b) * (e - b + 1) / 2 for _, b, e in spans)


def _delta_flops(tokens, hv):
    # per 64-token chunk and head: k k^T, q k^T, the two products with the triangular inverse, A v',
    # three products with the state, and the solve
    return tokens / 64.0 * hv * (4 * 2 * 64 * 64 * 128 + 2 * 64 * 64 * 128 + 3 * 2 * 64 * 128 * 128 + 2 * 64 ** 3 / 6)


def work(case):
    kind = case["kind"]
    spans = _spans(case)
    n = case.get("batch", 1) * case["T"]
    if kind == "gqa":
        per = (2 + case["gated"]) * case["hq"] + 2 * case["hkv"]
        return {"bytes": 2.0 * n * per * case["d"], "flops": _gqa_flops(spans, case["hq"], case["d"])}
    if kind == "delta":
        hk, hv = case["hk"], case["hv"]
        size = n * (2 * (2 * hk + (2 + case["norm"]) * hv) * 128 + hv * (4 + (4 if case["state"] else 2)))
        if case["state"]:
            size += 2 * 4 * len(spans) * hv * 128 * 128
        return {"bytes": float(size), "flops": _delta_flops(n, hv)}
    if kind == "conv":
        return {"bytes": n * (2.0 * 2 * 6144 + 2 * 2048 + 16 * 6) + 2 * 6144 * 4 + 2 * 32 * 2048,
                "flops": n * (2.0 * 4 * 6144 + 2.0 * 32 * 2048)}
    if kind == "norm":
        return {"bytes": 2.0 * (4 * n + 1) * case["width"], "flops": 5.0 * n * case["width"]}
    H, I, L = 2048, 6144, case["layers"]
    attn = L // 4
    mlp = 3 * I * H
    params = L * mlp + attn * (5120 * H + H * 2048) + (L - attn) * (8192 * H + 32 * H + 2048 * H) + LETTERS * H
    flops = 2.0 * n * params + attn * _gqa_flops(spans, 16, 128) + (L - attn) * _delta_flops(n, 16)
    return {"bytes": 2.0 * params + n * (8 + 2 * H + 4 * LETTERS), "flops": flops}


def tolerance(case):
    """About four times the distance from the 64-bit outputs (bf16 results: 0.002 to 0.004)."""
    kind = case["kind"]
    if kind == "norm":
        return {"rel": 8e-3, "max": 0.05}
    if kind == "conv":
        return {"rel": 1e-2, "max": 0.05}
    if kind == "gqa":
        return {"rel": 1.2e-2, "max": 0.1}
    if kind == "delta":
        return {"rel": 1.5e-2, "max": 0.2}
    # bf16 roundings travel through the layers: 0.027 from the 64-bit logits after 4, 0.11 after 28
    return {"rel": 0.1 if case["layers"] <= 4 else 0.3, "max": 0.95}


# ---------------------------------------------------------------- 64-bit outputs

def _attn64(q, k, v):
    """Causal attention of one request, q [T, hq, d], k and v [T, hkv, d], float64."""
    T, hq, d = q.shape
    group = hq // k.shape[1]
    out = torch.empty_like(q)
    for h in range(hq):
        kh, vh = k[:, h // group].contiguous(), v[:, h // group].contiguous()
        for a in range(0, T, 2048):
            b = min(T, a + 2048)
            s = (q[a:b, h].contiguous() @ kh[:b].T.contiguous()) * d ** -0.5
            rows = torch.arange(a, b, device=q.device)[:, None]
            s.masked_fill_(torch.arange(b, device=q.device)[None] > rows, float("-inf"))
            out[a:b, h] = torch.softmax(s, -1) @ vh[:b]
    return out


def _delta64(q, k, v, g, beta, state):
    """Gated delta rule of one request, [T, hv, 128] inputs in float64; state [hv, 128, 128]."""
    T, hv, D = v.shape
    q, k, v = (t.transpose(0, 1).contiguous() for t in (q * D ** -0.5, k, v))
    g, beta = g.T.contiguous(), beta.T.contiguous()
    out = torch.empty_like(v)
    for a in range(0, T, 64):
        b = min(T, a + 64)
        n = b - a
        qc, kc, vc, bc = q[:, a:b], k[:, a:b], v[:, a:b], beta[:, a:b, None]
        gc = g[:, a:b].cumsum(-1)
        dec = torch.exp((gc[:, :, None] - gc[:, None, :]).tril()).tril()
        kt = kc.transpose(1, 2).contiguous()
        low = (bc * (kc @ kt) * dec).tril(-1)
        eye = torch.eye(n, dtype=v.dtype, device=v.device).expand(hv, n, n)
        rhs = bc * (vc - torch.exp(gc)[..., None] * (kc @ state))
        vn = torch.linalg.solve_triangular(eye + low, rhs, upper=False, unitriangular=True)
        out[:, a:b] = torch.exp(gc)[..., None] * (qc @ state) + ((qc @ kt) * dec) @ vn
        last = gc[:, -1]
        keep = torch.exp(last[:, None] - gc)[..., None] * vn
        state = torch.exp(last)[:, None, None] * state + kt @ keep
    return out.transpose(0, 1), state


def _unit64(t):
    return t * torch.rsqrt((t * t).sum(-1, keepdim=True) + EPS)


def _rms64(t, gain):
    return t * torch.rsqrt((t * t).mean(-1, keepdim=True) + EPS) * gain


def _conv64(x, w):
    """Causal depthwise conv + SiLU of one request, x [T, C], w [C, W]."""
    W = w.shape[1]
    y = torch.zeros_like(x)
    for j in range(W):
        back = W - 1 - j
        if back < x.shape[0]:
            y[back:] += x[:x.shape[0] - back] * w[:, j]
    return F.silu(y)


def _gates64(x, w, a_log, dt_bias):
    ab = x @ w.T.contiguous()
    heads = w.shape[0] // 2
    return -torch.exp(a_log) * F.softplus(ab[..., :heads] + dt_bias), torch.sigmoid(ab[..., heads:])


def _rope64(x, cos, sin):
    """Rotary embedding of the first cos.shape[-1] features, x [T, h, d]."""
    r = cos.shape[-1]
    a, b = x[..., :r // 2], x[..., r // 2:r]
    turned = torch.cat([-b, a], -1)
    return torch.cat([x[..., :r] * cos[:, None] + turned * sin[:, None], x[..., r:]], -1)


def _forward64(case, seed):
    w, ids = _forward_weights(case, seed)
    spans = _spans(case)
    d64 = lambda name: w[name].double()
    lin = lambda x, name: x @ d64(name).T.contiguous()
    h = w["core.embed_tokens.weight"][ids[0]].double()
    T = h.shape[0]
    pos = torch.cat([torch.arange(b - a, device=DEV) for _, a, b in spans]).double()
    inv = 1e7 ** (-torch.arange(0, 32, 2, device=DEV).double() / 32)
    angle = (pos[:, None] * inv).repeat(1, 2)
    cos, sin = angle.cos(), angle.sin()
    for i in range(case["layers"]):
        p = f"core.layers.{i}."
        x = _rms64(h, 1.0 + d64(p + "input_layernorm.weight"))
        if i % 4 == 3:
            m = p + "self_attn."
            qg = lin(x, m + "q_proj.weight").view(T, 16, 256)
            q = _rope64(_rms64(qg[..., :128], 1.0 + d64(m + "q_norm.weight")), cos, sin)
            k = _rope64(_rms64(lin(x, m + "k_proj.weight").view(T, 4, 128), 1.0 + d64(m + "k_norm.weight")), cos, sin)
            v = lin(x, m + "v_proj.weight").view(T, 4, 128)
            o = torch.cat([_attn64(q[a:b], k[a:b], v[a:b]) for _, a, b in spans])
            o = lin((o * torch.sigmoid(qg[..., 128:])).reshape(T, 2048), m + "o_proj.weight")
        else:
            m = p + "linear_attn."
            qkv = lin(x, m + "in_proj_qkv.weight")
            qkv = torch.cat([_conv64(qkv[a:b], d64(m + "conv1d.weight")[:, 0]) for _, a, b in spans])
            q, k, v = (t.reshape(T, 16, 128) for t in qkv.split(2048, -1))
            g, beta = _gates64(x, torch.cat([d64(m + "in_proj_a.weight"), d64(m + "in_proj_b.weight")]),
                               d64(m + "A_log"), d64(m + "dt_bias"))
            zero = torch.zeros(16, 128, 128, dtype=torch.float64, device=DEV)
            q, k = _unit64(q), _unit64(k)
            o = torch.cat([_delta64(q[a:b], k[a:b], v[a:b], g[a:b], beta[a:b], zero)[0] for _, a, b in spans])
            z = lin(x, m + "in_proj_z.weight").view(T, 16, 128)
            o = lin((_rms64(o, d64(m + "norm.weight")) * F.silu(z)).reshape(T, 2048), m + "out_proj.weight")
        h = h + o
        x = _rms64(h, 1.0 + d64(p + "post_attention_layernorm.weight"))
        h = h + lin(F.silu(lin(x, p + "mlp.gate_proj.weight")) * lin(x, p + "mlp.up_proj.weight"), p + "mlp.down_proj.weight")
    return lin(_rms64(h, 1.0 + d64("core.norm.weight")), "letters")[None]


def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        if kind == "gqa":
            q, k, v, gate = _gqa_inputs(case, seed)
            out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
            for r, a, b in _spans(case):
                one = [t[r, :, a:b].transpose(0, 1).double() for t in (q, k, v)]
                out[r, :, a:b] = _attn64(*one).transpose(0, 1)
            return out if gate is None else out * torch.sigmoid(gate.double())
        if kind == "delta":
            q, k, v, g, beta, z, w, s0 = _delta_inputs(case, seed)
            hv, rep = case["hv"], case["hv"] // case["hk"]
            out = torch.empty(v.shape, dtype=torch.float64, device=DEV)
            final = []
            for n, (r, a, b) in enumerate(_spans(case)):
                qk = [t[r, a:b].double().repeat_interleave(rep, 1) for t in (q, k)]
                if z is not None:
                    qk = [_unit64(t) for t in qk]
                state = torch.zeros(hv, 128, 128, dtype=torch.float64, device=DEV) if s0 is None else s0[n].double()
                out[r, a:b], state = _delta64(*qk, v[r, a:b].double(), g[r, a:b].double(), beta[r, a:b].double(), state)
                final.append(state)
            if z is not None:
                out = _rms64(out, w.double()) * F.silu(z.double())
            return (out, torch.stack(final)) if case["state"] else out
        if kind == "conv":
            proj, weight, hidden, gate_weight, a_log, dt_bias = _conv_inputs(case, seed)
            B, T = case["batch"], case["T"]
            y = torch.empty(B, T, 6144, dtype=torch.float64, device=DEV)
            for r, a, b in _spans(case):
                y[r, a:b] = _conv64(proj[r, a:b, :6144].double(), weight[:, 0].double())
            g, beta = _gates64(hidden.double(), gate_weight.double(), a_log.double(), dt_bias.double())
            return (*(t.reshape(B, T, 16, 128) for t in y.split(2048, -1)), g, beta)
        if kind == "norm":
            x, residual, weight = _norm_inputs(case, seed)
            h = x.double() + residual.double()
            return _rms64(h, 1.0 + weight.double()), h
        # 28 layers of bf16 rounding leave 0.11 between any bf16 forward and the 64-bit one: no yardstick there
        return _forward64(case, seed) if case["layers"] <= 4 else None
