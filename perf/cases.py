"""The work a user of this framework has it do, as measurable cases.

Every case is one pass through public entry points of ``multiplex_amd``:

  step     one decode token per row, ``gated_delta_update``
  verify   a speculative round: outputs of the draft tokens, then the state
           after each row's accepted prefix (prepared plans, as a serving
           loop keeps them)
  prefill  the mixer's prefill from its mixed projection, ``gdn_conv_chunked``
  packed   ragged prompts packed into one ``gated_delta_update``
  mixer    a whole ``GatedDeltaNet`` layer (decode, or left-padded prompts)
  attn     a whole full-attention layer (``Attention``) over its KV cache
  mtp      the whole MTP draft head (``MTPHead``): one draft step

The GDN layers have 16 key and 32 value heads of 128 (hidden 2048); the
attention layers 16 query and 4 key/value heads of 256 (hidden 4096, MLP
12288).  Activations are bf16 and states fp32.
"""

from __future__ import annotations

import math

import torch

import multiplex_amd as mx

HK, HV, D = 16, 32, 128
KEY, VAL = HK * D, HV * D
CONV, TAPS = 2 * KEY + VAL, 4
HIDDEN = 2048
EPS = 1e-6
ATTN = dict(hidden_size=4096, num_attention_heads=16, num_key_value_heads=4, head_dim=256, intermediate_size=12288)
AH, AHQ, AHKV, AD, AI = 4096, 16, 4, 256, 12288
QKV_OUT = (2 * AHQ + 2 * AHKV) * AD
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}


def listed():
    return [
        # one user's decode: latency and launches
        {"name": "step_b1", "kind": "step", "B": 1, "dtype": "bf16"},
        # a full decode batch: the state stream
        {"name": "step_b64", "kind": "step", "B": 64, "dtype": "bf16"},
        # a speculative round of four drafts over half a batch
        {"name": "verify_b32_t4", "kind": "verify", "B": 32, "T": 4, "dtype": "bf16"},
        # the scheduler's 512-token prefill chunk, from a prefix state
        {"name": "prefill_t512", "kind": "prefill", "B": 1, "T": 512},
        # one long prompt
        {"name": "prefill_t4096", "kind": "prefill", "B": 1, "T": 4096},
        # three prompts of a continuous-batching step, from prefix states
        {"name": "packed_3", "kind": "packed", "lens": "1024,2560,7168"},
        # a GDN layer's decode step for a few users
        {"name": "mixer_decode_b8", "kind": "mixer", "B": 8, "S": 1},
        # a GDN layer on a left-padded batch of prompts of different lengths
        {"name": "mixer_prompts_b4", "kind": "mixer", "B": 4, "S": 301},
        # an attention layer's decode step for a few users at some context
        {"name": "attn_decode_b4", "kind": "attn", "B": 4, "T": 1, "L": 4000},
        # the scheduler's prefill chunk in an attention layer, over a long prefix
        {"name": "attn_chunk_t512", "kind": "attn", "B": 1, "T": 512, "L": 4096},
        # one long prompt in an attention layer
        {"name": "attn_prefill_t4096", "kind": "attn", "B": 1, "T": 4096, "L": 0},
        # a draft step of a full batch: weights and cache read once
        {"name": "mtp_step_b64", "kind": "mtp", "B": 64, "T": 1, "L": 4095},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["step", "verify", "prefill", "packed", "mixer_decode", "mixer_prompts", "attn_decode",
                       "attn_prefill", "mtp"])
    if kind == "step":
        return {"kind": "step", "B": _log(rng, 1, 64), "dtype": rng.choice(["bf16", "bf16", "f16"])}
    if kind == "verify":
        return {"kind": "verify", "B": _log(rng, 1, 32), "T": rng.randint(2, 8), "dtype": rng.choice(["bf16", "f16"])}
    if kind == "prefill":
        B = rng.choice([1, 1, 2, 3])
        return {"kind": "prefill", "B": B, "T": _log(rng, 64, 4096 // B)}
    if kind == "packed":
        n = rng.randint(2, 6)
        return {"kind": "packed", "lens": ",".join(str(_log(rng, 64, 10752 // n)) for _ in range(n))}
    if kind == "mixer_decode":
        return {"kind": "mixer", "B": _log(rng, 1, 64), "S": 1}
    if kind == "mixer_prompts":
        B = rng.choice([1, 2, 3, 4])
        return {"kind": "mixer", "B": B, "S": _log(rng, 64, 2048 // B)}
    if kind == "attn_decode":
        B = _log(rng, 1, 64)
        # one token, or the drafts of a verify
        return {"kind": "attn", "B": B, "T": rng.choice([1, 1, rng.randint(2, 8)]),
                "L": _log(rng, 128, min(16384, 64 * 4096 // B))}
    if kind == "attn_prefill":
        T = _log(rng, 32, 2048)
        return {"kind": "attn", "B": 1, "T": T, "L": rng.choice([0, _log(rng, 256, 8192 if T <= 1024 else 2048)])}
    return {"kind": "mtp", "B": _log(rng, 1, 64), "T": rng.choice([1, 1, 2]), "L": _log(rng, 64, 4000)}


# ------------------------------------------------------------------ inputs

class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)

    def n(self, *shape, dtype=torch.bfloat16, scale=1.0, mean=0.0):
        x = torch.randn(*shape, generator=self.g, device="cuda", dtype=torch.float32)
        return (x * scale + mean).to(dtype)

    def u(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(*shape, generator=self.g, device="cuda") * (hi - lo) + lo

    def i(self, lo, hi, n):
        return torch.randint(lo, hi + 1, (n,), generator=self.g, device="cuda", dtype=torch.int32)


def _unit(x):
    return x / x.norm(dim=-1, keepdim=True)


def _gdn_inputs(r, B, T, dtype, rows=None):
    q = _unit(r.n(B, T, HK, D, dtype=torch.float32)) / math.sqrt(D)
    k = _unit(r.n(B, T, HK, D, dtype=torch.float32))
    return {"q": q.to(dtype), "k": k.to(dtype), "v": r.n(B, T, HV, D, dtype=dtype), "a": r.n(B, T, HV, dtype=dtype),
            "b": r.n(B, T, HV, dtype=dtype), "A_log": r.u(HV, hi=math.log(16.0)), "dt_bias": r.u(HV, lo=-1.0),
            "state": r.n(rows or B, HV, D, D, dtype=torch.float32, scale=0.02)}


def _prefill_inputs(r, B, T):
    return {"qkv": r.n(B, T, CONV), "w": r.n(CONV, TAPS, scale=0.1), "a": r.n(B, T, HV), "b": r.n(B, T, HV),
            "A_log": r.u(HV, hi=math.log(16.0)), "dt_bias": r.u(HV, lo=-1.0),
            "state": r.n(B, HV, D, D, dtype=torch.float32, scale=0.02), "conv": r.n(B, TAPS - 1, CONV)}


def _mixer_inputs(r, B, S):
    m = mx.GatedDeltaNet(HIDDEN, HK, HV, D, D, device="cuda")
    with torch.no_grad():
        for lin in (m.in_proj_qkv, m.in_proj_z, m.in_proj_b, m.in_proj_a, m.out_proj):
            lin.weight.copy_(r.n(*lin.weight.shape, scale=lin.weight.shape[1] ** -0.5))
        m.conv1d_weight.copy_(r.n(CONV, TAPS, scale=0.1))
        m.A_log.copy_(r.u(HV, hi=math.log(16.0)))
        m.dt_bias.copy_(r.u(HV, lo=-1.0))
        m.norm_weight.copy_(r.n(D, scale=0.1, mean=1.0))
    m.requires_grad_(False)
    s = {"mixer": m, "x": r.n(B, S, HIDDEN), "conv": r.n(B, TAPS - 1, CONV),
         "state": r.n(B, HV, D, D, dtype=torch.float32, scale=0.02), "mask": None}
    if B > 1 and S > 1:  # prompts of different lengths, padded on the left; the first is the longest
        pad = r.i(0, S // 2, B)
        pad[0] = 0
        s["mask"] = torch.arange(S, device="cuda")[None, :] >= pad[:, None]
    return s


def _noisy_norms(r, module):
    for name, p in module.named_parameters():
        if p.dim() == 1:
            p.copy_(r.n(*p.shape, dtype=p.dtype, scale=0.1, mean=1.0))
        else:
            p.copy_(r.n(*p.shape, scale=p.shape[1] ** -0.5))


def _filled_cache(r, cache, L):
    if L:
        for t in (cache.keys, cache.values):
            t[:, :, :L].copy_(r.n(t.shape[0], t.shape[1], L, t.shape[3]))
        cache.advance(L)
    return cache


def prepare(case, seed):
    kind, r = case["kind"], _Rand(seed)
    with torch.no_grad():
        if kind == "step":
            return {"kind": kind, **_gdn_inputs(r, case["B"], 1, DTYPES[case["dtype"]])}
        if kind == "verify":
            B, T = case["B"], case["T"]
            s = _gdn_inputs(r, B, T, DTYPES[case["dtype"]])
            s["n"] = r.i(0, T, B)
            gates = (s["a"], s["b"], s["A_log"], s["dt_bias"], s["state"])
            verify = mx.prepare_recurrent(s["q"], s["k"], s["v"], *gates, write_state=False)
            commit = mx.prepare_recurrent(None, s["k"], s["v"], *gates, y=False, commit_len=s["n"],
                                          state_out=torch.empty_like(s["state"]))
            return {"kind": kind, **s, "verify": verify, "commit": commit}
        if kind == "prefill":
            return {"kind": kind, **_prefill_inputs(r, case["B"], case["T"])}
        if kind == "packed":
            lens = [int(n) for n in case["lens"].split(",")]
            cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32).cuda()
            return {"kind": kind, **_gdn_inputs(r, 1, sum(lens), torch.bfloat16, rows=len(lens)), "cu": cu,
                    "longest": max(lens)}
        if kind == "mixer":
            return {"kind": kind, **_mixer_inputs(r, case["B"], case["S"])}
        B, T, L = case["B"], case["T"], case["L"]
        args = mx.AttentionArgs(**ATTN)
        if kind == "attn":
            layer = mx.Attention(args, device="cuda")
            _noisy_norms(r, layer)
            cache = _filled_cache(r, mx.KVCache(B, AHKV, AD, L + T, "cuda"), L)
            return {"kind": kind, "layer": layer, "cache": cache, "x": r.n(B, T, AH), "L": L, "T": T}
        head = mx.MTPHead(args, n_layers=1, device="cuda")
        _noisy_norms(r, head)
        cache = head.make_cache(B, L + T)
        _filled_cache(r, cache[0], L)
        return {"kind": kind, "head": head, "cache": cache, "embed": r.n(B, T, AH), "hidden": r.n(B, T, AH), "L": L,
                "T": T}


def run(s):
    kind = s["kind"]
    if kind == "step":
        return mx.gated_delta_update(s["q"], s["k"], s["v"], s["a"], s["b"], s["A_log"], s["dt_bias"], s["state"])
    if kind == "verify":
        s["verify"].launch()
        s["commit"].launch()
        return s["verify"].outputs[0], s["commit"].outputs[1]
    if kind == "prefill":
        return mx.gdn_conv_chunked(s["qkv"], s["w"], HK, HV, D, D, s["a"], s["b"], s["A_log"], s["dt_bias"],
                                   s["state"], s["conv"], eps=EPS)
    if kind == "packed":
        return mx.gated_delta_update(s["q"], s["k"], s["v"], s["a"], s["b"], s["A_log"], s["dt_bias"], s["state"],
                                     cu_seqlens=s["cu"], max_seqlen=s["longest"])
    if kind == "mixer":
        cache = mx.ArraysCache(2)
        cache[0], cache[1] = s["conv"], s["state"]
        out = s["mixer"](s["x"], s["mask"], cache)
        return out, cache[0], cache[1]
    L, T = s["L"], s["T"]
    if kind == "attn":
        cache = s["cache"]
        out = s["layer"](s["x"], cache)
        cache.trim(T)  # the drafter's rollback: the next pass starts from the same prefix
    else:
        out = s["head"](s["embed"], s["hidden"], s["cache"])
        s["head"].trim_cache_to(s["cache"], L)
        cache = s["cache"][0]
    return out, cache.keys[:, :, L:L + T], cache.values[:, :, L:L + T]


# -------------------------------------------------------------------- work

def _attn_work(B, T, L):
    """An attention layer: its weights, activations and cache once; its
    projections and each query's visible keys."""
    kv = 2 * 2 * B * AHKV * AD
    pairs = B * (T * L + T * (T + 1) // 2)
    return {"bytes": 2 * (QKV_OUT * AH + AHQ * AD * AH) + 2 * 2 * B * T * AH + kv * (L + T),
            "flops": 2 * B * T * AH * (QKV_OUT + AHQ * AD) + 4 * AHQ * AD * pairs}


def work(case):
    kind = case["kind"]
    state = 4 * HV * D * D
    per_tok = 2 * (2 * KEY + 2 * VAL + 2 * HV)  # q, k, v, y, a, b
    # two products with the state and one update per token
    rec = 6 * HV * D * D
    # a 64-token chunk in the WY form: K K^T and Q K^T, the triangular
    # inverse, X_K, X_Q, U = T R, P U, the update
    chunk = HV * (2 * (2 * 64 * 64 * D) + 64 ** 3 // 3 + 3 * (2 * 64 * D * D) + 2 * (2 * 64 * 64 * D))
    if kind == "step":
        return {"bytes": case["B"] * (2 * state + per_tok), "flops": case["B"] * rec}
    if kind == "verify":
        return {"bytes": case["B"] * (2 * state + case["T"] * per_tok), "flops": case["B"] * case["T"] * rec}
    if kind == "prefill":
        B, T = case["B"], case["T"]
        return {"bytes": B * (2 * state + T * 2 * (CONV + VAL + 2 * HV) + 2 * 2 * 3 * CONV) + 2 * CONV * TAPS,
                "flops": B * (-(-T // 64) * chunk + 2 * TAPS * CONV * T)}
    if kind == "packed":
        lens = [int(n) for n in case["lens"].split(",")]
        return {"bytes": len(lens) * 2 * state + sum(lens) * per_tok, "flops": sum(-(-n // 64) for n in lens) * chunk}
    if kind == "mixer":
        B, S = case["B"], case["S"]
        n_in = CONV + VAL + 2 * HV
        gdn = B * (-(-S // 64) * chunk if S >= 64 else S * rec)
        return {"bytes": 2 * HIDDEN * (n_in + VAL) + 2 * 2 * B * S * HIDDEN + B * (2 * state + 2 * 2 * 3 * CONV),
                "flops": 2 * B * S * HIDDEN * (n_in + VAL) + gdn}
    w = _attn_work(case["B"], case["T"], case["L"])
    if kind == "mtp":
        rows, weights = case["B"] * case["T"], 2 * AH * AH + 3 * AI * AH
        w = {"bytes": w["bytes"] + 2 * weights + 2 * rows * AH, "flops": w["flops"] + 2 * rows * weights}
    return w


def tolerance(case):
    """About four times the error of a pass against :func:`exact` (bf16 y
    1.7e-3, f16 y 2.1e-4; 3.3e-3 where q, k and v are rounded too, 4.4e-3 to
    5.9e-3 for the layers), which 16-bit outputs and intermediates give."""
    if case.get("dtype") == "f16":
        return {"rel": 8e-4}
    return {"rel": {"step": 7e-3, "verify": 7e-3, "prefill": 1.3e-2, "packed": 7e-3, "mixer": 2.4e-2, "attn": 1.8e-2,
                    "mtp": 1.9e-2}[case["kind"]]}


# ------------------------------------------------------------------- exact

def _gdn_exact(q, k, v, a, b, A_log, dt_bias, S, mask=None):
    """The recurrence in 64 bits, token by token: (y, every state's last)."""
    q, k, v, a, b, S = (x.double() for x in (q, k, v, a, b, S))
    g = torch.exp(-torch.exp(A_log.double()) * torch.nn.functional.softplus(a + dt_bias.double()))
    beta = torch.sigmoid(b)
    if mask is not None:
        g = torch.where(mask[..., None], g, torch.ones_like(g))
        beta = beta * mask[..., None]
    rep = HV // HK
    q, k = q.repeat_interleave(rep, dim=2), k.repeat_interleave(rep, dim=2)
    y = torch.empty_like(v)
    states = []
    for t in range(v.shape[1]):
        S = S * g[:, t, :, None, None]
        kt = k[:, t, :, None, :]
        delta = (v[:, t] - (S * kt).sum(-1)) * beta[:, t, :, None]
        S = S + delta[..., None] * kt
        y[:, t] = (S * q[:, t, :, None, :]).sum(-1)
        if v.shape[1] <= 8:
            states.append(S)
    if mask is not None:
        y = y * mask[..., None, None]
    return y, S, states


def _conv_exact(qkv, w, conv, mask=None):
    x, w = qkv.double(), w.double()
    if mask is not None:
        x = torch.where(mask[..., None], x, torch.zeros_like(x))
    x = torch.cat([conv.double(), x], dim=1)
    T = qkv.shape[1]
    o = torch.nn.functional.silu(sum(w[:, i] * x[:, i:i + T] for i in range(TAPS)))
    B = qkv.shape[0]
    q, k, v = o[..., :KEY].reshape(B, T, HK, D), o[..., KEY:2 * KEY].reshape(B, T, HK, D), o[..., 2 * KEY:]

    def rms(z):
        return z * torch.rsqrt(z.square().mean(-1, keepdim=True) + EPS)

    return rms(q) / D, rms(k) / math.sqrt(D), v.reshape(B, T, HV, D), x[:, T:]


def _mixer_exact(s):
    m = s["mixer"]
    x = s["x"].double()
    qkv, z, b, a = (x @ lin.weight.double().T for lin in (m.in_proj_qkv, m.in_proj_z, m.in_proj_b, m.in_proj_a))
    q, k, v, conv = _conv_exact(qkv, m.conv1d_weight, s["conv"], s["mask"])
    y, S, _ = _gdn_exact(q, k, v, a, b, m.A_log, m.dt_bias, s["state"], s["mask"])
    n = y * torch.rsqrt(y.square().mean(-1, keepdim=True) + EPS) * m.norm_weight.double()
    n = n * torch.nn.functional.silu(z.reshape(n.shape))
    return n.flatten(2) @ m.out_proj.weight.double().T, conv, S


def _rms_exact(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _attn_exact(layer, x, cache, L):
    B, T, _ = x.shape
    rot = layer.args.rot
    qkv = x @ layer.qkv_proj.double().T
    qg = qkv[..., :2 * AHQ * AD].reshape(B, T, AHQ, 2 * AD)
    kv = qkv[..., 2 * AHQ * AD:].reshape(B, T, 2 * AHKV, AD)
    q = _rms_exact(qg[..., :AD], layer.q_norm.weight)
    k = _rms_exact(kv[:, :, :AHKV], layer.k_norm.weight)
    pos = torch.arange(L, L + T, device="cuda", dtype=torch.float64)
    ang = pos[:, None] * layer.args.rope_theta ** (-torch.arange(rot // 2, device="cuda", dtype=torch.float64) * 2 / rot)
    cs, sn = ang.cos()[None, :, None], ang.sin()[None, :, None]

    def rope(z):
        lo, hi = z[..., :rot // 2], z[..., rot // 2:rot]
        return torch.cat([lo * cs - hi * sn, hi * cs + lo * sn, z[..., rot:]], dim=-1)

    q, k, v = rope(q), rope(k).transpose(1, 2), kv[:, :, AHKV:].transpose(1, 2)
    out = torch.empty(B, T, AHQ, AD, device="cuda", dtype=torch.float64)
    seen = torch.arange(L + T, device="cuda")[None, :] <= torch.arange(L, L + T, device="cuda")[:, None]
    g = AHQ // AHKV
    for b in range(B):
        for h in range(AHKV):
            K = torch.cat([cache.keys[b, h, :L].double(), k[b, h]])
            V = torch.cat([cache.values[b, h, :L].double(), v[b, h]])
            for i in range(h * g, (h + 1) * g):
                p = (q[b, :, i] @ K.T) * AD ** -0.5
                out[b, :, i] = torch.softmax(p.masked_fill(~seen, -math.inf), dim=-1) @ V
    out = out * torch.sigmoid(qg[..., AD:])
    return out.flatten(2) @ layer.o_proj.double().T, k, v


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    with torch.no_grad():
        if kind in ("step", "verify"):
            y, S, states = _gdn_exact(s["q"], s["k"], s["v"], s["a"], s["b"], s["A_log"], s["dt_bias"], s["state"])
            if kind == "step":
                return y, S
            every = torch.stack([s["state"].double()] + states, dim=1)
            return y, every[torch.arange(case["B"], device="cuda"), s["n"].long()]
        if kind == "prefill":
            q, k, v, conv = _conv_exact(s["qkv"], s["w"], s["conv"])
            y, S, _ = _gdn_exact(q, k, v, s["a"], s["b"], s["A_log"], s["dt_bias"], s["state"])
            return y, S, conv
        if kind == "packed":
            ys, Ss, at = [], [], 0
            for i, n in enumerate(int(x) for x in case["lens"].split(",")):
                part = [s[t][:, at:at + n] for t in ("q", "k", "v", "a", "b")]
                y, S, _ = _gdn_exact(*part, s["A_log"], s["dt_bias"], s["state"][i:i + 1])
                ys.append(y)
                Ss.append(S)
                at += n
            return torch.cat(ys, dim=1), torch.cat(Ss)
        if kind == "mixer":
            return _mixer_exact(s)
        L = case["L"]
        if kind == "attn":
            return _attn_exact(s["layer"], s["x"].double(), s["cache"], L)
        h = s["head"]
        eh = torch.cat([_rms_exact(s["embed"].double(), h.pre_fc_norm_embedding.weight),
                        _rms_exact(s["hidden"].double(), h.pre_fc_norm_hidden.weight)], dim=-1)
        x = eh @ h.fc.double().T
        layer = h.layers[0]
        o, k, v = _attn_exact(layer.self_attn, _rms_exact(x, layer.input_layernorm.weight), s["cache"][0], L)
        x = x + o
        gu = _rms_exact(x, layer.post_attention_layernorm.weight) @ layer.mlp.gate_up_proj.double().T
        x = x + (torch.nn.functional.silu(gu[..., :AI]) * gu[..., AI:]) @ layer.mlp.down_proj.double().T
        return _rms_exact(x, h.norm.weight), k, v
