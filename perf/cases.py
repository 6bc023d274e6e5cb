"""Workloads of the verify-and-accept library: what a decode or prefill program has it do.

Each case is a dict of plain values with a "kind"; `prepare` makes on the GPU what such a
program holds before the call (weights, caches, recurrent state, inputs, captured graphs),
`run` makes one pass through the public entry points, `exact` computes the same in 64-bit
torch. Widths are the 27B model's on one GPU (hidden 5120, DeltaNet 16 k / 48 v heads of 128,
GQA 24 q / 4 kv heads of 256, MLP 17408) or one of four ranks' share of them (4 / 12 heads,
one kv head with 6 q heads, MLP 4352).

Kinds:
  step        one verify + accept + rollback step of a 4-layer slice (3 DeltaNet, 1 GQA, each
              with its MLP), rejection sampling over 151936 logits, as a serving loop runs it:
              a graph replay on state at fixed addresses
  dn_verify   a DeltaNet layer's T-token verify from the previous step's checkpoints, and the
              conv window's rollback (deltanet::verify_from_ckpt, deltanet::conv_rollback)
  dn_decode   one decode token of B sequences through deltanet::full_batched, captured
  dn_token    one decode token of one sequence with the fp8 in-projections folded in
              (deltanet::full_fp8), captured
  gqa_verify  a GQA layer's T-token verify attention with the KV append, bf16 cache
              (gqa::tail_verify_append)
  gqa_decode  one decode token's attention tail over the static fp32 cache (gqa::tail), captured
  prefill     chunked DeltaNet prefill of a prompt (deltanet::chunked_prefill)
  mlp         gate/up + SwiGLU and down projections on M rows, fp8 weights
              (fp8::matmul_swiglu, fp8::matmul)
  accept      rejection sampling over given logits (spec::accept_rejection)
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "neuron-pytorch-native_amd")
for _p in (_PKG, os.path.join(_PKG, "kernels")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

import npn_ops  # noqa: E402,F401  (registers the torch.ops)
import spec_verify_step as svs  # noqa: E402

DEV = "cuda"
D = 128          # DeltaNet head size
DH = 256         # attention head size
HIDDEN = 5120
BF, F32, F64 = torch.bfloat16, torch.float32, torch.float64
EPS = 1e-6


def listed():
    return [
        # one user's request: the whole step at the smallest batch, where launches count
        {"name": "step_b1", "kind": "step", "B": 1, "K": 7, "kv_lo": 4096, "kv_hi": 32768},
        # the serving batch the framework's benchmark quotes
        {"name": "step_b32", "kind": "step", "B": 32, "K": 7, "kv_lo": 4096, "kv_hi": 32768},
        # plain decode (no drafts) of one sequence at full width, fp8 projections
        {"name": "dn_token", "kind": "dn_token", "hk": 16, "hv": 48},
        # plain decode of eight sequences on one of four ranks
        {"name": "dn_decode_b8", "kind": "dn_decode", "B": 8, "hk": 4, "hv": 12},
        # a DeltaNet layer's verify at a middle batch
        {"name": "dn_verify_b8", "kind": "dn_verify", "B": 8, "T": 8, "hk": 16, "hv": 48},
        # plain decode's attention of eight sequences, one rank's kv head, 4k static cache
        {"name": "gqa_decode_b8", "kind": "gqa_decode", "B": 8, "hq": 6, "S": 4096},
        # a GQA layer's verify over mixed long caches
        {"name": "gqa_verify_b16", "kind": "gqa_verify", "B": 16, "T": 8, "kv_lo": 4096,
         "kv_hi": 32768},
        # a long prompt at full width
        {"name": "prefill_48x4096", "kind": "prefill", "hv": 48, "S": 4096},
        # an ordinary prompt of ragged length on one of four ranks
        {"name": "prefill_12x1000", "kind": "prefill", "hv": 12, "S": 1000},
        # the MLP at a small verify batch (8 sequences, 4 drafts)
        {"name": "mlp_m40", "kind": "mlp", "M": 40, "inter": 17408},
        # the MLP over a prompt's rows
        {"name": "mlp_m2048", "kind": "mlp", "M": 2048, "inter": 17408},
        # acceptance alone at a middle batch
        {"name": "accept_b8", "kind": "accept", "B": 8, "K": 7, "V": 151936},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["step", "dn_verify", "dn_decode", "dn_token", "gqa_verify", "gqa_decode",
                       "gqa_decode", "prefill", "prefill", "mlp", "mlp", "accept"])
    heads = rng.choice([(16, 48), (4, 12)])
    if kind == "step":
        lo = _log_int(rng, 256, 8192)
        return {"kind": kind, "B": _log_int(rng, 1, 32), "K": rng.randint(1, 7), "kv_lo": lo,
                "kv_hi": _log_int(rng, lo, 32768)}
    if kind == "dn_verify":
        return {"kind": kind, "B": _log_int(rng, 1, 32), "T": rng.randint(2, 16), "hk": heads[0],
                "hv": heads[1]}
    if kind == "dn_decode":
        return {"kind": kind, "B": _log_int(rng, 1, 64), "hk": heads[0], "hv": heads[1]}
    if kind == "dn_token":  # any whole share of the heads, with or without grouped k heads
        hk = rng.randint(1, 16)
        return {"kind": kind, "hk": hk, "hv": hk * rng.randint(1, 3)}
    if kind == "gqa_verify":
        lo = _log_int(rng, 64, 8192)
        return {"kind": kind, "B": _log_int(rng, 1, 32), "T": rng.randint(1, 8), "kv_lo": lo,
                "kv_hi": _log_int(rng, lo, 32768)}
    if kind == "gqa_decode":
        return {"kind": kind, "B": _log_int(rng, 1, 16), "hq": rng.randint(1, 8),
                "S": _log_int(rng, 128, 16384)}
    if kind == "prefill":
        return {"kind": kind, "hv": heads[1], "S": _log_int(rng, 64, 8192)}
    if kind == "mlp":
        return {"kind": kind, "M": _log_int(rng, 1, 2048), "inter": rng.choice([17408, 4352])}
    return {"kind": kind, "B": _log_int(rng, 1, 32), "K": rng.randint(1, 7),
            "V": rng.choice([32000, 151936, 248320])}


# ---- what a program holds -------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _kv_lens(c, seed):
    """Cache lengths spread evenly over [kv_lo, kv_hi], in an order of the seed's."""
    n = c["B"]
    lens = [(c["kv_lo"] + c["kv_hi"]) // 2] if n == 1 else \
        [c["kv_lo"] + (c["kv_hi"] - c["kv_lo"]) * i // (n - 1) for i in range(n)]
    order = torch.randperm(n, generator=torch.Generator().manual_seed(seed)).tolist()
    return [lens[i] for i in order]


def _captured(fn):
    """fn's launches as a HIP graph, and the outputs that a replay writes."""
    fn()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = fn()
    return {"graph": g, "out": out}


def _dn_weights(g, hk, hv):
    qkv = (2 * hk + hv) * D
    return {"conv_weight": torch.randn(qkv, 4, generator=g, device=DEV) * 0.5,
            "conv_bias": torch.randn(qkv, generator=g, device=DEV) * 0.1,
            "A_log": torch.randn(hv, generator=g, device=DEV) * 0.5,
            "dt_bias": torch.randn(hv, generator=g, device=DEV),
            "norm_weight": torch.randn(D, generator=g, device=DEV) * 0.1 + 1.0}


def _dn_inputs(g, B, T, hk, hv):
    qkv = (2 * hk + hv) * D
    return {"mixed_qkv": torch.randn(B * T * qkv, generator=g, device=DEV).to(BF),
            "conv_state": torch.randn(B * qkv, 3, generator=g, device=DEV).to(BF),
            "a_out": torch.randn(B * T * hv, generator=g, device=DEV),
            "b_out": torch.randn(B * T * hv, generator=g, device=DEV),
            "z": torch.randn(B * T * hv, D, generator=g, device=DEV).to(BF)}


_DN_ARGS = ("mixed_qkv", "conv_state", "conv_weight", "conv_bias", "a_out", "b_out", "z", "A_log",
            "dt_bias", "norm_weight")


def prepare(case, seed):
    c, g = case, _gen(seed)
    kind = c["kind"]
    if kind == "step":
        lens = _kv_lens(c, seed)
        model = svs.VerifySlice(c["B"], c["K"], lens, max(lens) + 3 * (c["K"] + 1), seed=seed,
                                device=DEV)
        x = torch.randn(c["B"] * (c["K"] + 1), HIDDEN, generator=g, device=DEV).to(BF)
        sets = [svs.synthetic_logits(c["B"], c["K"], 151936, 2 * seed + i, DEV) for i in (0, 1)]
        model.step(x, *sets[0])
        model.make_persistent()
        s = {"model": model, "x": x, "sets": sets, "kv0": model.kv_len.clone()}
        model.capture(x, sets)
        return s
    if kind == "dn_verify":
        B, T, hv = c["B"], c["T"], c["hv"]
        s = {**_dn_weights(g, c["hk"], hv), **_dn_inputs(g, B, T, c["hk"], hv)}
        s["prev"] = torch.randn(B * T * hv * D, D, generator=g, device=DEV) * 0.02
        s["index"] = torch.randint(0, T, (B,), generator=g, device=DEV, dtype=torch.int32)
        s["accepted"] = torch.randint(0, T, (B,), generator=g, device=DEV, dtype=torch.int32)
        return s
    if kind == "dn_decode":
        s = {**_dn_weights(g, c["hk"], c["hv"]), **_dn_inputs(g, c["B"], 1, c["hk"], c["hv"])}
        s["state"] = torch.randn(c["B"] * c["hv"] * D, D, generator=g, device=DEV) * 0.1
        s.update(_captured(lambda: torch.ops.deltanet.full_batched(
            s["state"], *[s[n] for n in _DN_ARGS])))
        return s
    if kind == "dn_token":
        hk, hv = c["hk"], c["hv"]
        qkv = (2 * hk + hv) * D
        s = _dn_weights(g, hk, hv)
        s["x"] = torch.randn(1, HIDDEN, generator=g, device=DEV).to(BF)
        s["state"] = torch.randn(hv * D, D, generator=g, device=DEV) * 0.1
        s["conv_state"] = torch.randn(qkv, 3, generator=g, device=DEV).to(BF)
        s["proj"] = [t for n in (qkv, hv * D, hv, hv)
                     for t in svs.random_fp8_linear(n, HIDDEN, g, DEV)]
        s.update(_captured(lambda: torch.ops.deltanet.full_fp8(
            s["x"], s["state"], s["conv_state"], s["conv_weight"], s["conv_bias"], s["A_log"],
            s["dt_bias"], s["norm_weight"], *s["proj"])))
        return s
    if kind == "gqa_verify":
        B, T, hq, hkv = c["B"], c["T"], 24, 4
        lens = _kv_lens(c, seed)
        s_max = max(lens) + T
        cos, sin = svs.rope_tables(torch.arange(s_max, device=DEV))
        r = lambda *n: torch.randn(*n, generator=g, device=DEV)  # noqa: E731
        s = {"query": r(B, T, hq, DH).to(BF), "gate": r(B, T, hq, DH).to(BF),
             "key": r(B, T, hkv, DH).to(BF), "value": r(B, T, hkv, DH).to(BF),
             "q_norm": r(DH) * 0.1, "k_norm": r(DH) * 0.1, "cos": cos, "sin": sin,
             "cache_k": r(B, hkv, s_max, DH).to(BF), "cache_v": r(B, hkv, s_max, DH).to(BF),
             "kv_len": torch.tensor(lens, dtype=torch.int32, device=DEV)}
        return s
    if kind == "gqa_decode":
        B, hq, S = c["B"], c["hq"], c["S"]
        r = lambda *n: torch.randn(*n, generator=g, device=DEV)  # noqa: E731
        valid = S - S // 4  # the rows decoded so far of the static cache
        cos, sin = svs.rope_tables(torch.tensor([valid - 1], device=DEV))
        mask = (torch.arange(S, device=DEV) < valid).float().reshape(1, S).contiguous()
        s = {"query": r(B * hq, DH), "gate": r(B * hq, DH), "q_norm": r(1, DH) * 0.1,
             "cos": cos, "sin": sin, "cached_k": r(B * S, DH), "cached_v": r(B * S, DH),
             "mask": mask}
        args = [s[n] for n in ("query", "gate", "q_norm", "cos", "sin", "cached_k", "cached_v",
                               "mask")]
        s.update(_captured(lambda: torch.ops.gqa.tail(*args)))
        return s
    if kind == "prefill":
        hv, S = c["hv"], c["S"]
        r = lambda *n: torch.randn(*n, generator=g, device=DEV)  # noqa: E731
        i = torch.arange(64, device=DEV)
        return {"state": r(hv * D, D) * 0.02, "q": r(hv * S, D), "k": r(hv * S, D),
                "v": r(hv * S, D), "g": -torch.nn.functional.softplus(r(hv * S, 1)),
                "beta": torch.sigmoid(r(hv * S, 1)),
                "const": [(i[:, None] >= i).float(), (i[:, None] > i).float(),
                          torch.eye(64, device=DEV)]}
    if kind == "mlp":
        return {"x": torch.randn(c["M"], HIDDEN, generator=g, device=DEV).to(BF),
                "gate_up": svs.random_fp8_linear(2 * c["inter"], HIDDEN, g, DEV),
                "down": svs.random_fp8_linear(HIDDEN, c["inter"], g, DEV)}
    return {"args": svs.synthetic_logits(c["B"], c["K"], c["V"], seed, DEV)}


def run(state):
    s = state
    if "model" in s:
        # the batch's sequences start this step from the same cache lengths every time
        s["model"].kv_len.copy_(s["kv0"])
        m = s["model"]
        hidden, accepted, ids = m.replay()
        dn = [L for L in m.layers if L["kind"] == "D"]
        return {"hidden": hidden, "accepted": accepted, "ids": ids, "kv_len": m.kv_len,
                "ckpt": [L["ckbuf"][m.parity] for L in dn], "conv": [L["conv_state"] for L in dn]}
    if "graph" in s:
        s["graph"].replay()
        return s["out"]
    if "prev" in s:
        ckpt, out = torch.ops.deltanet.verify_from_ckpt(s["prev"], s["index"],
                                                        *[s[n] for n in _DN_ARGS])
        conv = torch.ops.deltanet.conv_rollback(s["mixed_qkv"], s["conv_state"], s["accepted"],
                                                s["A_log"].numel())
        return {"ckpt": ckpt, "out": out, "conv": conv}
    if "cache_k" in s:
        out = torch.ops.gqa.tail_verify_append(
            s["query"], s["gate"], s["key"], s["value"], s["q_norm"], s["k_norm"], s["cos"],
            s["sin"], s["cache_k"], s["cache_v"], s["kv_len"])
        return {"out": out, "cache_k": s["cache_k"], "cache_v": s["cache_v"]}
    if "const" in s:
        return torch.ops.deltanet.chunked_prefill(s["state"], s["q"], s["k"], s["v"], s["g"],
                                                  s["beta"], *s["const"])
    if "gate_up" in s:
        act = torch.ops.fp8.matmul_swiglu(s["x"], *s["gate_up"])
        return torch.ops.fp8.matmul(act, *s["down"])
    return torch.ops.spec.accept_rejection(*s["args"])


# ---- what a pass cannot do without ----------------------------------------------------------

def _dn_work(B, T, hk, hv):
    """One state read, T checkpoints written, the token vectors, the conv window in and out."""
    qkv = (2 * hk + hv) * D
    return (4 * D * D * hv * B * (1 + T) + 2 * B * T * qkv + 8 * B * T * hv
            + 4 * B * T * hv * D + 12 * B * qkv + 20 * qkv), 8.0 * D * D * hv * B * T


def _gqa_work(B, T, hq, hkv, rows):
    """`rows`: cache rows read over all sequences."""
    return (rows * hkv * DH * 4 + 6 * B * T * hq * DH + 8 * B * T * hkv * DH,
            4.0 * T * hq * DH * rows)


def _gemm_work(M, K, N):
    return K * N + 4 * N + 2 * M * (K + N), 2.0 * M * K * N


def work(case):
    c = case
    kind = c["kind"]
    if kind == "step":
        B, T = c["B"], c["K"] + 1
        M, V = B * T, 151936
        lens = _kv_lens(c, 0)
        parts = [_dn_work(B, T, 16, 48)] * 3
        parts += [_gqa_work(B, T, 24, 4, sum(lens) + B * T)]
        parts += [_gemm_work(M, HIDDEN, svs.DN_IN_N), _gemm_work(M, svs.DN_VAL, HIDDEN)] * 3
        parts += [_gemm_work(M, HIDDEN, 14336), _gemm_work(M, 6144, HIDDEN)]
        parts += [_gemm_work(M, HIDDEN, 2 * svs.INTER), _gemm_work(M, svs.INTER, HIDDEN)] * 4
        parts += [((2 * T - 1 + 2) * B * V * 4, 0.0)]
    elif kind == "dn_verify":
        parts = [_dn_work(c["B"], c["T"], c["hk"], c["hv"])]
    elif kind == "dn_decode":
        parts = [_dn_work(c["B"], 1, c["hk"], c["hv"])]
    elif kind == "dn_token":
        hk, hv = c["hk"], c["hv"]
        parts = [_dn_work(1, 1, hk, hv)]
        parts += [_gemm_work(1, HIDDEN, n) for n in ((2 * hk + hv) * D, hv * D, hv, hv)]
    elif kind == "gqa_verify":
        parts = [_gqa_work(c["B"], c["T"], 24, 4, sum(_kv_lens(c, 0)) + c["B"] * c["T"])]
    elif kind == "gqa_decode":
        B, hq, S = c["B"], c["hq"], c["S"]
        parts = [(8 * B * S * DH + 12 * B * hq * DH + 4 * S, 4.0 * B * hq * S * DH)]
    elif kind == "prefill":
        hv, S = c["hv"], c["S"]
        # the chunked form with 64-token chunks (A and q k^T over 128, the substitution, k S and
        # q S, T Z and the intra product, k^T v_new); q, k, v and out once, the state both ways
        parts = [(hv * S * (4 * D * 4 + 8) + 8 * hv * D * D, hv * S / 64 * 8488320.0)]
    elif kind == "mlp":
        parts = [_gemm_work(c["M"], HIDDEN, 2 * c["inter"]),
                 _gemm_work(c["M"], c["inter"], HIDDEN)]
    else:
        B, K, V = c["B"], c["K"], c["V"]
        parts = [((2 * K + 3) * B * V * 4, 0.0)]
    return {"bytes": float(sum(p[0] for p in parts)), "flops": float(sum(p[1] for p in parts))}


def tolerance(case):
    kind = case["kind"]
    if kind == "accept":
        return "exact"
    if kind == "step":  # bf16 residual stream through eight sublayers (1.4e-2 from 64 bits,
        # which rounds nothing in between); the decisions, on given logits, are exact
        return {"rel": 2e-2, "max": 0.3}
    if kind == "prefill":  # fp32 results, products of values split over two bf16: 7e-6
        return {"rel": 3e-5, "max": 3e-3}
    if kind == "gqa_decode":  # fp32 throughout, 1.3e-6 from 64 bits
        return {"rel": 5e-6, "max": 2e-4}
    # bf16 results: a rounding that falls the other way is one unit in the last place (2^-8
    # of a value's own size), in the MLP through the second projection too
    return {"rel": 4e-3, "max": 6e-2}


# ---- the same in 64 bits --------------------------------------------------------------------

def _fp8_mm(x, w, scale):
    return (x.to(F64) @ w.view(torch.float8_e4m3fn).to(F32).to(F64)) * scale.reshape(-1).to(F64)


def _silu(x):
    return x * torch.sigmoid(x)


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _rope(x, cos, sin):
    """Rotary on x[..., :64]; cos, sin broadcast against it."""
    r = x[..., :64]
    rot = torch.cat([-r[..., 32:], r[..., :32]], -1)
    return torch.cat([r * cos + rot * sin, x[..., 64:]], -1)


def _dn_exact(state, w, mixed, conv, a, b, z, hk):
    """state [B, Hv, D, D], mixed [B, T, QKV], conv [B, QKV, 3], a, b [B, T, Hv],
    z [B, T, Hv, D] -> checkpoints [B, T, Hv, D, D], outputs [B, T, Hv, D]."""
    S = state.to(F64)
    B, T = mixed.shape[:2]
    hv = S.shape[1]
    seq = torch.cat([conv.to(F64), mixed.to(F64).transpose(1, 2)], -1)
    decay = torch.exp(-torch.exp(w["A_log"].to(F64))
                      * torch.nn.functional.softplus(a.to(F64) + w["dt_bias"].to(F64)))
    beta = torch.sigmoid(b.to(F64))
    cks, outs = [], []
    for t in range(T):
        y = _silu((seq[:, :, t:t + 4] * w["conv_weight"].to(F64)).sum(-1)
                  + w["conv_bias"].to(F64))
        q, k, v = y.split([hk * D, hk * D, hv * D], 1)
        unit = lambda u: u * torch.rsqrt((u * u).sum(-1, keepdim=True) + EPS)  # noqa: E731
        q = unit(q.reshape(B, hk, D)).repeat_interleave(hv // hk, 1) / math.sqrt(D)
        k = unit(k.reshape(B, hk, D)).repeat_interleave(hv // hk, 1)
        S = S * decay[:, t, :, None, None]
        delta = (v.reshape(B, hv, D) - (S * k[..., None]).sum(2)) * beta[:, t, :, None]
        S = S + k[..., None] * delta[:, :, None, :]
        o = (S * q[..., None]).sum(2)
        cks.append(S)
        outs.append(_rms(o, w["norm_weight"].to(F64)) * _silu(z[:, t].to(F64)))
    return torch.stack(cks, 1), torch.stack(outs, 1)


def _gqa_exact(query, gate, key, value, q_norm, k_norm, cos, sin, cache_k, cache_v, kv_len):
    B, T, hq, _ = query.shape
    hkv = cache_k.shape[1]
    out = []
    for b in range(B):
        n = int(kv_len[b])
        c, s = cos[n:n + T, None].to(F64), sin[n:n + T, None].to(F64)
        q = _rope(_rms(query[b].to(F64), 1 + q_norm.to(F64)), c, s)
        # the cache holds bf16: the norm and the rotation are each rounded to it
        kn = _rms(key[b].to(F64), 1 + k_norm.to(F64)).to(BF).to(F64)
        kn = _rope(kn, c, s).to(BF).to(F64)
        see = torch.arange(n + T, device=DEV)[None, :] <= n + torch.arange(T, device=DEV)[:, None]
        heads = []
        for h in range(hkv):
            kk = torch.cat([cache_k[b, h, :n].to(F64), kn[:, h]])
            vv = torch.cat([cache_v[b, h, :n].to(F64), value[b, :, h].to(F64)])
            grp = hq // hkv
            qq = q[:, h * grp:(h + 1) * grp].reshape(T * grp, DH)
            a = (qq @ kk.t()) / 16.0
            a = a.masked_fill(~see.repeat_interleave(grp, 0), -math.inf).softmax(-1)
            heads.append((a @ vv).reshape(T, grp, DH))
        out.append(torch.cat(heads, 1) * torch.sigmoid(gate[b].to(F64)))
    return torch.stack(out)


def _mlp_exact(x, gate_up, down):
    gu = _fp8_mm(x, *gate_up)
    n = gu.shape[1] // 2
    return _fp8_mm(_silu(gu[:, :n]) * gu[:, n:], *down)


def _step_exact(s):
    """The hidden state of the first replay after prepare()."""
    m = s["model"]
    B, T, hk, hv = m.B, m.T, svs.DN_HK, svs.DN_HV
    h = s["x"].to(F64)
    for L in m.layers:
        y = _rms(h, 1 + L["in_norm"].to(F64))
        if L["kind"] == "D":
            qkv, z, a, b, _ = _fp8_mm(y, *L["in_proj"]).split(
                [svs.DN_QKV, svs.DN_VAL, hv, hv, svs.DN_IN_PAD - svs.DN_IN_N], 1)
            w = {"A_log": L["A_log"], "dt_bias": L["dt_bias"], "norm_weight": L["norm_w"],
                 "conv_weight": L["conv_w"], "conv_bias": L["conv_b"]}
            ck = L["ckbuf"][0].reshape(B, T, hv, D, D)
            state = torch.stack([ck[i, int(m.prev_accepted[i])] for i in range(B)])
            _, o = _dn_exact(state, w, qkv.reshape(B, T, -1), L["conv_state"].reshape(B, -1, 3),
                             a.reshape(B, T, hv), b.reshape(B, T, hv), z.reshape(B, T, hv, D), hk)
            h = h + _fp8_mm(o.reshape(B * T, -1), *L["out_proj"])
        else:
            p = _fp8_mm(y, *L["qkv_proj"])
            qg, k, v = p.split([svs.GQA_QG, svs.GQA_HKV * DH, svs.GQA_HKV * DH], 1)
            qg = qg.reshape(B, T, svs.GQA_HQ, 2, DH)
            o = _gqa_exact(qg[..., 0, :], qg[..., 1, :], k.reshape(B, T, svs.GQA_HKV, DH),
                           v.reshape(B, T, svs.GQA_HKV, DH), L["q_norm"], L["k_norm"], m.rope_cos,
                           m.rope_sin, L["cache_k"], L["cache_v"], s["kv0"])
            h = h + _fp8_mm(o.reshape(B * T, -1), *L["o_proj"])
        h = h + _mlp_exact(_rms(h, 1 + L["post_norm"].to(F64)), L["gate_up"], L["down"])
    return h


def exact(case, seed):
    c = case
    kind = c["kind"]
    if kind == "accept":  # whole numbers
        return None
    s = prepare(c, seed)
    if kind == "step":
        return {"hidden": _step_exact(s)}
    if kind == "gqa_verify":
        return {"out": _gqa_exact(*[s[n] for n in (
            "query", "gate", "key", "value", "q_norm", "k_norm", "cos", "sin", "cache_k",
            "cache_v", "kv_len")])}
    if kind == "mlp":
        return _mlp_exact(s["x"], s["gate_up"], s["down"])
    if kind == "gqa_decode":
        B, hq, S = c["B"], c["hq"], c["S"]
        q = _rope(_rms(s["query"].to(F64), 1 + s["q_norm"].to(F64)), s["cos"].to(F64),
                  s["sin"].to(F64)).reshape(B, hq, DH)
        k = s["cached_k"].to(F64).reshape(B, S, DH)
        v = s["cached_v"].to(F64).reshape(B, S, DH)
        a = torch.stack([q[b] @ k[b].t() for b in range(B)]) / 16.0
        a = (a - (1 - s["mask"].to(F64)) * 1e9).softmax(-1)
        o = torch.stack([a[b] @ v[b] for b in range(B)]).reshape(B * hq, DH)
        return o * torch.sigmoid(s["gate"].to(F64))
    if kind == "prefill":
        hv, S = c["hv"], c["S"]
        f = lambda t: t.to(F64).reshape(hv, S, -1)  # noqa: E731
        q, k, v, decay, beta = f(s["q"]), f(s["k"]), f(s["v"]), f(s["g"]).exp(), f(s["beta"])
        unit = lambda u: u * torch.rsqrt((u * u).sum(-1, keepdim=True) + EPS)  # noqa: E731
        q, k = unit(q) / math.sqrt(D), unit(k)
        St = s["state"].to(F64).reshape(hv, D, D)
        out = torch.empty(hv, S, D, dtype=F64, device=DEV)
        for t in range(S):
            St = St * decay[:, t, :, None]
            delta = (v[:, t] - (St * k[:, t, :, None]).sum(1)) * beta[:, t]
            St = St + k[:, t, :, None] * delta[:, None, :]
            out[:, t] = (St * q[:, t, :, None]).sum(1)
        return out.reshape(hv * S, D), St.reshape(hv * D, D)
    hk, hv = c["hk"], c["hv"]
    qkv = (2 * hk + hv) * D
    if kind == "dn_token":
        p = s["proj"]
        mixed = _fp8_mm(s["x"], p[0], p[1])
        z, a, b = (_fp8_mm(s["x"], p[i], p[i + 1]) for i in (2, 4, 6))
        conv = s["conv_state"]
        ck, out = _dn_exact(s["state"].reshape(1, hv, D, D), s, mixed.reshape(1, 1, qkv),
                            conv.reshape(1, qkv, 3), a.reshape(1, 1, hv), b.reshape(1, 1, hv),
                            z.reshape(1, 1, hv, D), hk)
        window = torch.cat([conv[:, 1:].to(F64), mixed.reshape(qkv, 1)], 1)
        return ck.reshape(hv * D, D), window, out.reshape(hv, D)
    B, T = c["B"], c.get("T", 1)
    mixed, conv = s["mixed_qkv"].reshape(B, T, qkv), s["conv_state"].reshape(B, qkv, 3)
    state = s["state"].reshape(B, hv, D, D) if kind == "dn_decode" else torch.stack(
        [s["prev"].reshape(B, T, hv, D, D)[i, int(s["index"][i])] for i in range(B)])
    ck, out = _dn_exact(state, s, mixed, conv, s["a_out"].reshape(B, T, hv),
                        s["b_out"].reshape(B, T, hv), s["z"].reshape(B, T, hv, D), hk)
    seq = torch.cat([conv, mixed.transpose(1, 2)], -1).to(F64)
    last = [0] * B if kind == "dn_decode" else s["accepted"].tolist()
    window = torch.stack([seq[i, :, a + 1:a + 4] for i, a in enumerate(last)]).reshape(B * qkv, 3)
    if kind == "dn_decode":
        return ck.reshape(B * hv * D, D), window, out.reshape(B * hv, D)
    return {"ckpt": ck.reshape(B * T * hv * D, D), "out": out.reshape(B * T * hv, D),
            "conv": window}
