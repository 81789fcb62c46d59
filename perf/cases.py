"""What a serving engine has this op set do, as cases that can be timed and
checked: one pass of a case is the call, or the few calls in a row, that an
engine makes at that point, through the C++ API (`_xk_torch`).

Families (the "op" of a case):

  norm     Gemma RMSNorm of the hidden states before a layer's projections
  rope     q/k RMSNorm + neox RoPE of a full-attention layer's prefill
  conv     varlen causal conv1d prefill with cached conv-state slots
  chunk    chunked gated delta rule (prefill): batches of ragged sequences,
           one prompt alone on a rank's share of the heads, a long prompt, and
           many short prompts
  stages   the same prefill driven stage by stage (cumsum, scaled K K^T,
           triangular inverse, w/u, states, outputs)
  prefill  a linear-attention layer's prefill between its projections:
           split -> conv1d -> gating -> chunked rule on views of the conv's
           output -> gated RMSNorm
  decode   the same layer's decode step (input norm, split, fused conv +
           gating + recurrent step, gated RMSNorm), replayed from a HIP graph
           as engines run it: one token for each sequence of the batch
  verify   the same layer for speculative decoding: a few draft tokens per
           sequence, conv window and per-token state slots

Gates follow the usual initialisation of these layers (A in [1, 16), dt
log-uniform in [1e-3, 0.1]): some heads forget within a few tokens and some
carry their state over thousands.
"""
import math
import random

import torch

from torch_npu_ops_amd import _xk_torch as xt

BF16 = torch.bfloat16
DEV = "cuda"
K = 128  # head dim of every linear-attention head here
WIDTH = 4  # conv taps
EPS = 1e-6

# (qk heads, v heads): 16/32 and its shares over 2, 4 and 8 ranks, and the
# other groupings of the parity tests.
HEADS = [(16, 32), (8, 16), (4, 8), (2, 4), (16, 16), (4, 4), (8, 24), (4, 16)]


def listed():
    return [
        # Prefill of a full batch: the input norm over every token.
        {"name": "norm_prefill", "op": "norm", "rows": 16384, "hidden": 4096},
        # A full-attention layer's prefill of one 8k prompt.
        {"name": "rope_prefill", "op": "rope", "tokens": 8191, "hq": 32, "hkv": 8,
         "dtype": "bf16"},
        # Conv of a full prefill batch, 8 ragged prompts, all 8192 channels.
        {"name": "conv_prefill", "op": "conv", "tokens": 16384, "seqs": 8, "dim": 8192},
        # Chunked rule of a full prefill batch on one GPU.
        {"name": "chunk_batch", "op": "chunk", "tokens": 16384, "seqs": 8, "h": 16, "hv": 32},
        # One 4k prompt on one of four ranks.
        {"name": "chunk_one", "op": "chunk", "tokens": 4096, "seqs": 1, "h": 4, "hv": 8},
        # One long prompt on one of four ranks.
        {"name": "chunk_long", "op": "chunk", "tokens": 32768, "seqs": 1, "h": 4, "hv": 8},
        # Many short prompts that arrived together.
        {"name": "chunk_short", "op": "chunk", "tokens": 6007, "seqs": 64, "h": 16, "hv": 32},
        # A caller that keeps the intermediates drives the stages itself.
        {"name": "stages", "op": "stages", "tokens": 6144, "seqs": 3, "h": 8, "hv": 16},
        # A layer's prefill of a few prompts on one of two ranks.
        {"name": "prefill_layer", "op": "prefill", "tokens": 8192, "seqs": 4, "h": 8, "hv": 16},
        # A single user's token: the smallest calls, all latency.
        {"name": "decode_1", "op": "decode", "batch": 1, "h": 16, "hv": 32},
        # A full decode batch: the states' stream.
        {"name": "decode_256", "op": "decode", "batch": 256, "h": 16, "hv": 32},
        # Speculative decoding: 3 draft tokens and the last accepted one.
        {"name": "verify_32", "op": "verify", "batch": 32, "tokens": 4, "h": 16, "hv": 32},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    op = rng.choice(["norm", "rope", "conv", "chunk", "chunk", "chunk", "stages", "prefill",
                     "prefill", "decode", "decode", "verify"])
    h, hv = rng.choice(HEADS)
    if op == "norm":
        return {"op": op, "rows": _log(rng, 64, 16384), "hidden": 8 * _log(rng, 64, 1024)}
    if op == "rope":
        hkv = rng.choice([1, 2, 4, 8])
        return {"op": op, "tokens": _log(rng, 64, 16384), "hq": hkv * rng.choice([4, 8]),
                "hkv": hkv, "dtype": rng.choice(["bf16", "bf16", "f32"])}
    if op == "conv":
        seqs = _log(rng, 1, 16)
        return {"op": op, "tokens": _log(rng, 64 * seqs, 16384), "seqs": seqs,
                "dim": 2 * h * K + hv * K}
    if op in ("chunk", "prefill"):
        seqs = _log(rng, 1, 64)
        return {"op": op, "tokens": _log(rng, 48 * seqs, 16384), "seqs": seqs, "h": h, "hv": hv}
    if op == "stages":
        seqs = _log(rng, 1, 8)
        return {"op": op, "tokens": _log(rng, 128 * seqs, 6144), "seqs": seqs, "h": h, "hv": hv}
    if op == "decode":
        return {"op": op, "batch": _log(rng, 1, 256), "h": h, "hv": hv}
    return {"op": op, "batch": _log(rng, 1, 48), "tokens": rng.randint(2, 5), "h": h, "hv": hv}


def _lengths(case):
    """Ragged sequence lengths that sum to the case's tokens (a property of
    the case, not of the seed)."""
    n, total = case["seqs"], case["tokens"]
    rng = random.Random(1000003 * n + total)
    w = [rng.uniform(0.25, 1.75) for _ in range(n)]
    lens = [max(1, int(total * x / sum(w))) for x in w]
    lens[lens.index(max(lens))] += total - sum(lens)
    return lens


def _bounds(lens):
    at = [0]
    for n in lens:
        at.append(at[-1] + n)
    return at


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def n(self, *shape, std=1.0, mean=0.0, dtype=BF16):
        x = torch.randn(*shape, generator=self.g, device=DEV, dtype=torch.float32)
        return x.mul_(std).add_(mean).to(dtype)

    def u(self, lo, hi, *shape):
        return torch.rand(*shape, generator=self.g, device=DEV) * (hi - lo) + lo

    def slots(self, n, lines):
        return torch.randperm(lines, generator=self.g, device=DEV)[:n].to(torch.int32)


def _gate_weights(r, hv):
    """A_log and dt_bias (fp32), with softplus(dt_bias) = dt."""
    a_log = torch.log(r.u(1.0, 16.0, hv))
    dt = torch.exp(r.u(math.log(1e-3), math.log(0.1), hv))
    return a_log, dt + torch.log(-torch.expm1(-dt))


def _unit(x):
    x = x.float()
    return (x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)).to(BF16)


def _cu(lens):
    return torch.tensor(_bounds(lens), dtype=torch.int32, device=DEV)


def _layer_weights(r, h, hv):
    d = 2 * h * K + hv * K
    a_log, dt_bias = _gate_weights(r, hv)
    return {"conv_w": r.n(d, WIDTH, std=0.5), "A_log": a_log, "dt_bias": dt_bias,
            "norm_w": r.n(K, std=0.1, mean=1.0)}


def _inputs(case, seed):
    r, op = _Rand(seed), case["op"]
    if op == "norm":
        return {"x": r.n(case["rows"], case["hidden"]), "w": r.n(case["hidden"], std=0.1)}
    if op == "rope":
        dt = BF16 if case["dtype"] == "bf16" else torch.float32
        t, hq, hkv = case["tokens"], case["hq"], case["hkv"]
        pos = torch.randint(0, 4096, (t,), generator=r.g, device=DEV)
        inv = 1.0 / 1e6 ** (torch.arange(0, K, 2, device=DEV, dtype=torch.float64) / K)
        f = pos[:, None].double() * inv
        return {"qkv": r.n(t, (hq + 2 * hkv) * K, dtype=dt),
                "sin": torch.cat([f.sin()] * 2, -1).to(dt),
                "cos": torch.cat([f.cos()] * 2, -1).to(dt),
                "qw": r.n(K, std=0.1, mean=1.0, dtype=dt),
                "kw": r.n(K, std=0.1, mean=1.0, dtype=dt)}
    if op == "conv":
        lens, d = _lengths(case), case["dim"]
        lines = 2 * len(lens)
        return {"x": r.n(case["tokens"], d), "w": r.n(d, WIDTH, std=0.5),
                "state": r.n(lines, d, WIDTH - 1), "slots": r.slots(len(lens), lines),
                "cu": _cu(lens), "longest": max(lens)}
    if op in ("chunk", "stages"):
        lens, t, h, hv = _lengths(case), case["tokens"], case["h"], case["hv"]
        a_log, dt_bias = _gate_weights(r, hv)
        a, b = r.n(1, t, hv, dtype=torch.float32), r.n(1, t, hv, dtype=torch.float32)
        return {"q": _unit(r.n(1, t, h, K)), "k": _unit(r.n(1, t, h, K)), "v": r.n(1, t, hv, K),
                "g": -a_log.exp() * torch.nn.functional.softplus(a + dt_bias),
                "beta": torch.sigmoid(b).to(BF16), "cu": _cu(lens),
                "h0": r.n(len(lens), hv, K, K, std=0.02, dtype=torch.float32)}
    h, hv = case["h"], case["hv"]
    d = 2 * h * K + hv * K
    s = _layer_weights(r, h, hv)
    if op == "prefill":
        lens, t = _lengths(case), case["tokens"]
        lines = 2 * len(lens)
        s.update(qkvz=r.n(t, d + hv * K), ba=r.n(t, 2 * hv),
                 conv_state=torch.zeros(lines, d, WIDTH - 1, dtype=BF16, device=DEV),
                 slots=r.slots(len(lens), lines), cu=_cu(lens), longest=max(lens),
                 h0=torch.zeros(len(lens), hv, K, K, device=DEV))
        return s
    n = case["batch"]
    if op == "decode":
        s.update(x=r.n(n, 2048), in_w=r.n(2048, std=0.1), qkvz=r.n(n, d + hv * K),
                 ba=r.n(n, 2 * hv), conv_state=r.n(n, d, WIDTH - 1),
                 ssm=r.n(n, hv, K, K, std=0.02, dtype=torch.float32), slots=r.slots(n, n))
        return s
    t = case["tokens"]
    s.update(qkvz=r.n(n * t, d + hv * K), ba=r.n(n * t, 2 * hv),
             conv_state=r.n(n, d, WIDTH - 1 + t - 1), slots=r.slots(n, n),
             ssm=r.n(n * t, hv, K, K, std=0.02, dtype=torch.float32),
             ssm_slots=r.slots(n * t, n * t).view(n, t), cu=_cu([t] * n),
             accepted=torch.randint(1, t + 1, (n,), generator=r.g, device=DEV).to(torch.int32))
    return s


# --------------------------------------------------------------------------
# the calls
# --------------------------------------------------------------------------
def _gated_norm(s, o, z):
    rows = o.reshape(-1, K)
    return xt.layer_norm_fwd(rows, s["norm_w"], s["no_bias"], EPS, z.reshape(-1, K), K, True, True)


def _decode(s):
    h, hv = s["h"], s["hv"]
    rstd, x = xt.npu_ops_gemma_rms_norm(s["x"], s["in_w"], EPS)
    qkv, z, b, a = xt.npu_fused_qkvzba_split_reshape_cat(s["qkvz"], s["ba"], h, hv, K, K)
    o = xt.npu_gdn_conv_sigmoid_gating_decode(
        qkv, s["conv_state"], s["conv_w"], s["A_log"], a, s["dt_bias"], b, s["ssm"], h, hv,
        conv_state_indices=s["slots"], ssm_state_indices=s["slots"])
    return {"x": x, "y": _gated_norm(s, o, z), "conv_state": s["conv_state"], "ssm": s["ssm"]}


def _split_heads(qkv, h, hv):
    """q, k, v as views of the conv's output, as engines hand them on."""
    t = qkv.size(0)
    q, k, v = qkv.split([h * K, h * K, hv * K], -1)
    return q.view(1, t, h, K), k.view(1, t, h, K), v.view(1, t, hv, K)


def prepare(case, seed):
    s = _inputs(case, seed)
    s.update({key: val for key, val in case.items() if key in ("op", "h", "hv", "hq", "hkv")})
    s["no_bias"] = torch.empty(0, dtype=BF16, device=DEV)
    if case["op"] != "decode":
        return s
    # The engine captures the decode step once per batch size, then replays it.
    kept = {key: s[key].clone() for key in ("conv_state", "ssm")}
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _decode(s)
    torch.cuda.current_stream().wait_stream(side)
    for key, val in kept.items():
        s[key].copy_(val)
    s["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(s["graph"]):
        s["out"] = _decode(s)
    return s


def run(s):
    op = s["op"]
    if op == "norm":
        rstd, y = xt.npu_ops_gemma_rms_norm(s["x"], s["w"], EPS)
        return {"y": y, "rstd": rstd}
    if op == "rope":
        return xt.npu_split_rmsnorm_rope(s["qkv"], s["sin"], s["cos"], s["qw"], s["kw"],
                                         s["hq"] * K, s["hkv"] * K, K, EPS)
    if op == "conv":
        y = xt.npu_causal_conv1d_update_v2(s["x"], s["state"], s["w"], True,
                                           conv_state_indices=s["slots"],
                                           query_start_loc=s["cu"], max_query_len=s["longest"])
        return {"y": y, "state": s["state"]}
    if op == "chunk":
        o, fin = xt.npu_chunk_gated_delta_rule(s["q"], s["k"], s["v"], s["g"], s["beta"],
                                               initial_state=s["h0"], output_final_state=True,
                                               cu_seqlens=s["cu"])
        return {"o": o, "final": fin}
    if op == "stages":
        gc = xt.npu_chunk_local_cumsum(s["g"], 64, s["cu"])
        a = xt.npu_chunk_scaled_dot_kkt_fwd(s["k"], s["beta"], gc, 64, s["cu"])
        ai = xt.npu_solve_tril(a, 64, s["cu"], BF16)
        w, u = xt.npu_recompute_w_u_fwd(s["k"], s["v"], s["beta"], gc, ai, s["cu"])
        h, v_new, fin = xt.npu_chunk_gated_delta_rule_fwd_h(s["k"], w, u, gc, s["h0"], True, 64,
                                                            True, s["cu"])
        o = xt.npu_chunk_fwd_o(s["q"], s["k"], v_new, h, gc, K ** -0.5, 64, s["cu"])
        return {"gc": gc, "o": o, "final": fin}
    if op == "decode":
        s["graph"].replay()
        return s["out"]
    h, hv = s["h"], s["hv"]
    qkv, z, b, a = xt.npu_fused_qkvzba_split_reshape_cat(s["qkvz"], s["ba"], h, hv, K, K)
    g, beta = xt.npu_fused_gdn_gating(s["A_log"], a, b, s["dt_bias"])
    if op == "prefill":
        qkv = xt.npu_causal_conv1d_update_v2(qkv, s["conv_state"], s["conv_w"], True,
                                             conv_state_indices=s["slots"],
                                             query_start_loc=s["cu"], max_query_len=s["longest"])
        q, k, v = _split_heads(qkv, h, hv)
        o, fin = xt.npu_chunk_gated_delta_rule(q, k, v, g, beta, initial_state=s["h0"],
                                               output_final_state=True, cu_seqlens=s["cu"],
                                               use_qk_l2norm_in_kernel=True)
        return {"y": _gated_norm(s, o, z), "conv_state": s["conv_state"], "final": fin}
    qkv = xt.npu_causal_conv1d_update_v2(qkv, s["conv_state"], s["conv_w"], True,
                                         conv_state_indices=s["slots"], query_start_loc=s["cu"],
                                         max_query_len=s["ssm_slots"].size(1),
                                         num_accepted_tokens=s["accepted"])
    q, k, v = _split_heads(qkv, h, hv)
    o, _ = xt.npu_fused_recurrent_gated_delta_rule(
        q, k, v, g, beta, initial_state=s["ssm"], inplace_final_state=True, cu_seqlens=s["cu"],
        ssm_state_indices=s["ssm_slots"], num_accepted_tokens=s["accepted"],
        use_qk_l2norm_in_kernel=True)
    return {"y": _gated_norm(s, o, z), "conv_state": s["conv_state"], "ssm": s["ssm"]}


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------
def work(case):
    op = case["op"]
    if op == "norm":
        n, m = case["rows"], case["hidden"]
        return {"bytes": 4 * n * m + 4 * n + 2 * m, "flops": 5 * n * m}
    if op == "rope":
        e = 2 if case["dtype"] == "bf16" else 4
        t, q, kv = case["tokens"], case["hq"] * K, case["hkv"] * K
        return {"bytes": e * t * (2 * (q + 2 * kv) + 2 * K), "flops": 10 * t * (q + kv)}
    if op == "conv":
        t, d, n = case["tokens"], case["dim"], case["seqs"]
        return {"bytes": 4 * t * d + 2 * d * WIDTH + 4 * n * d * (WIDTH - 1),
                "flops": (2 * WIDTH + 5) * t * d}
    h, hv = case["h"], case["hv"]
    d = 2 * h * K + hv * K
    if op in ("chunk", "stages", "prefill"):
        lens, c = _lengths(case), 64
        chunks = sum(-(-n // c) for n in lens)
        per = 3 * 2 * c * c * K + 2 * 2 * c * c * K + 3 * 2 * c * K * K + c ** 3 / 3
        flops = chunks * hv * per
        t, n = case["tokens"], case["seqs"]
        states = 2 * n * hv * K * K * 4
        if op == "prefill":
            io = 2 * t * (d + hv * K) + 4 * t * hv + 2 * t * hv * K + 4 * n * d * (WIDTH - 1)
            return {"bytes": io + states, "flops": flops + 13 * t * d}
        return {"bytes": 2 * t * d + 2 * t * hv * K + 6 * t * hv + states, "flops": flops}
    n = case["batch"]
    if op == "decode":
        return {"bytes": 4 * n * 2048 + 2 * n * (d + 2 * hv * K + 2 * hv) +
                4 * n * d * (WIDTH - 1) + 2 * d * WIDTH + 2 * n * hv * K * K * 4,
                "flops": n * hv * 7 * K * K}
    t = case["tokens"]
    return {"bytes": 2 * n * t * (d + 2 * hv * K + 2 * hv) + 4 * n * d * (WIDTH + t - 2) +
            2 * d * WIDTH + (1 + t) * n * hv * K * K * 4,
            "flops": n * t * hv * 7 * K * K}


def tolerance(case):
    """About four times the error measured against exact(): 16-bit outputs are
    off by their own rounding (1.7e-3), layers by the roundings between their
    calls too (chunk 2.9e-3, stages 3.3e-3, whole layers up to 3.8e-3)."""
    op = case["op"]
    if op == "rope" and case["dtype"] == "f32":
        return {"rel": 1e-5}
    if op in ("norm", "rope", "conv"):
        return {"rel": 7e-3}
    return {"rel": 1.5e-2 if op in ("prefill", "verify", "stages") else 1.2e-2}


# --------------------------------------------------------------------------
# the same in 64 bits
# --------------------------------------------------------------------------
def _silu(x):
    return x * torch.sigmoid(x)


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _conv(x, hist, w):
    """x [t, d], hist [d, width - 1] -> silu(conv) [t, d]."""
    full = torch.cat([hist.t(), x], 0)
    y = torch.zeros_like(x)
    for j in range(WIDTH):
        y += full[j:j + x.size(0)] * w[:, j]
    return _silu(y)


def _conv_varlen(x, state, w, slots, lens, longest):
    """Outputs and updated states of a varlen prefill: a sequence keeps its
    last width - 1 - (longest - length) inputs, history included."""
    y, new = torch.empty_like(x), state.clone()
    at = _bounds(lens)
    for i, slot in enumerate(slots.tolist()):
        xi = x[at[i]:at[i + 1]]
        y[at[i]:at[i + 1]] = _conv(xi, state[slot], w)
        keep = WIDTH - 1 - (longest - lens[i])
        if keep > 0:
            full = torch.cat([state[slot].t(), xi], 0)
            new[slot, :, :keep] = full[full.size(0) - keep:].t()
    return y, new


def _delta_rule(q, k, v, g, beta, states, lens, scale):
    """Token by token, all sequences and heads at once; a sequence that has
    ended keeps its state.  q, k [t, h, K], v [t, hv, K], g, beta [t, hv],
    states [n, hv, K, K] -> o [t, hv, K], per-token states if asked, final."""
    rep = v.size(1) // q.size(1)
    at, n = _bounds(lens), len(lens)
    order = sorted(range(n), key=lambda i: -lens[i])
    first = torch.tensor([at[i] for i in order], device=v.device)
    s = states[order]
    o = torch.empty_like(v)
    for step in range(max(lens)):
        live = sum(1 for i in order if lens[i] > step)
        tok = first[:live] + step
        qs = q[tok].repeat_interleave(rep, 1) * scale
        ks = k[tok].repeat_interleave(rep, 1)
        part = s[:live]
        part *= g[tok].exp()[..., None, None]
        vn = (v[tok] - (part * ks[..., None]).sum(-2)) * beta[tok][..., None]
        part += ks[..., None] * vn[..., None, :]
        o[tok] = (part * qs[..., None]).sum(-2)
        yield step, live, order, s
    out = torch.empty_like(s)
    out[order] = s
    yield None, o, order, out


def _delta_final(*args):
    for step, o, _, s in _delta_rule(*args):
        pass
    return o, s


def _norm64(x):
    return x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)


def _gates64(s, ba, h, hv):
    r = hv // h
    ba = ba.view(ba.size(0), h, 2, r)
    b, a = ba[:, :, 0].reshape(-1, hv), ba[:, :, 1].reshape(-1, hv)
    return -s["A_log"].exp() * torch.nn.functional.softplus(a + s["dt_bias"]), torch.sigmoid(b)


def _split64(qkvz, h, hv):
    t, r = qkvz.size(0), hv // h
    x = qkvz.view(t, h, (2 + 2 * r) * K)
    q, k, v, z = x.split([K, K, r * K, r * K], -1)
    qkv = torch.cat([q.reshape(t, -1), k.reshape(t, -1), v.reshape(t, -1)], -1)
    return qkv, z.reshape(t, hv, K)


def _heads64(qkv, h, hv):
    t = qkv.size(0)
    q, k, v = qkv.split([h * K, h * K, hv * K], -1)
    return _norm64(q.reshape(t, h, K)), _norm64(k.reshape(t, h, K)), v.reshape(t, hv, K)


def exact(case, seed):
    s = {key: val.double() if torch.is_tensor(val) and val.is_floating_point() else val
         for key, val in _inputs(case, seed).items()}
    op = case["op"]
    if op == "norm":
        rstd = torch.rsqrt((s["x"] * s["x"]).mean(-1, keepdim=True) + EPS)
        return {"y": s["x"] * rstd * (1 + s["w"]), "rstd": rstd}
    if op == "rope":
        t, hq, hkv = case["tokens"], case["hq"], case["hkv"]
        q, k, v = s["qkv"].split([hq * K, hkv * K, hkv * K], -1)

        def turn(x, w):
            x = _rms(x.reshape(t, -1, K), w)
            half = torch.cat([-x[..., K // 2:], x[..., :K // 2]], -1)
            return (x * s["cos"][:, None] + half * s["sin"][:, None]).reshape(t, -1)
        return turn(q, s["qw"]), turn(k, s["kw"]), v
    if op == "conv":
        y, state = _conv_varlen(s["x"], s["state"], s["w"], s["slots"], _lengths(case),
                                s["longest"])
        return {"y": y, "state": state}
    h, hv, scale = case["h"], case["hv"], K ** -0.5
    if op in ("chunk", "stages"):
        lens = _lengths(case)
        o, fin = _delta_final(s["q"][0], s["k"][0], s["v"][0], s["g"][0], s["beta"][0], s["h0"],
                              lens, scale)
        if op == "chunk":
            return {"o": o[None], "final": fin}
        gc, at = torch.empty_like(s["g"]), _bounds(lens)
        for i, n in enumerate(lens):
            for c in range(at[i], at[i] + n, 64):
                e = min(c + 64, at[i] + n)
                gc[0, c:e] = s["g"][0, c:e].cumsum(0)
        return {"gc": gc, "o": o[None], "final": fin}
    g, beta = _gates64(s, s["ba"], h, hv)
    qkv, z = _split64(s["qkvz"], h, hv)

    def out(o):
        return (_rms(o, s["norm_w"]) * _silu(z)).reshape(-1, K)
    if op == "prefill":
        lens = _lengths(case)
        y, state = _conv_varlen(qkv, s["conv_state"], s["conv_w"], s["slots"], lens, s["longest"])
        o, fin = _delta_final(*_heads64(y, h, hv), g, beta, s["h0"], lens, scale)
        return {"y": out(o), "conv_state": state, "final": fin}
    n = case["batch"]
    t = case.get("tokens", 1)
    slots = s["slots"].long()
    conv, ssm = s["conv_state"].clone(), s["ssm"]
    if op == "decode":
        full = torch.cat([conv[slots], qkv[..., None]], -1)
        y = _silu((full * s["conv_w"]).sum(-1))
        conv[slots] = full[..., 1:]
        o, fin = _delta_final(*_heads64(y, h, hv), g, beta, ssm[slots], [1] * n, scale)
        ssm = ssm.clone()
        ssm[slots] = fin
        return {"x": _rms(s["x"], 1 + s["in_w"]), "y": out(o), "conv_state": conv, "ssm": ssm}
    y = torch.empty_like(qkv)
    for i, slot in enumerate(slots.tolist()):
        off = int(s["accepted"][i]) - 1
        xi = qkv[i * t:(i + 1) * t]
        y[i * t:(i + 1) * t] = _conv(xi, conv[slot, :, off:off + WIDTH - 1], s["conv_w"])
        conv[slot] = torch.cat([conv[slot, :, off + 1:off + WIDTH - 1], xi.t()], -1)
    table = s["ssm_slots"].long()
    start = ssm[table.gather(1, s["accepted"].long()[:, None] - 1)[:, 0]]
    new = ssm.clone()
    for step, o, order, st in _delta_rule(*_heads64(y, h, hv), g, beta, start, [t] * n, scale):
        if step is not None:
            new[table[order, step]] = st
    return {"y": out(o), "conv_state": conv, "ssm": new}
