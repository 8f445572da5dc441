"""Performance cases of the attention, Gated-DeltaNet and MoE blocks.

Each case is one block (or a few like blocks in a row, where one alone would
be a few microseconds) of the Qwen3.6-35B-A3B geometry, called through the
entry points that an engine calls: the per-layer mixers
(``qwen36_attn.mixers``), the MoE block (``qwen36_attn.moe``) and the packed
batched DeltaNet update (``qwen36_attn.gated_deltanet``).  One-token decode is
replayed from a HIP graph, as a decode loop runs it; prefill, whose sizes
change from call to call, is launched eagerly.

  listed()            the cases
  draw(rng)           one more case of the same ranges
  prepare(case, seed) weights, caches, states and inputs on the GPU
  run(state)          one pass; its outputs, with the state that it updates
  work(case)          bytes and operations that one pass cannot do without
  tolerance(case)     what two correct implementations may differ by
  exact(case, seed)   the same outputs in 64 bits, in plain torch
"""
from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "aima-amd395-qwen36-35b-linux-engine_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

BF16 = torch.bfloat16
HIDDEN = 2048
HQ, HKV, D = 16, 2, 256                  # gated GQA attention
HK, HV, DK, DV = 16, 32, 128, 128        # Gated DeltaNet
CONV, VALUE = 2 * HK * DK + HV * DV, HV * DV
EXPERTS, TOP_K, INTER = 256, 8, 512      # MoE block
ATTN_WEIGHTS = (9216 + 4096) * HIDDEN    # q|gate, k, v rows and o_proj
GDN_WEIGHTS = (12352 + 4096) * HIDDEN    # qkv, z, b, a rows and out_proj


def listed():
    return [
        # one token early in a chat: launches and latency, little cache to read
        {"name": "attn_decode_2k", "kind": "attn_decode", "layers": 4, "context": 2051},
        # one token at the end of a long context: the KV cache stream
        {"name": "attn_decode_128k", "kind": "attn_decode", "layers": 4, "context": 131072},
        # one token through linear-attention layers: weights and 2 MiB of state a layer
        {"name": "gdn_decode", "kind": "gdn_decode", "layers": 6},
        # one token through MoE blocks: the selected experts' weights
        {"name": "moe_decode", "kind": "moe_decode", "layers": 4},
        # the MoE block over a short turn: about three quarters of the experts, few rows each
        {"name": "moe_prefill_45", "kind": "moe_prefill", "tokens": 45},
        # ... over an ordinary prompt: every expert, about 30 rows each
        {"name": "moe_prefill_1000", "kind": "moe_prefill", "tokens": 1000},
        # ... over a full prefill block
        {"name": "moe_prefill_8192", "kind": "moe_prefill", "tokens": 8192},
        # a short new turn over a cached conversation (exact-prefix hit)
        {"name": "attn_prefill_turn", "kind": "attn_prefill", "tokens": 93, "prefix": 24000},
        # a full prefill block from an empty cache
        {"name": "attn_prefill_8192", "kind": "attn_prefill", "tokens": 8192, "prefix": 0},
        # linear attention over an ordinary, ragged prompt
        {"name": "gdn_prefill_1000", "kind": "gdn_prefill", "tokens": 1000},
        # ... over a full prefill block
        {"name": "gdn_prefill_8192", "kind": "gdn_prefill", "tokens": 8192},
        # batched one-token update of many sequences' states (vLLM's packed decode)
        {"name": "gdn_batch_48", "kind": "gdn_batch", "sequences": 48},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attn_decode", "attn_decode", "gdn_decode", "moe_decode", "moe_prefill",
                       "moe_prefill", "moe_prefill", "attn_prefill", "attn_prefill",
                       "attn_prefill", "gdn_prefill", "gdn_prefill", "gdn_batch"])
    if kind == "attn_decode":
        return {"kind": kind, "layers": rng.randint(2, 4), "context": _log_int(rng, 128, 131072)}
    if kind == "gdn_decode":
        return {"kind": kind, "layers": rng.randint(2, 12)}
    if kind == "moe_decode":
        return {"kind": kind, "layers": rng.randint(1, 4)}
    if kind == "moe_prefill":
        return {"kind": kind, "tokens": _log_int(rng, 2, 8192)}
    if kind == "attn_prefill":
        t = _log_int(rng, 8, 8192)
        # at most the pairs of the full block from an empty cache
        most = 8192 * 8193 // 2 // t - (t + 1) // 2
        prefix = 0 if rng.random() < 0.4 or most < 64 else _log_int(rng, 64, min(65536, most))
        return {"kind": kind, "tokens": t, "prefix": prefix}
    if kind == "gdn_prefill":
        return {"kind": kind, "tokens": _log_int(rng, 8, 8192)}
    return {"kind": kind, "sequences": _log_int(rng, 1, 256)}


# ---- inputs, from the seed alone ---------------------------------------------

def _gen(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * int(seed) + 17)
    return g


def _randn(g, shape, scale=1.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=BF16).mul_(scale)


def _attn_weights(g):
    return {"q_proj": _randn(g, (2 * HQ * D, HIDDEN), 0.02),
            "k_proj": _randn(g, (HKV * D, HIDDEN), 0.02),
            "v_proj": _randn(g, (HKV * D, HIDDEN), 0.02),
            "o_proj": _randn(g, (HIDDEN, HQ * D), 0.02),
            "q_norm": _randn(g, (D,), 0.02), "k_norm": _randn(g, (D,), 0.02)}


def _gdn_weights(g):
    a = torch.rand(HV, generator=g, device="cuda") * 16.0
    return {"linear_in_proj_qkv": _randn(g, (CONV, HIDDEN), 0.02),
            "linear_in_proj_z": _randn(g, (VALUE, HIDDEN), 0.02),
            "linear_in_proj_a": _randn(g, (HV, HIDDEN), 0.02),
            "linear_in_proj_b": _randn(g, (HV, HIDDEN), 0.02),
            "linear_conv1d": _randn(g, (CONV, 1, 4), 0.5),
            "linear_A_log": a.clamp_min(1e-4).log(),
            "linear_dt_bias": torch.randn(HV, generator=g, device="cuda") * 0.5,
            "linear_norm": 1.0 + _randn(g, (DV,), 0.1),
            "linear_out_proj": _randn(g, (HIDDEN, VALUE), 0.02)}


def _gdn_states(g):
    conv = _randn(g, (CONV, 3), 0.9)
    ssm = torch.randn(HV, DK, DV, generator=g, device="cuda") * 0.1
    return conv, ssm


def _moe_weights(g):
    return {"post_attention_layernorm": _randn(g, (HIDDEN,), 0.1),
            "router": _randn(g, (EXPERTS, HIDDEN), 0.05),
            "expert_gate_up": _randn(g, (EXPERTS, 2 * INTER, HIDDEN), 0.02),
            "expert_down": _randn(g, (EXPERTS, HIDDEN, INTER), 0.02),
            "shared_gate": _randn(g, (1, HIDDEN), 0.02),
            "shared_gate_proj": _randn(g, (INTER, HIDDEN), 0.02),
            "shared_up_proj": _randn(g, (INTER, HIDDEN), 0.02),
            "shared_down_proj": _randn(g, (HIDDEN, INTER), 0.02)}


def _moe_tokens(g, t):
    """Residual rows and attention outputs.  A prompt's tokens are alike, so
    its experts are loaded unevenly: each row leans towards one of 16 topics."""
    topics = _randn(g, (16, HIDDEN))
    which = torch.randint(0, 16, (t,), generator=g, device="cuda")
    return 0.4 * topics[which] + _randn(g, (t, HIDDEN)), _randn(g, (t, HIDDEN), 0.5)


def _attn_layer(case, g, tokens, start):
    """Weights, input rows and caches whose rows before ``start`` are filled."""
    w = _attn_weights(g)
    x = _randn(g, (tokens, HIDDEN))
    rows = start + tokens
    k = _randn(g, (rows, HKV, D))
    v = _randn(g, (rows, HKV, D))
    k[start:] = 0
    v[start:] = 0
    return w, x, k, v


def _batch(case, g):
    n = case["sequences"]
    mixed = _randn(g, (n, CONV), 0.9)
    a, b = _randn(g, (n, HV)), _randn(g, (n, HV))
    a_log = (torch.rand(HV, generator=g, device="cuda") * 16.0).clamp_min(1e-4).log()
    dt_bias = torch.randn(HV, generator=g, device="cuda") * 0.5
    slots = n + max(1, n // 8)           # a pool with a few free slots
    pool = torch.randn(slots, HV, DV, DK, generator=g, device="cuda") * 0.1
    index = torch.randperm(slots, generator=g, device="cuda")[:n].to(torch.int32)
    return mixed, a, b, a_log, dt_bias, pool, index


# ---- prepare and run -----------------------------------------------------------

def _graph(call):
    """``call`` captured after two eager passes, as a decode loop sets it up."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
        call()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    return {"graph": graph, "out": out}


def prepare(case, seed):
    from qwen36_attn import gated_deltanet as gd
    from qwen36_attn import mixers
    from qwen36_attn.moe import MoEBlock

    kind, g = case["kind"], _gen(case, seed)
    if kind in ("attn_decode", "attn_prefill"):
        tokens = 1 if kind == "attn_decode" else case["tokens"]
        start = case["context"] - 1 if kind == "attn_decode" else case["prefix"]
        state = mixers.MixerState("cuda")
        xs, ws = [], []
        for i in range(case.get("layers", 1)):
            w, x, k, v = _attn_layer(case, g, tokens, start)
            state.full_attention_kv_caches[i] = (k, v)
            xs.append(x)
            ws.append(w)
        caches = [state.full_attention_kv_caches[i] for i in range(len(xs))]
        state.set_position_window(start, tokens, "decode" if kind == "attn_decode" else "prefill")
        full, _ = mixers.bind(state)
        if kind == "attn_decode":
            s = _graph(lambda: [full(x, i, w) for i, (x, w) in enumerate(zip(xs, ws))])
            return {**s, "state": state, "inputs": (xs, ws), "updated": caches}
        state.fused_projection(0, "qkv", ws[0]["q_proj"], ws[0]["k_proj"], ws[0]["v_proj"])
        return {"call": lambda: full(xs[0], 0, ws[0]), "updated": caches}
    if kind in ("gdn_decode", "gdn_prefill"):
        tokens = 1 if kind == "gdn_decode" else case["tokens"]
        state = mixers.MixerState("cuda")
        xs, ws = [], []
        for i in range(case.get("layers", 1)):
            ws.append(_gdn_weights(g))
            xs.append(_randn(g, (tokens, HIDDEN)))
            state.add_linear_attention_layer(i, *_gdn_states(g))
        state.set_position_window(0, tokens, "decode" if kind == "gdn_decode" else "prefill")
        _, linear = mixers.bind(state)
        updated = [(state.linear_attention_conv_states[i], state.linear_attention_ssm_states[i])
                   for i in range(len(xs))]
        if kind == "gdn_decode":
            s = _graph(lambda: [linear(x, i, w) for i, (x, w) in enumerate(zip(xs, ws))])
            return {**s, "state": state, "inputs": (xs, ws), "updated": updated}
        w = ws[0]
        state.fused_projection(0, "qkvzba", w["linear_in_proj_qkv"], w["linear_in_proj_z"],
                               w["linear_in_proj_b"], w["linear_in_proj_a"])
        return {"call": lambda: linear(xs[0], 0, w), "updated": updated}
    if kind == "moe_decode":
        blocks, rows = [], []
        for _ in range(case["layers"]):
            blocks.append(MoEBlock(_moe_weights(g)))
            rows.append(_moe_tokens(g, 1))
        s = _graph(lambda: [b.decode(x, a) for b, (x, a) in zip(blocks, rows)])
        return {**s, "inputs": (blocks, rows), "updated": []}
    if kind == "moe_prefill":
        block = MoEBlock(_moe_weights(g))
        x, a = _moe_tokens(g, case["tokens"])
        return {"call": lambda: block.prefill(x, a), "updated": []}
    mixed, a, b, a_log, dt_bias, pool, index = _batch(case, g)
    return {"call": lambda: gd.fused_recurrent_gated_delta_rule_packed_decode(
                mixed, a, b, a_log, dt_bias, DK ** -0.5, pool, ssm_state_indices=index),
            "updated": []}


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return {"out": state["out"], "updated": state["updated"]}
    return {"out": state["call"](), "updated": state["updated"]}


# ---- work and tolerance ----------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "attn_decode":
        n, s = case["layers"], case["context"]
        # weights, the K and V rows, a few KB of rows in and out
        return {"bytes": n * (2 * ATTN_WEIGHTS + 2048 * s + 8192), "flops": n * (2 * ATTN_WEIGHTS + 16384 * s)}
    if kind == "attn_prefill":
        t, p = case["tokens"], case["prefix"]
        pairs = t * p + t * (t + 1) // 2
        return {"bytes": 2 * ATTN_WEIGHTS + 2048 * (p + t) + 2 * 2 * HIDDEN * t,
                "flops": 2 * t * ATTN_WEIGHTS + 16384 * pairs}
    if kind == "gdn_decode":
        n = case["layers"]
        state = 2 * (4 * HV * DK * DV + 2 * CONV * 3)      # read and written
        return {"bytes": n * (2 * GDN_WEIGHTS + state + 8192), "flops": n * (2 * GDN_WEIGHTS + 8 * HV * DK * DV)}
    if kind == "gdn_prefill":
        t = case["tokens"]
        state = 2 * (4 * HV * DK * DV + 2 * CONV * 3)
        # the rule itself: one decay, two products and one rank-1 update a token
        return {"bytes": 2 * GDN_WEIGHTS + state + 2 * 2 * HIDDEN * t,
                "flops": 2 * t * GDN_WEIGHTS + 8 * t * HV * DK * DV}
    expert = 3 * INTER * HIDDEN                             # gate, up and down of one expert
    router = (EXPERTS + 1) * HIDDEN
    if kind == "moe_decode":
        n = case["layers"]
        weights = router + (TOP_K + 1) * expert
        return {"bytes": n * (2 * weights + 3 * 2 * HIDDEN), "flops": n * 2 * weights}
    if kind == "moe_prefill":
        t = case["tokens"]
        # experts that at least one of the tokens selects, were they drawn evenly
        used = EXPERTS * (1.0 - (1.0 - TOP_K / EXPERTS) ** t)
        return {"bytes": 2 * (router + (used + 1) * expert) + 3 * 2 * HIDDEN * t,
                "flops": 2 * t * (router + (TOP_K + 1) * expert)}
    n = case["sequences"]
    return {"bytes": n * (2 * 4 * HV * DK * DV + 2 * CONV + 2 * VALUE), "flops": 8 * n * HV * DK * DV}


def tolerance(case):
    # About four times the error against 64 bits that each path shows (bf16
    # rows with several roundings on the way; 2-norms): attention 4.8e-3, the
    # DeltaNet layer 6.1e-3, the MoE block, whose residual rows weigh most,
    # 1.8e-3, the batched update's bf16 rows 1.7e-3.
    return {"rel": {"attn_decode": 2e-2, "attn_prefill": 2e-2, "gdn_decode": 2.4e-2,
                    "gdn_prefill": 2.4e-2, "moe_decode": 8e-3, "moe_prefill": 8e-3,
                    "gdn_batch": 7e-3}[case["kind"]]}


# ---- the same in 64 bits ----------------------------------------------------------

def _rope(x, start):
    """Rotates the first 64 dims of [T, H, 256] for positions from ``start``."""
    pos = torch.arange(start, start + x.shape[0], device=x.device, dtype=torch.float64)
    freq = 1.0e7 ** (-torch.arange(0, 64, 2, device=x.device, dtype=torch.float64) / 64.0)
    ang = (pos[:, None] * freq[None, :])[:, None, :]
    a, b = x[..., :32], x[..., 32:64]
    return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin(), x[..., 64:]], -1)


def _exact_attn(w, x, k, v, start):
    t = x.shape[0]
    x = x.double()
    w = {n: y.double() for n, y in w.items()}
    qg = (x @ w["q_proj"].t()).view(t, HQ, 2 * D)
    q, gate = qg[..., :D], qg[..., D:]

    def norm(y, weight):
        return y * torch.rsqrt(y.square().mean(-1, keepdim=True) + 1e-6) * (weight + 1.0)

    q = _rope(norm(q, w["q_norm"]), start)
    k, v = k.double(), v.double()
    k[start:] = _rope(norm((x @ w["k_proj"].t()).view(t, HKV, D), w["k_norm"]), start)
    v[start:] = (x @ w["v_proj"].t()).view(t, HKV, D)
    keys = torch.arange(k.shape[0], device="cuda")
    attn = torch.empty(t, HQ, D, device="cuda", dtype=torch.float64)
    step = max(1, (1 << 26) // k.shape[0])
    for h in range(HQ):
        kh, vh = k[:, h // (HQ // HKV)], v[:, h // (HQ // HKV)]
        for r in range(0, t, step):
            s = (q[r:r + step, h] @ kh.t()) / 16.0
            last = torch.arange(r, min(t, r + step), device="cuda") + start
            s.masked_fill_(keys[None, :] > last[:, None], -math.inf)
            attn[r:r + step, h] = torch.softmax(s, -1) @ vh
    out = (attn * torch.sigmoid(gate)).reshape(t, HQ * D) @ w["o_proj"].t()
    return out, k, v


def _silu(x):
    return x * torch.sigmoid(x)


def _unit(x):
    return x * torch.rsqrt(x.square().sum(-1, keepdim=True) + 1e-6)


def _exact_gdn(w, x, conv, ssm):
    t = x.shape[0]
    x = x.double()
    w = {n: y.double() for n, y in w.items()}
    mixed = x @ w["linear_in_proj_qkv"].t()
    z = (x @ w["linear_in_proj_z"].t()).view(t, HV, DV)
    beta = torch.sigmoid(x @ w["linear_in_proj_b"].t())
    dt = torch.nn.functional.softplus(x @ w["linear_in_proj_a"].t() + w["linear_dt_bias"])
    decay = torch.exp(-w["linear_A_log"].exp() * dt)
    full = torch.cat([conv.double().t(), mixed], 0)
    taps = w["linear_conv1d"].view(CONV, 4)
    y = _silu(sum(full[j:j + t] * taps[:, j] for j in range(4)))
    q = _unit(y[:, :HK * DK].view(t, HK, DK)).repeat_interleave(2, 1) * DK ** -0.5
    k = _unit(y[:, HK * DK:2 * HK * DK].view(t, HK, DK)).repeat_interleave(2, 1)
    v = y[:, 2 * HK * DK:].view(t, HV, DV)
    s = ssm.double().clone()
    core = torch.empty(t, HV, DV, device="cuda", dtype=torch.float64)
    for i in range(t):
        s.mul_(decay[i][:, None, None])
        delta = (v[i] - (k[i][:, None, :] @ s)[:, 0]) * beta[i][:, None]
        s.baddbmm_(k[i][:, :, None], delta[:, None, :])
        torch.matmul(q[i][:, None, :], s, out=core[i][:, None, :])
    core = core * torch.rsqrt(core.square().mean(-1, keepdim=True) + 1e-6) * w["linear_norm"]
    out = (core * _silu(z)).reshape(t, VALUE) @ w["linear_out_proj"].t()
    return out, full[t:].t().contiguous(), s


def _exact_moe(w, x, a):
    # the residual row, the normalised row and the logits are bf16 values by
    # definition: the routing is a selection among bf16 logits, ties to the
    # lower expert
    t = x.shape[0]
    after = (x.float() + a.float()).to(BF16).double()
    h2 = (after * torch.rsqrt(after.square().mean(-1, keepdim=True) + 1e-6)
          * (w["post_attention_layernorm"].double() + 1.0)).to(BF16).double()
    logits = (h2 @ w["router"].double().t()).to(BF16)
    vals, ids = torch.sort(logits.float(), dim=-1, descending=True, stable=True)
    vals, ids = vals[:, :TOP_K].double(), ids[:, :TOP_K]
    rw = torch.softmax(vals, -1)

    def expert(rows, gate, up, down):
        return (_silu(rows @ gate.double().t()) * (rows @ up.double().t())) @ down.double().t()

    moe = torch.zeros(t, HIDDEN, device="cuda", dtype=torch.float64)
    for e in torch.unique(ids).tolist():
        row, rank = torch.nonzero(ids == e, as_tuple=True)
        gu = w["expert_gate_up"][e]
        moe.index_add_(0, row, expert(h2[row], gu[:INTER], gu[INTER:], w["expert_down"][e])
                       * rw[row, rank][:, None])
    shared = expert(h2, w["shared_gate_proj"], w["shared_up_proj"], w["shared_down_proj"])
    return after + moe + torch.sigmoid(h2 @ w["shared_gate"].double().t()) * shared


def exact(case, seed):
    kind, g = case["kind"], _gen(case, seed)
    if kind in ("attn_decode", "attn_prefill"):
        tokens = 1 if kind == "attn_decode" else case["tokens"]
        start = case["context"] - 1 if kind == "attn_decode" else case["prefix"]
        outs, caches = [], []
        for _ in range(case.get("layers", 1)):
            w, x, k, v = _attn_layer(case, g, tokens, start)
            out, k, v = _exact_attn(w, x, k, v, start)
            outs.append(out)
            caches.append((k, v))
        return {"out": outs if kind == "attn_decode" else outs[0], "updated": caches}
    if kind in ("gdn_decode", "gdn_prefill"):
        tokens = 1 if kind == "gdn_decode" else case["tokens"]
        outs, states = [], []
        for _ in range(case.get("layers", 1)):
            w = _gdn_weights(g)
            x = _randn(g, (tokens, HIDDEN))
            out, conv, ssm = _exact_gdn(w, x, *_gdn_states(g))
            outs.append(out)
            states.append((conv, ssm))
        return {"out": outs if kind == "gdn_decode" else outs[0], "updated": states}
    if kind == "moe_decode":
        outs = []
        for _ in range(case["layers"]):
            w = _moe_weights(g)
            outs.append(_exact_moe(w, *_moe_tokens(g, 1)))
        return {"out": outs, "updated": []}
    if kind == "moe_prefill":
        w = _moe_weights(g)
        return {"out": _exact_moe(w, *_moe_tokens(g, case["tokens"])), "updated": []}
    mixed, a, b, a_log, dt_bias, pool, index = _batch(case, g)
    n = case["sequences"]
    mixed, index = mixed.double(), index.long()
    q = _unit(mixed[:, :HK * DK].view(n, HK, DK)).repeat_interleave(2, 1) * DK ** -0.5
    k = _unit(mixed[:, HK * DK:2 * HK * DK].view(n, HK, DK)).repeat_interleave(2, 1)
    v = mixed[:, 2 * HK * DK:].view(n, HV, DV)
    beta = torch.sigmoid(b.double())
    decay = torch.exp(-a_log.double().exp()
                      * torch.nn.functional.softplus(a.double() + dt_bias.double()))
    s = pool[index].double() * decay[:, :, None, None]            # [n, HV, dv, dk]
    delta = (v - (s * k[:, :, None, :]).sum(-1)) * beta[:, :, None]
    s = s + delta[..., None] * k[:, :, None, :]
    out = (s * q[:, :, None, :]).sum(-1)
    pool = pool.double()
    pool[index] = s
    return {"out": (out.view(n, 1, HV, DV), pool), "updated": []}
