"""The work that a user of q35hip has it do, as cases that can be timed and compared.

A case is a dict of plain values with a "kind":

  completion   a whole model call: reset, prefill a short prompt on every row, then graph-replayed decode steps
  head         the LM head with the greedy pick over the decode step's rows
  gdn_decode   a Gated DeltaNet mixer over one token per row (norm, projections, conv, recurrence, output projection)
  gdn_prefill  a Gated DeltaNet mixer over a prompt or a chunk of one, continuing the rows' states
  attn_prefill a gated attention mixer over a prompt from position 0 (its keys and values appended to the caches)
  attn_chunk   a gated attention mixer over a chunk of a prompt that continues over the KV cache
  mlp          the second norm and the SwiGLU MLP with its neuron pushes, accumulated into the residual
  gdn_op       the chunked delta rule on bf16 q, k, v (the function that a transformers model plugs in)
  attn_op      the causal gated attention on bf16 q, k, v (the same)
  attn_decode  split-K decode attention over a bf16 KV cache

Sizes are those of the Qwen3.5-0.8B shape in q35hip.workloads.Q35Config: hidden 1024, MLP 3584, 24 layers, 16 linear
heads of 128, 8 query and 2 key heads of 256, vocabulary 151,936; int8 weights with one fp32 scale per group of 128
inputs, the MLP also with one per output row ("mlp_group" 0). A steering experiment decodes three rows (boosted, as
it is, suppressed); other programs hold one row, or up to four (eight in the head and the mixers alone).
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "duo-mech-interp_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from q35hip import layers, ops, workloads  # noqa: E402
from q35hip.model import HybridModel, mlp, mlp_weights  # noqa: E402

DEV = "cuda"
CFG = workloads.Q35Config()
H, I, V = CFG.hidden, CFG.inter, CFG.vocab
HV, DV = CFG.lin_v_heads, CFG.lin_dv
HQ, HKV, D = CFG.n_heads, CFG.n_kv, CFG.head_dim
EPS = CFG.eps
CDIM = CFG.conv_dim
GDN_N = CDIM + HV * DV + 2 * HV
ATTN_N = HQ * 2 * D + 2 * HKV * D


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the steering experiment: three rows, a chat-sized prompt, a short answer with the vector added at layer 12
        dict(name="completion_r3", kind="completion", rows=3, T=48, steps=16, mlp_group=0, steer=True),
        # one row continued, all weights in the engine's group-128 format
        dict(name="completion_r1", kind="completion", rows=1, T=21, steps=12, mlp_group=128, steer=False),
        # the logits of one decode step, five rows
        dict(name="head_r5", kind="head", rows=5),
        # the smallest call: one token of one row through one mixer, eagerly
        dict(name="gdn_decode_r1", kind="gdn_decode", rows=1),
        # a 2048-token prompt on three rows, layer by layer (the stack's prefill)
        dict(name="gdn_prefill_3x2048", kind="gdn_prefill", B=3, T=2048),
        dict(name="attn_prefill_3x2048", kind="attn_prefill", B=3, T=2048),
        dict(name="mlp_6144", kind="mlp", B=3, T=2048, mlp_group=0),
        # a chat-sized prompt through one MLP: few rows, the engine's format
        dict(name="mlp_111", kind="mlp", B=3, T=37, mlp_group=128),
        # a long prompt sent in chunks: 128 tokens more over 1500 to 1900 cached ones
        dict(name="attn_chunk_3x128", kind="attn_chunk", B=3, T=128, ctx=1900),
        # the kernels behind a transformers model's plug-in points, one long sequence
        dict(name="gdn_op_4096", kind="gdn_op", B=1, T=4096, state=False),
        dict(name="attn_op_4096", kind="attn_op", B=1, T=4096),
        # serving many long contexts: one token for each of 32 rows over 8192 keys
        dict(name="attn_decode_b32", kind="attn_decode", B=32, ctx=8192),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["completion", "head", "gdn_decode", "gdn_prefill", "attn_prefill", "mlp", "mlp", "attn_chunk",
                       "gdn_op", "attn_op", "attn_decode"])
    group = rng.choice([0, 128])
    if kind == "completion":
        return dict(kind=kind, rows=rng.randint(1, 4), T=_log(rng, 5, 64), steps=rng.randint(4, 16), mlp_group=group,
                    steer=rng.choice([True, False]))
    if kind in ("head", "gdn_decode"):
        return dict(kind=kind, rows=rng.randint(1, 8))
    if kind in ("gdn_prefill", "attn_prefill"):
        return dict(kind=kind, B=rng.randint(1, 3), T=_log(rng, 5, 2048))
    if kind == "mlp":
        return dict(kind=kind, B=rng.randint(1, 3), T=_log(rng, 3, 2048), mlp_group=group)
    if kind == "attn_chunk":
        return dict(kind=kind, B=rng.randint(1, 3), T=_log(rng, 2, 256), ctx=_log(rng, 64, 1900))
    if kind == "gdn_op":
        return dict(kind=kind, B=rng.randint(1, 2), T=_log(rng, 16, 2048), state=rng.choice([True, False]))
    if kind == "attn_op":
        return dict(kind=kind, B=rng.randint(1, 2), T=_log(rng, 16, 2896))
    return dict(kind=kind, B=_log(rng, 1, 32), ctx=_log(rng, 33, 8192))


# ---------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _q8(g, n, k, group=128):
    return workloads.quantize_int8(_randn(g, n, k) * CFG.init_std, group)


def _put(p, name, g, n, k, group=128):
    q, s = _q8(g, n, k, group)
    p[name + ".q"], p[name + ".s"], p[name] = q, s, workloads.dequantize_int8(q, s)


def _gdn_params(g):
    p = {}
    _put(p, "in_proj_qkv", g, CDIM, H)
    _put(p, "in_proj_z", g, HV * DV, H)
    _put(p, "in_proj_b", g, HV, H)
    _put(p, "in_proj_a", g, HV, H)
    _put(p, "out_proj", g, H, HV * DV)
    p["conv1d"] = _randn(g, CDIM, CFG.conv_k) * 0.3
    p["dt_bias"] = torch.ones(HV, device=DEV)
    p["A_log"] = (torch.rand(HV, generator=g, device=DEV) * 15.9 + 0.1).log()
    p["norm"] = 1.0 + 0.1 * _randn(g, DV)
    return p


def _attn_params(g):
    p = {}
    _put(p, "q_proj", g, HQ * 2 * D, H)
    _put(p, "k_proj", g, HKV * D, H)
    _put(p, "v_proj", g, HKV * D, H)
    _put(p, "o_proj", g, H, HQ * D)
    p["q_norm"], p["k_norm"] = 0.1 * _randn(g, D), 0.1 * _randn(g, D)
    return p


def _mlp_params(g, group):
    p = {}
    _put(p, "gate_proj", g, I, H, group)
    _put(p, "up_proj", g, I, H, group)
    _put(p, "down_proj", g, H, I, group)
    return p


def _model_weights(g, group):
    W = {"norm": 0.1 * _randn(g, H)}
    W["embed.q"], W["embed.s"] = _q8(g, V, H)
    for l in range(CFG.layers):
        p = _attn_params(g) if CFG.is_attention(l) else _gdn_params(g)
        p.update(_mlp_params(g, group))
        p["input_layernorm"], p["post_attention_layernorm"] = 0.1 * _randn(g, H), 0.1 * _randn(g, H)
        W.update({f"layers.{l}.{n}": t for n, t in p.items()})
    return W


def _delta_inputs(g, B, T, state):
    """q, k, v as the causal conv's SiLU leaves them, the log decays and betas of the gates."""
    silu = torch.nn.functional.silu
    q, k, v = (silu(_randn(g, B, T, HV, DV)).bfloat16() for _ in range(3))
    decay = -torch.nn.functional.softplus(_randn(g, B, T, HV))
    beta = torch.sigmoid(_randn(g, B, T, HV))
    return q, k, v, decay, beta, _randn(g, B, HV, DV, DV) * 0.1 if state else None


def _inputs(case, seed):
    g = _gen(seed)
    kind, s = case["kind"], dict(case=case)
    if kind == "completion":
        s["W"] = _model_weights(g, case["mlp_group"])
        s["prompt"] = torch.randint(0, V, (case["rows"], case["T"]), generator=g, device=DEV)
        s["ids"] = torch.randint(0, V, (case["steps"], case["rows"]), generator=g, device=DEV).int()
        s["vecs"] = _randn(g, 2, H) * 0.5 if case["steer"] else None
        s["vec_of_row"] = [(0, -1, 1)[r % 3] for r in range(case["rows"])]
    elif kind == "head":
        s["x"], s["norm"] = _randn(g, case["rows"], H) * 3, 0.1 * _randn(g, H)
        s["q"], s["s"] = _q8(g, V, H)
    elif kind in ("gdn_decode", "gdn_prefill"):
        B, T = (case["rows"], 1) if kind == "gdn_decode" else (case["B"], case["T"])
        s["p"], s["norm"] = _gdn_params(g), 0.1 * _randn(g, H)
        s["x"] = _randn(g, B, T, H) * 3
        s["conv"], s["rec"] = _randn(g, B, CFG.conv_k - 1, CDIM), _randn(g, B, HV, DV, DV) * 0.1
    elif kind in ("attn_prefill", "attn_chunk"):
        B, T = case["B"], case["T"]
        n = (T + case.get("ctx", 0) + 64 + 63) // 64 * 64
        s["p"], s["norm"] = _attn_params(g), 0.1 * _randn(g, H)
        s["x"] = _randn(g, B, T, H) * 3
        s["k"], s["v"] = (_randn(g, B, HKV, n, D).bfloat16() for _ in range(2))
        # the rows' lengths differ by up to a fifth
        s["at"] = [case["ctx"] - (case["ctx"] // 5) * b // max(B - 1, 1) for b in range(B)] if "ctx" in case else 0
    elif kind == "mlp":
        s["p"], s["norm"] = _mlp_params(g, case["mlp_group"]), 0.1 * _randn(g, H)
        s["x"] = _randn(g, case["B"], case["T"], H) * 3
        s["push"] = [(17, "add", [8.0, 0.0, -8.0])]
    elif kind == "gdn_op":
        s["delta"] = _delta_inputs(g, case["B"], case["T"], case["state"])
    elif kind == "attn_op":
        B, T = case["B"], case["T"]
        s["q"], s["k"], s["v"] = (_randn(g, B, T, h, D).bfloat16() for h in (HQ, HKV, HKV))
        s["gate"] = _randn(g, B, T, HQ * D).bfloat16()
    else:
        B, n = case["B"], case["ctx"]
        cap = (n + 63) // 64 * 64
        s["q"], s["gate"] = _randn(g, B, HQ, D).bfloat16(), _randn(g, B, HQ * D).bfloat16()
        s["k"], s["v"] = (_randn(g, B, HKV, cap, D).bfloat16() for _ in range(2))
        s["len"] = torch.full((B,), n, dtype=torch.int32, device=DEV)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "completion":
        m = HybridModel(CFG, s.pop("W"), torch.device(DEV, torch.cuda.current_device()), rows=case["rows"],
                        max_len=case["T"] + case["steps"] + 8)
        m.set_pushes({5: [(100, "add", [8.0, 0.0, -8.0])]})
        m.set_vectors(s["vecs"], s["vec_of_row"])
        m.enable_decode_graph()
        s["model"] = m
        s["logits"] = torch.empty(case["steps"] + 1, case["rows"], V, device=DEV)
    elif kind == "head":
        s["slots"] = torch.zeros(case["rows"], dtype=torch.int64, device=DEV)
        s["logits"] = torch.empty(case["rows"], V, device=DEV)
        s["idx"] = torch.empty(case["rows"], dtype=torch.int32, device=DEV)
    elif kind in ("gdn_decode", "gdn_prefill"):
        layers.gdn_in_weight(s["p"])
    elif kind in ("attn_prefill", "attn_chunk"):
        layers.attn_in_weight(s["p"])
        layers.rope_tables(s["k"].shape[2], CFG.rot, CFG.rope_theta, s["x"].device)
        if kind == "attn_chunk":
            s["pos"] = torch.tensor(s["at"], dtype=torch.int32, device=DEV)
    elif kind == "mlp":
        mlp_weights(s["p"])
        s["p"]["_pushes"][:1].copy_(ops.pack_pushes(s["push"], "cpu"))
        s["out"] = torch.empty_like(s["x"])
    elif kind in ("attn_op", "attn_decode"):
        n = case["T"] if kind == "attn_op" else s["k"].shape[2]
        s["cos"], s["sin"] = (t.to(DEV) for t in workloads.rope_tables(n))
    return s


# ---------------------------------------------------------------- one pass
@torch.no_grad()
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "completion":
        m, out = s["model"], s["logits"]
        m.reset()
        out[0].copy_(m.forward(s["prompt"])[0])
        for t in range(case["steps"]):
            out[t + 1].copy_(m.decode_step(s["ids"][t]))
        return out
    if kind == "head":
        return ops.gemv_norm_argmax(s["x"], s["q"], s["s"], (None, s["norm"], EPS, None), s["slots"], out=s["logits"],
                                    idx=s["idx"])
    if kind == "gdn_decode":
        y = layers.gated_deltanet_layer(s["x"], s["p"], s["conv"], s["rec"], eps=EPS,
                                        prenorm=(None, s["norm"], EPS, None))
        return y, s["conv"], s["rec"]
    if kind == "gdn_prefill":
        h = ops.add_rmsnorm_(s["x"], None, s["norm"], EPS, split=True)
        return layers.gated_deltanet_layer(h, s["p"], s["conv"], s["rec"], eps=EPS), s["conv"], s["rec"]
    if kind in ("attn_prefill", "attn_chunk"):
        h = ops.add_rmsnorm_(s["x"], None, s["norm"], EPS, split=True)
        y = layers.gated_attention_layer(h, s["p"], s["k"], s["v"], s["pos"] if kind == "attn_chunk" else 0, eps=EPS)
        return y, s["k"], s["v"]
    if kind == "mlp":
        # the residual is kept and the MLP's output accumulated into a copy of it, as a caller that reads both does
        x = s["out"].copy_(s["x"])
        h = ops.add_rmsnorm_(x, None, s["norm"], EPS, split=True)
        return mlp(s["p"], h, x)
    if kind == "gdn_op":
        q, k, v, g, beta, S = s["delta"]
        return ops.chunk_gated_delta_rule(q, k, v, g, beta, initial_state=S, output_final_state=True,
                                          use_qk_l2norm_in_kernel=True)
    if kind == "attn_op":
        return ops.gated_attention_prefill(s["q"], s["k"], s["v"], s["gate"], s["cos"], s["sin"])
    return ops.gated_attention_decode(s["q"], s["k"], s["v"], s["gate"], s["len"], s["cos"], s["sin"])


# ---------------------------------------------------------------- work and tolerance
def _w8(n, k, group=128):
    """Bytes of an int8 weight and its fp32 scales."""
    return n * k + 4 * (n * (k // group) if group else n)


def _gdn_work(B, T):
    """Beside the projections: the recurrence's products per token and head (k S, the rank-1 update, q S) and the
    states read and written once."""
    M = B * T
    w = _w8(GDN_N, H) + _w8(H, HV * DV) + 4 * CDIM * CFG.conv_k
    state = 2 * 4 * B * (HV * DV * DV + (CFG.conv_k - 1) * CDIM)
    return w + state, 2 * M * (GDN_N * H + H * HV * DV) + 7 * M * HV * DV * DV


def _attn_work(B, T, ctx):
    """ctx: cached keys per row before the call's own."""
    M = B * T
    pairs = sum(T * c + T * (T + 1) // 2 for c in ctx)
    kv = sum(2 * 2 * HKV * D * (c + T) for c in ctx)
    return _w8(ATTN_N, H) + _w8(H, HQ * D) + kv, 2 * M * (ATTN_N * H + H * HQ * D) + 4 * D * HQ * pairs


def _mlp_work(M, group):
    return 2 * _w8(I, H, group) + _w8(H, I, group), 2 * M * 3 * I * H


def work(case):
    kind = case["kind"]
    if kind == "completion":
        B, T, n = case["rows"], case["T"], case["steps"]
        by = fl = 0
        for tok, at in [(T, 0)] + [(1, T + i) for i in range(n)]:
            for l in range(CFG.layers):
                b, f = _attn_work(B, tok, [at] * B) if CFG.is_attention(l) else _gdn_work(B, tok)
                b2, f2 = _mlp_work(B * tok, case["mlp_group"])
                by, fl = by + b + b2, fl + f + f2
            by, fl = by + _w8(V, H) + 4 * B * V, fl + 2 * B * V * H
        return dict(bytes=by, flops=fl)
    if kind == "head":
        M = case["rows"]
        return dict(bytes=_w8(V, H) + 4 * M * (V + H), flops=2 * M * V * H)
    if kind in ("gdn_decode", "gdn_prefill"):
        B, T = (case["rows"], 1) if kind == "gdn_decode" else (case["B"], case["T"])
        b, f = _gdn_work(B, T)
        return dict(bytes=b + 8 * B * T * H, flops=f)
    if kind in ("attn_prefill", "attn_chunk"):
        B, T = case["B"], case["T"]
        b, f = _attn_work(B, T, [case.get("ctx", 0) * (10 - i) // 10 for i in range(B)])
        return dict(bytes=b + 8 * B * T * H, flops=f)
    if kind == "mlp":
        M = case["B"] * case["T"]
        b, f = _mlp_work(M, case["mlp_group"])
        return dict(bytes=b + 8 * M * H, flops=f)
    if kind == "gdn_op":
        M = case["B"] * case["T"] * HV
        states = (2 if case["state"] else 1) * 4 * case["B"] * HV * DV * DV
        return dict(bytes=M * (4 * 2 * DV + 8) + states, flops=7 * M * DV * DV)
    if kind == "attn_op":
        B, T = case["B"], case["T"]
        return dict(bytes=2 * B * T * D * (3 * HQ + 2 * HKV), flops=4 * D * HQ * B * T * (T + 1) // 2)
    B, n = case["B"], case["ctx"]
    return dict(bytes=B * (2 * 2 * HKV * D * n + 3 * 2 * HQ * D), flops=4 * B * HQ * D * n)


def tolerance(case):
    """About four times the error against 64 bits that was measured, which is what the path's number formats give:
    fp32 sums; the prefill products' activations in two bf16 pieces (the recurrent state amplifies their rounding);
    q, k, v and the output of attention in bf16; a whole model's logits after six attention layers of that."""
    return {
        "completion": {"rel": 1.2e-2},
        "head": {"rel": 1e-6},
        "gdn_decode": {"rel": 2e-6},
        "gdn_prefill": {"rel": 1.2e-4},
        "attn_prefill": {"rel": 1.3e-2},
        "attn_chunk": {"rel": 1.3e-2},
        "mlp": {"rel": 2e-6},
        "gdn_op": {"rel": 1.3e-2},
        "attn_op": {"rel": 1e-2},
        "attn_decode": {"rel": 8e-3},
    }[case["kind"]]


# ---------------------------------------------------------------- 64-bit results
def _lin(x, p, name):
    return x @ workloads.dequantize_int8(p[name + ".q"], p[name + ".s"]).double().T


def _norm(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * (1.0 + w.double())


def _silu(x):
    return x * torch.sigmoid(x)


def _delta(q, k, v, g, beta, S):
    """The gated delta rule token by token (l2 norms on q and k). Returns (o, S)."""
    B, T, h, d = q.shape
    q, k = (t * torch.rsqrt((t * t).sum(-1, keepdim=True) + EPS) for t in (q, k))
    q = q / math.sqrt(d)
    S = torch.zeros(B, h, d, v.shape[-1], dtype=torch.float64, device=q.device) if S is None else S.double()
    decay, o = g.exp(), []
    for t in range(T):
        S = S * decay[:, t, :, None, None]
        u = (v[:, t] - (k[:, t, :, None, :] @ S)[:, :, 0]) * beta[:, t, :, None]
        S = S + k[:, t, :, :, None] * u[:, :, None, :]
        o.append((q[:, t, :, None, :] @ S)[:, :, 0])
    return torch.stack(o, 1), S


def _gdn(p, h, conv, rec):
    B, T, _ = h.shape
    full = torch.cat([conv.double(), _lin(h, p, "in_proj_qkv")], 1)
    w = p["conv1d"].double()
    c = _silu(sum(full[:, i:i + T] * w[:, i] for i in range(CFG.conv_k)))
    q, k, v = (t.reshape(B, T, HV, DV) for t in c.split(HV * DV, -1))
    z = _lin(h, p, "in_proj_z").reshape(B, T, HV, DV)
    beta = torch.sigmoid(_lin(h, p, "in_proj_b"))
    a = _lin(h, p, "in_proj_a") + p["dt_bias"].double()
    g = -p["A_log"].double().exp() * torch.nn.functional.softplus(a)
    o, rec = _delta(q, k, v, g, beta, rec)
    o = o * torch.rsqrt(o.pow(2).mean(-1, keepdim=True) + EPS) * p["norm"].double() * _silu(z)
    return _lin(o.reshape(B, T, -1), p, "out_proj"), full[:, -(CFG.conv_k - 1):], rec


def _rope(x, pos):
    """x [T, heads, D] rotated at the positions pos [T] (the angles in fp32, as the tables hold them)."""
    half = CFG.rot // 2
    inv = 1.0 / (CFG.rope_theta ** (torch.arange(0, CFG.rot, 2, device=x.device).float() / CFG.rot))
    ang = (pos.float()[:, None] * inv).double()[:, None]
    a, b = x[..., :half], x[..., half:2 * half]
    return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin(), x[..., 2 * half:]], -1)


def _softmax_attn(q, k, v, gate, first):
    """q [T, HQ, D] at positions first .., k and v [S, HKV, D]; returns [T, HQ * D] gated."""
    T, S = q.shape[0], k.shape[0]
    rep = HQ // HKV
    mask = torch.arange(S, device=q.device)[None] > first + torch.arange(T, device=q.device)[:, None]
    out = []
    for h in range(HQ):
        w = (q[:, h] @ k[:, h // rep].T / math.sqrt(D)).masked_fill(mask, -math.inf)
        out.append(torch.softmax(w, -1) @ v[:, h // rep])
    return torch.cat(out, -1) * torch.sigmoid(gate)


def _attn(p, h, k_old, v_old, at):
    """The mixer over h [B, T, H]; k_old, v_old: per row [HKV, at[b], D] (rotated). Returns y and the rows' keys,
    values."""
    B, T, _ = h.shape
    qg = _lin(h, p, "q_proj").reshape(B, T, HQ, 2 * D)
    q, gate = _norm(qg[..., :D], p["q_norm"]), qg[..., D:].reshape(B, T, HQ * D)
    k = _norm(_lin(h, p, "k_proj").reshape(B, T, HKV, D), p["k_norm"])
    v = _lin(h, p, "v_proj").reshape(B, T, HKV, D)
    out, ks, vs = [], [], []
    for b in range(B):
        pos = at[b] + torch.arange(T, device=h.device)
        ks.append(torch.cat([k_old[b].double().transpose(0, 1), _rope(k[b], pos)], 0))
        vs.append(torch.cat([v_old[b].double().transpose(0, 1), v[b]], 0))
        out.append(_softmax_attn(_rope(q[b], pos), ks[b], vs[b], gate[b], at[b]))
    return _lin(torch.stack(out), p, "o_proj"), ks, vs


def _mlp(p, h, pushes, T):
    a = _silu(_lin(h, p, "gate_proj")) * _lin(h, p, "up_proj")
    for neuron, _, vals in pushes:  # adds; one value per batch row, the row clamped to 3
        v = torch.tensor((list(vals) + [0.0] * 4)[:4], dtype=torch.float64, device=h.device)
        a[..., neuron] += v[torch.arange(h.shape[0], device=h.device).clamp(max=3)][:, None]
    return _lin(a, p, "down_proj")


def _whole_model(s):
    case, W = s["case"], s["W"]
    B, T, n = case["rows"], case["T"], case["steps"]
    embed = workloads.dequantize_int8(W["embed.q"], W["embed.s"]).double()
    x = embed[torch.cat([s["prompt"], s["ids"].long().T], 1)]
    for l in range(CFG.layers):
        p = {k[len(f"layers.{l}."):]: t for k, t in W.items() if k.startswith(f"layers.{l}.")}
        h = _norm(x, p["input_layernorm"])
        if CFG.is_attention(l):
            none = [torch.zeros(HKV, 0, D, device=DEV)] * B
            x = x + _attn(p, h, none, none, [0] * B)[0]
        else:
            x = x + _gdn(p, h, torch.zeros(B, CFG.conv_k - 1, CDIM, device=DEV), None)[0]
        push = [(100, "add", [8.0, 0.0, -8.0])] if l == 5 else []
        x = x + _mlp(p, _norm(x, p["post_attention_layernorm"]), push, T + n)
        if l == 12 and s["vecs"] is not None:
            for b, r in enumerate(s["vec_of_row"]):
                if r >= 0:
                    x[b] += s["vecs"][r].double()
    return (_norm(x[:, T - 1:], W["norm"]) @ embed.T).transpose(0, 1)


@torch.no_grad()
def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "completion":
        return _whole_model(s)
    if kind == "head":
        return _norm(s["x"].double(), s["norm"]) @ workloads.dequantize_int8(s["q"], s["s"]).double().T, None
    if kind in ("gdn_decode", "gdn_prefill"):
        return _gdn(s["p"], _norm(s["x"].double(), s["norm"]), s["conv"], s["rec"])
    if kind in ("attn_prefill", "attn_chunk"):
        B, T = case["B"], case["T"]
        at = s["at"] if kind == "attn_chunk" else [0] * B
        old = [[t[b, :, :at[b]] for b in range(B)] for t in (s["k"], s["v"])]
        y, ks, vs = _attn(s["p"], _norm(s["x"].double(), s["norm"]), *old, at)
        kc, vc = s["k"].double(), s["v"].double()
        for b in range(B):
            kc[b, :, :at[b] + T], vc[b, :, :at[b] + T] = ks[b].transpose(0, 1), vs[b].transpose(0, 1)
        return y, kc, vc
    if kind == "mlp":
        x = s["x"].double()
        return x + _mlp(s["p"], _norm(x, s["norm"]), s["push"], case["T"])
    if kind == "gdn_op":
        q, k, v, g, beta, S = s["delta"]
        return _delta(q.double(), k.double(), v.double(), g.double(), beta.double(), S)
    if kind == "attn_op":
        B, T = case["B"], case["T"]
        pos = torch.arange(T, device=DEV)
        return torch.stack([_softmax_attn(_rope(s["q"][b].double(), pos), _rope(s["k"][b].double(), pos),
                                          s["v"][b].double(), s["gate"][b].double(), 0) for b in range(B)])
    n = case["ctx"]
    at = torch.tensor([n - 1], device=DEV)
    return torch.cat([_softmax_attn(_rope(s["q"][b:b + 1].double(), at), s["k"][b, :, :n].double().transpose(0, 1),
                                    s["v"][b, :, :n].double().transpose(0, 1), s["gate"][b:b + 1].double(), n - 1)
                      for b in range(case["B"])])
