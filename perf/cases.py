"""The work this package does for its users, as cases that can be timed and checked.

A case is one call of a public entry point as a serving loop makes it: one decode step of one or several requests on the
dense, MoE and hybrid routes, or one prompt through the hybrid route's prefill.  Weights are random (the models are named by
their shapes); a decode step starts behind a filled cache.  ``exact`` evaluates the same step in 64 bits with plain torch.
"""
from __future__ import annotations

import math
import types

import torch

from __graft_entry__ import load_package

load_package()
from qimeng_megakernel_amd import decode_batch, decode_hybrid, registry, synthetic  # noqa: E402
from qimeng_megakernel_amd.decode_schedule import mk_kernel as dense_mk  # noqa: E402
from qimeng_megakernel_amd.decode_schedule.model_config import LlamaConfig  # noqa: E402
from qimeng_megakernel_amd.decode_schedule_hybrid import mk_kernel as hybrid_mk  # noqa: E402
from qimeng_megakernel_amd.decode_schedule_hybrid.state import RequestTable  # noqa: E402
from qimeng_megakernel_amd.decode_schedule_mb import mk_kernel as tiles_mk, rows_kernel as rows_mk  # noqa: E402
from qimeng_megakernel_amd.decode_schedule_moe import mk_kernel as moe_mk, rows_kernel as moe_rows_mk  # noqa: E402
from qimeng_megakernel_amd.decode_schedule_moe.model_config import QwenMoeConfig  # noqa: E402

DEVICE, BF16, F64 = "cuda", torch.bfloat16, torch.float64
SPARE = 32          # positions a decode request's cache holds behind the present one
DENSE = ("llama-3.2-1b", "qwen3-1.7b")
MOE = ("qwen1.5-moe-a2.7b", "qwen3-30b-a3b")
HYBRID = ("lusupel-1b", "givopel-1b", "lusupel-2b", "givopel-2b")


def listed():
    return [
        # A chat request in the middle of its answer: the headline workload, the smallest call in bytes.
        dict(name="llama_step", kind="dense", model="llama-3.2-1b", rows=1, context=1024),
        # The same behind a long document: the cache is a fifth of the bytes.
        dict(name="llama_step_long", kind="dense", model="llama-3.2-1b", rows=1, context=16384),
        # A few requests decoded together, each at its own position (the row-streaming engine).
        dict(name="llama_step_3_rows", kind="dense", model="llama-3.2-1b", rows=3, context=900),
        # A small server's batch of the second dense family: heads of 128, a norm per head (the matrix-core engine).
        dict(name="qwen_step_8_rows", kind="dense", model="qwen3-1.7b", rows=8, context=500),
        # One request of a mixture of experts with a shared expert.
        dict(name="qwen_moe_step", kind="moe", model="qwen1.5-moe-a2.7b", rows=1, context=300),
        # Four requests of a large mixture in one launch: the most bytes of a step.
        dict(name="a3b_step_4_rows", kind="moe", model="qwen3-30b-a3b", rows=4, context=500),
        # A decode step of each hybrid design.
        dict(name="lusupel_step", kind="hybrid", model="lusupel-1b", dtype="bfloat16", past=1000, tokens=1),
        dict(name="givopel_step", kind="hybrid", model="givopel-1b", dtype="bfloat16", past=600, tokens=1),
        # The next turn of a conversation: a few words behind what is already held.
        dict(name="lusupel_turn", kind="hybrid", model="lusupel-2b", dtype="bfloat16", past=400, tokens=43),
        # A short prompt in the exact mode that checks a port or a checkpoint.
        dict(name="lusupel_prompt_f32", kind="hybrid", model="lusupel-2b", dtype="float32", past=0, tokens=200),
        # An ordinary prompt, of no round length.
        dict(name="lusupel_prompt", kind="hybrid", model="lusupel-1b", dtype="bfloat16", past=0, tokens=1531),
        # A long prompt: two portions, the second behind the first.
        dict(name="givopel_prompt", kind="hybrid", model="givopel-1b", dtype="bfloat16", past=0, tokens=4096),
    ]


def _spread(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("dense", "dense", "dense", "moe", "hybrid", "hybrid", "hybrid"))
    if kind == "dense":
        rows = rng.choice((1, 1, 1, 2, 3, 4, rng.randint(5, 16)))
        return dict(kind=kind, model=rng.choice(DENSE), rows=rows, context=_spread(rng, 16, 16384 if rows == 1 else 2000))
    if kind == "moe":
        model = rng.choice(MOE)
        return dict(kind=kind, model=model, rows=1 if model == MOE[0] else rng.randint(1, 4), context=_spread(rng, 16, 1000))
    dtype = rng.choice(("bfloat16", "bfloat16", "bfloat16", "float32"))
    if rng.random() < 0.4:
        return dict(kind=kind, model=rng.choice(HYBRID), dtype=dtype, past=_spread(rng, 100, 2000), tokens=1)
    tokens = _spread(rng, 2, 3900 if dtype == "bfloat16" else 400)
    # A request's first tokens are ill-conditioned in one of the designs (a norm over a delta rule's first output leaves its
    # sign): in bfloat16 its prompts start at a length where they no longer decide the outcome.
    past = 0 if tokens > 2048 else rng.choice((0, 0, _spread(rng, 16, 1000)))
    names = HYBRID[:2] if tokens > 2048 else HYBRID if dtype == "float32" or past + tokens >= 100 else HYBRID[::2]
    return dict(kind=kind, model=rng.choice(names), dtype=dtype, past=past, tokens=tokens)


# ---- inputs: from the seed alone, on the GPU -----------------------------------------------------------------------

def _contexts(case):
    """Positions every row of a step attends to: ragged, the last row at the case's context."""
    rows, last = case["rows"], case["context"]
    return [last - (last // 2) * (rows - 1 - r) // max(rows - 1, 1) for r in range(rows)]


class _Draws:
    def __init__(self, seed):
        self.gen = torch.Generator(device=DEVICE)
        self.gen.manual_seed(seed)

    def normal(self, *size, std=0.02, mean=0.0, dtype=BF16):
        return torch.empty(*size, dtype=dtype, device=DEVICE).normal_(mean, std, generator=self.gen)

    def tokens(self, n, vocab):
        return torch.randint(0, vocab, (n,), generator=self.gen, device=DEVICE)


def _rope(shape, positions):
    """fp32 cos and sin of angles in 64 bits, a column per dimension of a head, rotation pairs side by side."""
    freq = shape.rope_theta ** (-torch.arange(0, shape.head_dim, 2, dtype=F64, device=DEVICE) / shape.head_dim)
    angle = torch.outer(torch.arange(positions, dtype=F64, device=DEVICE), freq).repeat_interleave(2, dim=1)
    return angle.cos().float(), angle.sin().float()


def _attention_weights(d, s, positions):
    L, H = s.num_hidden_layers, s.hidden_size
    w = dict(embed_tokens=d.normal(s.vocab_size, H, std=1.0), qkv_weights=d.normal(L, s.qkv_out_dim, H),
             o_proj_weights=d.normal(L, H, s.num_attention_heads * s.head_dim, std=0.02 / math.sqrt(2 * L)),
             attn_norm_weights=d.normal(L, H, std=0.1, mean=1.0), mlp_norm_weights=d.normal(L, H, std=0.1, mean=1.0),
             lm_head_norm_weights=d.normal(H, std=0.1, mean=1.0))
    w["rope_cos"], w["rope_sin"] = _rope(s, positions)
    if s.qk_norm:
        w["q_norm_weights"], w["k_norm_weights"] = (d.normal(L, s.head_dim, std=0.1, mean=1.0) for _ in range(2))
    return w


def _step_inputs(case, seed):
    """Weights, one token per row, and every row's cache rows ``[L, positions, kv heads, head size]``.  The projections that
    add to the residual are drawn smaller by the root of their number, so that the model stays as calm as a trained one."""
    s, d, positions = registry.shape_of(case["model"]), _Draws(seed), case["context"] + SPARE
    L, H = s.num_hidden_layers, s.hidden_size
    w = _attention_weights(d, s, positions)
    if case["kind"] == "dense":
        F = s.intermediate_size
        w.update(up_proj_weights=d.normal(L, F, H), gate_proj_weights=d.normal(L, F, H), down_proj_weights=d.normal(L, H, F, std=0.02 / math.sqrt(2 * L)))
        w["lm_head_weights"] = w["embed_tokens"] if s.tie_word_embeddings else d.normal(s.vocab_size, H)
    else:
        F, Fm, E = s.intermediate_size, s.moe_intermediate_size, s.num_experts
        w.update(router_weights=d.normal(L, E, H), expert_gate_up_proj_weights=d.normal(L, E, 2 * Fm, H), expert_down_proj_weights=d.normal(L, E, H, Fm, std=0.02 / math.sqrt(2 * L)),
                 lm_head_weights=d.normal(s.vocab_size, H))
        if s.qkv_bias:
            w["qkv_bias"] = d.normal(L, s.qkv_out_dim)
        if s.has_shared_expert:
            w.update(shared_expert_gate_proj_weights=d.normal(L, F, H), shared_expert_up_proj_weights=d.normal(L, F, H),
                     shared_expert_down_proj_weights=d.normal(L, H, F, std=0.02 / math.sqrt(2 * L)), shared_expert_gate_weights=d.normal(L, 1, H))
    tokens = d.tokens(case["rows"], s.vocab_size)
    past = [tuple(d.normal(L, positions, s.num_key_value_heads, s.head_dim, std=1.0) for _ in range(2)) for _ in range(case["rows"])]
    return s, w, tokens, past


def _hybrid_inputs(case, seed):
    shape = registry.shape_of(case["model"])
    weights = synthetic.random_hybrid_weights(shape, seed, DEVICE)
    return shape, weights, _Draws(seed + 1_000_003).tokens(case["past"] + case["tokens"], shape.vocab)


def prepare(case, seed):
    if case["kind"] == "hybrid":
        from qimeng_megakernel_amd.decode_schedule_hybrid import HybridConfig, weights as packing
        from qimeng_megakernel_amd.decode_schedule_hybrid.globs import build_globals

        shape, tensors, tokens = _hybrid_inputs(case, seed)
        HybridConfig.set_shape(shape)
        past, n = case["past"], case["tokens"]
        globs = build_globals(shape, packing.pack(shape, tensors, DEVICE), dtype=getattr(torch, case["dtype"]), max_positions=past + n + SPARE)
        mk, table = hybrid_mk.get_mk(), RequestTable(globs)
        if past:
            decode_hybrid.run_tokens(globs, mk, table.get("request"), tokens[:past])
        return types.SimpleNamespace(case=case, globs=globs, mk=mk, table=table, tokens=tokens[past:].contiguous())

    s, w, tokens, past = _step_inputs(case, seed)
    rows, capacity, contexts = case["rows"], case["context"] + SPARE, _contexts(case)
    positions = torch.tensor([c - 1 for c in contexts], dtype=torch.int32, device=DEVICE)
    if case["kind"] == "moe":
        QwenMoeConfig.set_shape(s)
        if rows == 1:
            globs, mk = synthetic.build_moe_globals(w, s, capacity, DEVICE), moe_mk.get_mk()
            globs.position_id = contexts[0] - 1
            caches = [(globs.k_cache[:, 0], globs.v_cache[:, 0])]
            moe_mk.build(globs, mk)
        else:
            globs, mk = moe_rows_mk.build_rows_globals(w, s, capacity, rows, DEVICE), moe_rows_mk.get_mk()
            globs.position_ids.copy_(positions)
            caches = [(globs.k_cache[r, :, 0], globs.v_cache[r, :, 0]) for r in range(rows)]
            moe_rows_mk.build(globs)
    else:
        LlamaConfig.set_shape(s)
        if rows == 1:
            globs, mk = synthetic.build_globals(w, s, capacity, DEVICE), dense_mk.get_mk()
            globs.position_id = contexts[0] - 1
            dense_mk._scheduler.build(globs)
        else:
            launcher = rows_mk if rows <= decode_batch.ROWS_ENGINE_MAX_BATCH else tiles_mk
            globs, mk = synthetic.build_batch_globals(w, s, capacity, rows, DEVICE), launcher.get_mk()
            globs.position_ids.copy_(positions)
            launcher.build(globs)
        caches = [(globs.k_cache[:, r], globs.v_cache[:, r]) for r in range(rows)]
    for (k, v), (k0, v0) in zip(caches, past):
        k.copy_(k0)
        v.copy_(v0)
    return types.SimpleNamespace(case=case, globs=globs, mk=mk, tokens=tokens, contexts=contexts, caches=caches)


def run(state):
    case, globs, mk = state.case, state.globs, state.mk
    if case["kind"] == "hybrid":
        if case["past"]:
            request = state.table.get("request")
            request.position = case["past"]
        else:                       # a prompt: the request that is answered next takes the slot of the one before
            if "request" in state.table.live:
                state.table.close("request")
            request = state.table.open("request")
        logits = decode_hybrid.run_tokens(globs, mk, request, state.tokens, want=[case["tokens"] - 1])
        return {"logits": logits, "states": [l["state"][0] for l in globs.layer_state if "state" in l],
                "caches": [l["cache"][0] for l in globs.layer_state if "cache" in l]}
    rows = case["rows"]
    if rows == 1:
        globs.hidden_states.copy_(globs.embed_tokens[state.tokens].view(-1))
        (moe_mk if case["kind"] == "moe" else dense_mk).call_mk(globs, mk)
    else:
        globs.hidden_states.copy_(globs.embed_tokens[state.tokens])
        if case["kind"] == "moe":
            mk(globs)
        else:
            (rows_mk if rows <= decode_batch.ROWS_ENGINE_MAX_BATCH else tiles_mk).call_mk(globs, mk)
    appended = [(k[:, c - 1], v[:, c - 1]) for (k, v), c in zip(state.caches, state.contexts)]
    return {"logits": globs.logits.view(rows, -1), "hidden": globs.hidden_states.view(rows, -1), "k": [k for k, _ in appended], "v": [v for _, v in appended]}


# ---- what a pass cannot do without, and how close two right answers are ---------------------------------------------

def work(case):
    s = registry.shape_of(case["model"])
    if case["kind"] == "hybrid":
        n, past, item = case["tokens"], case["past"], 2 if case["dtype"] == "bfloat16" else 4
        flops = s.prefill_flops(n, past) + 2.0 * s.vocab * s.width
        cache = sum((min(past + n, e.shape.window) * (e.shape.rank + e.shape.rot_dim) if e.type == "latent_attention"
                     else (past + n) * e.shape.kv_heads * (e.shape.dim + e.shape.v_dim) if e.type == "attention" else 0) * item for e in s.entries)
        held = (s.step_bytes(past + 1, item) if n == 1 else s.step_bytes(0, item) + cache) + 4 * s.vocab
        return {"bytes": held, "flops": flops}
    contexts = _contexts(case)
    kv, logits = s.kv_bytes_per_context_token(), 2 * s.vocab_size
    weights = s.weight_bytes_per_token()
    if case["kind"] == "moe" and case["rows"] > 1:      # experts that several rows pick are read once
        k, E, B = s.num_experts_per_tok, s.num_experts, case["rows"]
        weights += s.num_hidden_layers * 6 * s.moe_intermediate_size * s.hidden_size * (E * (1 - (1 - k / E) ** B) - k)
    attention = sum(4.0 * s.num_hidden_layers * c * s.num_attention_heads * s.head_dim for c in contexts)
    return {"bytes": weights + sum(kv * c + kv + logits for c in contexts), "flops": s.weight_bytes_per_token() * case["rows"] + attention}


def tolerance(case):
    # Each side is this far from 64 bits: 0.007 to 0.018 with bf16 matrix operands, cache or residual (a sum taken in another
    # order turns single roundings, and 16 to 48 layers carry them on), 0.3e-5 to 1e-5 in float32.
    return {"rel": 5e-5, "max": 5e-3} if case.get("dtype") == "float32" else {"rel": 0.03, "max": 0.9}


# ---- the same in 64 bits -------------------------------------------------------------------------------------------

def _rms(x, eps, weight=None):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if weight is None else y * weight


def _turn(x, cos, sin):
    """Neighbouring pairs of the last dimension turned; cos and sin one value per pair."""
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack((a * cos - b * sin, b * cos + a * sin), dim=-1).flatten(-2)


def _silu(z):
    return z * torch.sigmoid(z)


def exact(case, seed):
    if case["kind"] == "hybrid":
        return _exact_hybrid(case, seed)
    s, w, tokens, past = _step_inputs(case, seed)
    nq, nkv, dim, eps = s.num_attention_heads, s.num_key_value_heads, s.head_dim, s.rms_norm_eps
    out = {"logits": [], "hidden": [], "k": [], "v": []}
    x = w["embed_tokens"][tokens].to(F64)
    at = torch.tensor([c - 1 for c in _contexts(case)], device=DEVICE)
    cos, sin = (w[n][at][:, None, ::2].to(F64) for n in ("rope_cos", "rope_sin"))
    new_k, new_v = [], []
    for layer in range(s.num_hidden_layers):
        def m(name):
            return w[name][layer].to(F64)

        qkv = _rms(x, eps, m("attn_norm_weights")) @ m("qkv_weights").T + (m("qkv_bias") if "qkv_bias" in w else 0)
        q, k, v = (t.view(case["rows"], -1, dim) for t in qkv.split((nq * dim, nkv * dim, nkv * dim), dim=-1))
        if s.qk_norm:
            q, k = _rms(q, eps, m("q_norm_weights")), _rms(k, eps, m("k_norm_weights"))
        q, k = _turn(q, cos, sin), _turn(k, cos, sin)
        new_k.append(k)
        new_v.append(v)
        o = torch.empty_like(q)
        for r, (k0, v0) in enumerate(past):
            n = int(at[r])
            for h in range(nkv):
                heads = slice(h * nq // nkv, (h + 1) * nq // nkv)
                keys, values = (torch.cat((old[layer, :n, h].to(F64), new[r, h : h + 1])) for old, new in ((k0, k), (v0, v)))
                o[r, heads] = torch.softmax(q[r, heads] @ keys.T / math.sqrt(dim), dim=-1) @ values
        x = x + o.flatten(1) @ m("o_proj_weights").T
        h = _rms(x, eps, m("mlp_norm_weights"))
        if case["kind"] == "dense":
            x = x + (_silu(h @ m("gate_proj_weights").T) * (h @ m("up_proj_weights").T)) @ m("down_proj_weights").T
        else:
            x = x + _mixture(s, m, {n: w[n][layer] for n in ("expert_gate_up_proj_weights", "expert_down_proj_weights")}, h)
    out["hidden"] = x
    out["logits"] = _rms(x, eps, w["lm_head_norm_weights"].to(F64)) @ w["lm_head_weights"].to(F64).T
    out["k"], out["v"] = ([torch.stack([t[r] for t in new]) for r in range(case["rows"])] for new in (new_k, new_v))
    return out


def _mixture(s, m, experts, h):
    share, pick = torch.softmax(h @ m("router_weights").T, dim=-1).topk(s.num_experts_per_tok, dim=-1)
    if s.norm_topk_prob:
        share = share / share.sum(-1, keepdim=True)
    y = torch.zeros_like(h)
    for r, row in enumerate(pick.tolist()):
        for slot, e in enumerate(row):
            gate, up = (experts["expert_gate_up_proj_weights"][e].to(F64) @ h[r]).chunk(2)
            y[r] += share[r, slot] * (experts["expert_down_proj_weights"][e].to(F64) @ (_silu(gate) * up))
    if s.has_shared_expert:
        shared = (_silu(h @ m("shared_expert_gate_proj_weights").T) * (h @ m("shared_expert_up_proj_weights").T)) @ m("shared_expert_down_proj_weights").T
        y = y + torch.sigmoid(h @ m("shared_expert_gate_weights").T) * shared
    return y


def _convolved(x, taps, bias=None):
    n, y = taps.shape[1], torch.zeros_like(x) if bias is None else bias.expand_as(x).clone()
    for j in range(n):
        back = n - 1 - j
        if back < x.shape[0]:
            y[back:] += taps[:, j] * x[: x.shape[0] - back]
    return y


def _attended(q, k, v, scale, window=None):
    """q [T, H, d], k [T, G, d], v [T, G, e]: causal, at most ``window`` keys back."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    i = torch.arange(T, device=DEVICE)
    distance = i[:, None] - i[None, :]
    hidden = (distance < 0) | (distance >= (window or T))
    return torch.stack([torch.softmax((q[:, h] @ k[:, h * G // H].T * scale).masked_fill(hidden, -math.inf), dim=-1) @ v[:, h * G // H] for h in range(H)], dim=1)


def _angles(T, dims, base, scaling=None):
    freq, magnitude = base ** (-torch.arange(0, dims, 2, dtype=F64, device=DEVICE) / dims), 1.0
    if scaling is not None:             # YaRN: slow pairs interpolated, fast ones not, a ramp between them
        factor, original, fast, slow = scaling
        low, high = (dims * math.log(original / (2 * math.pi * turns)) / (2 * math.log(base)) for turns in (fast, slow))
        low, high = max(math.floor(low), 0), min(math.ceil(high), dims - 1)
        ramp = ((torch.arange(dims // 2, dtype=F64, device=DEVICE) - low) / max(high - low, 0.001)).clamp(0, 1)
        freq, magnitude = freq / factor * ramp + freq * (1 - ramp), 0.1 * math.log(factor) + 1
    angle = torch.outer(torch.arange(T, dtype=F64, device=DEVICE), freq)[:, None]
    return angle.cos() * magnitude, angle.sin() * magnitude


def _rglru(h, w, l, eps, keep):
    y = torch.nn.functional.gelu(h @ w("y").T + w("y.b"), approximate="tanh")
    u = _convolved(h @ w("x").T + w("x.b"), w("conv"), w("conv.b"))
    r, i = (torch.sigmoid(torch.cat([part @ m.T + b for part, m, b in zip(u.chunk(l.blocks, dim=1), w(n), w(n + ".b"))], dim=1)) for n in ("ra", "ri"))
    log_a = -8 * r * torch.nn.functional.softplus(w("lam"))
    a, b = log_a.exp(), torch.sqrt(-torch.expm1(2 * log_a)) * i * u
    s, states = torch.zeros_like(u[0]), torch.empty_like(u)
    for t in range(len(u)):
        s = torch.addcmul(b[t], a[t], s)
        states[t] = s
    keep("state", s)
    return (states * y) @ w("o").T


def _latent(h, w, l, eps, keep):
    T, H = len(h), l.heads
    cos, sin = _angles(T, l.rot_dim, l.rope_base)
    q = (h @ w("q").T).view(T, H, l.dim + l.rot_dim)
    down = h @ w("dkv").T
    c, turned = _rms(down[:, : l.rank], eps, w("dkv.norm")), _turn(down[:, None, l.rank :], cos, sin)
    k = torch.cat(((c @ w("uk").T).view(T, H, l.dim), turned.expand(T, H, l.rot_dim)), dim=-1)
    q = torch.cat((q[..., : l.dim], _turn(q[..., l.dim :], cos, sin)), dim=-1)
    keep("cache", None)
    o = _attended(q, k, (c @ w("uv").T).view(T, H, l.v_dim), l.scale, l.window).flatten(1)
    return (o * torch.sigmoid(h @ w("g").T)) @ w("o").T


def _wkv(h, w, l, eps, keep):
    T, H, n = len(h), l.heads, l.dim
    before = torch.cat((torch.zeros_like(h[:1]), h[:-1]))
    mixed = {x: h + (before - h) * w("mu." + x) for x in "rkvgw"}
    r, k, v = ((mixed[x] @ w(x).T).view(T, H, n) for x in "rkv")
    decay = torch.exp(-torch.exp(torch.tanh(mixed["w"] @ w("w1").T) @ w("w2").T + w("w0"))).view(T, H, n, 1)
    s, o, bonus = h.new_zeros(H, n, n), torch.empty_like(r), w("u")[..., None]
    for t in range(T):
        kv = k[t][..., None] * v[t][:, None, :]
        o[t] = ((s + bonus * kv) * r[t][..., None]).sum(1)
        s = torch.addcmul(kv, decay[t], s)
    keep("state", s)
    return (_rms(o, eps).flatten(1) * w("norm") * _silu(mixed["g"] @ w("g").T)) @ w("o").T


def _attention(h, w, l, eps, keep):
    T = len(h)
    cos, sin = _angles(T, l.rot_dim, l.rope_base, l.rope_scaling)
    q, k, v = ((h @ w(n).T).view(T, heads, -1) for n, heads in (("q", l.heads), ("k", l.kv_heads), ("v", l.kv_heads)))
    q, k = (torch.cat((_turn(x[..., : l.rot_dim], cos, sin), x[..., l.rot_dim :]), dim=-1) for x in (q, k))
    keep("cache", None)
    return (_attended(q, k, v, l.scale).flatten(1) * torch.sigmoid(h @ w("g").T)) @ w("o").T


def _delta(h, w, l, eps, keep):
    T, H = len(h), l.heads
    q, k, v = (_silu(_convolved(h @ w(n).T, w(n + ".conv"))).view(T, heads, -1) for n, heads in (("q", l.kv_heads), ("k", l.kv_heads), ("v", H)))
    q, k = (torch.repeat_interleave(x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6), H // l.kv_heads, dim=1) for x in (q, k))
    beta = torch.sigmoid(h @ w("b").T)[..., None]
    rate = torch.nn.functional.softplus(h @ w("a1").T @ w("a2").T + w("dt_bias")).view(T, H, l.dim)
    decay = torch.exp(-torch.exp(w("A_log"))[None, :, None] * rate)[..., None]
    s, o = h.new_zeros(H, l.dim, l.v_dim), torch.empty_like(v)
    for t in range(T):
        s = decay[t] * s
        s = s + k[t][..., None] * (beta[t] * (v[t] - (s * k[t][..., None]).sum(1)))[:, None, :]
        o[t] = (s * q[t][..., None]).sum(1) * l.dim**-0.5
    keep("state", s)
    return (_rms(o, eps, w("norm")).flatten(1) * torch.sigmoid(h @ w("g1").T @ w("g2").T)) @ w("o").T


def _gla(h, w, l, eps, keep):
    T, H = len(h), l.heads
    q, k, v = ((h @ w(n).T).view(T, H, -1) for n in "qkv")
    decay = torch.exp(torch.nn.functional.logsigmoid(h @ w("a1").T @ w("a2").T + w("a2.b")) / l.tau).view(T, H, l.dim, 1)
    s, o = h.new_zeros(H, l.dim, l.v_dim), torch.empty_like(v)
    for t in range(T):
        s = torch.addcmul(k[t][..., None] * v[t][:, None, :], decay[t], s)
        o[t] = (s * q[t][..., None]).sum(1) * l.dim**-0.5
    keep("state", s)
    return (_rms(o, eps, w("norm")).flatten(1) * _silu(h @ w("g").T)) @ w("o").T


_MIXERS = {"rglru": _rglru, "latent_attention": _latent, "wkv": _wkv, "attention": _attention, "delta": _delta, "gla": _gla}


def _exact_hybrid(case, seed):
    shape, weights, tokens = _hybrid_inputs(case, seed)
    eps, kept = shape.eps, {"state": [], "cache": []}

    def w(name):
        return weights[name].to(F64)

    def keep(name, value):
        kept[name].append(value)

    def layer_norm(x, weight):
        d = x - x.mean(-1, keepdim=True)
        return _rms(d, eps, weight)

    x = x0 = w("embed")[tokens]
    if shape.plain:
        for i, enters in shape.layer_runs():
            l, n = shape.layers[i], f"l{i}."
            if enters:
                x = torch.cat((x, x0), dim=-1) @ w("loop.in").T
            h = layer_norm(x, w(n + "norm1"))
            if l.branches:
                y = 0.5 * sum(_rms(_MIXERS[b.type](h, lambda k: w(f"{n}mix.{side}.{k}"), b, eps, keep), eps, w(f"{n}mix.{side}.out"))
                              for side, b in zip(("left", "right"), l.branches))
            else:
                y = _MIXERS[l.type](h, lambda k: w(f"{n}mix.{k}"), l, eps, keep)
            if l.ff:
                y = y + (_silu(h @ w(n + "mlp.gate").T) * (h @ w(n + "mlp.up").T)) @ w(n + "mlp.down").T
            x = x + y
        z = layer_norm(x[-1:], w("final.norm")) @ w("head").T * shape.logit_scale
        logits = shape.logit_softcap * torch.tanh(z / shape.logit_softcap) if shape.logit_softcap else z
    else:
        x = x[:, None].repeat(1, shape.streams, 1)

        def connected(x, name, sublayer):
            y = sublayer(torch.einsum("s,tsd->td", w(name + ".in"), x))
            return torch.einsum("su,tsd->tud", w(name + ".mix"), x) + w(name + ".out")[None, :, None] * y[:, None]

        for i, l in enumerate(shape.layers):
            n = f"l{i}."
            x = connected(x, n + "hc1", lambda u: _MIXERS[l.type](_rms(u, eps, w(n + "norm1")), lambda k: w(f"{n}mix.{k}"), l, eps, keep))
            if l.ff:
                def mlp(u):
                    h = _rms(u, eps, w(n + "norm2"))
                    return (torch.nn.functional.gelu(h @ w(n + "mlp.gate").T, approximate="tanh") * (h @ w(n + "mlp.up").T)) @ w(n + "mlp.down").T

                x = connected(x, n + "hc2", mlp)
        logits = _rms(x[-1:].sum(1), eps, w("final.norm")) @ w("head").T
    return {"logits": logits, "states": kept["state"], "caches": kept["cache"]}
