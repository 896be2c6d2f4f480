"""Performance cases of the framework: the calls a serving program makes, from
one token of one sequence to a batch of long prompts.

`listed()` names the fixed cases and `draw(rng)` gives more of the same ranges.
`prepare(case, seed)` makes on the GPU what a program holds before the call
(weights, caches, tables, the captured decode step), `run(state)` makes one
pass through the public entry points, `work(case)` says what the pass cannot do
without, and `exact(case, seed)` computes the same outputs in float64 with
plain torch.

Kinds:
  step    one decode step of a whole model, replayed from its captured graph
  decode  batched decode attention over a dense or paged KV cache
  prompt  fused QK-norm + RoPE + KV append, then causal prefill attention
  attn    the attention half of a decoder layer over a prompt (norm, qkv_proj,
          append, prefill, o_proj, residual add + norm)
  mlp     the MLP half (gate_up with SiLU * up, down, residual add + norm)
  select  token selection: greedy argmax and top-k over the logits
"""
from __future__ import annotations

import math

import numpy as np
import torch

from crane_amd import ops
from crane_amd.decoder import LayerWeights
from crane_amd.model import DecodeGraph, DecoderModel, ModelConfig

D = 128
EPS = 1e-6
THETA = 1e6
VOCAB = 151936
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
ORDER = {"qwen3": "norm_then_rope", "qwen2": "rope_only", "hunyuan": "rope_then_norm"}

# model: hidden, q heads, kv heads, intermediate, layers, family
MODELS = {
    "qwen3-0.6b": (1024, 16, 8, 3072, 28, "qwen3"),
    "qwen3-8b": (4096, 32, 8, 12288, 36, "qwen3"),
    "qwen2.5-7b": (3584, 28, 4, 18944, 28, "qwen2"),
}


def listed():
    return [
        # Interactive chat: one user, one token at a time, the smallest model.
        {"name": "step_0.6b_b1", "kind": "step", "model": "qwen3-0.6b", "layers": 28, "batch": 1, "lo": 1000,
         "hi": 1000},
        # A loaded server: 32 sequences of 512 to 4096 tokens, one step.
        {"name": "step_8b_b32", "kind": "step", "model": "qwen3-8b", "layers": 36, "batch": 32, "lo": 512,
         "hi": 4096},
        # One layer's attention for one sequence in f32, the smallest call.
        {"name": "decode_f32_one", "kind": "decode", "dtype": "f32", "paged": False, "batch": 1, "hq": 16, "hkv": 8,
         "lo": 1025, "hi": 1025},
        # One layer's attention of the loaded server.
        {"name": "decode_ragged", "kind": "decode", "dtype": "bf16", "paged": False, "batch": 32, "hq": 32, "hkv": 8,
         "lo": 513, "hi": 4097},
        # Long documents on a wide model, their rows in pages.
        {"name": "decode_long_paged", "kind": "decode", "dtype": "bf16", "paged": True, "batch": 8, "hq": 64,
         "hkv": 8, "lo": 30000, "hi": 32769},
        # A first prompt into an empty cache, the small model.
        {"name": "prompt_one", "kind": "prompt", "dtype": "bf16", "family": "qwen3", "batch": 1, "seq": 2048,
         "hq": 16, "hkv": 8, "start": 0},
        # Long prompts of a whole batch.
        {"name": "prompt_batch", "kind": "prompt", "dtype": "bf16", "family": "qwen2", "batch": 8, "seq": 4096,
         "hq": 28, "hkv": 4, "start": 0},
        # A follow-up turn: odd chunks over caches of different lengths.
        {"name": "prompt_chunk", "kind": "prompt", "dtype": "bf16", "family": "hunyuan", "batch": 3, "seq": 217,
         "hq": 32, "hkv": 8, "start": 3001},
        # A prompt in f32, as a model loaded without a narrower type runs.
        {"name": "prompt_f32", "kind": "prompt", "dtype": "f32", "family": "qwen3", "batch": 1, "seq": 731,
         "hq": 16, "hkv": 8, "start": 0},
        # Attention half of a layer over two short prompts, with the qkv bias.
        {"name": "attn_short", "kind": "attn", "model": "qwen2.5-7b", "batch": 2, "seq": 150, "start": 0},
        # MLP half of a layer over a short prompt, or a decode batch past 32.
        {"name": "mlp_77", "kind": "mlp", "model": "qwen3-8b", "rows": 77},
        # Token selection for a batch of 16 sequences.
        {"name": "select_16", "kind": "select", "rows": 16, "vocab": VOCAB, "k": 64},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["step", "decode", "prompt", "attn", "mlp", "select"])
    if kind == "step":
        model = rng.choice(sorted(MODELS))
        layers = 28 if model == "qwen3-0.6b" else rng.randint(4, 12)
        hi = _log(rng, 64, 4096)
        return {"kind": kind, "model": model, "layers": layers, "batch": _log(rng, 1, 48),
                "lo": rng.randint(max(1, hi // 8), hi), "hi": hi}
    if kind == "decode":
        hkv = rng.choice([2, 4, 8])
        hq = hkv * rng.choice([1, 2, 4, 7, 8])
        hi = _log(rng, 100, 32769)
        batch = _log(rng, 1, max(1, min(96, 300000 // hi)))
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "bf16", "f32"]), "paged": rng.random() < 0.4,
                "batch": batch, "hq": hq, "hkv": hkv, "lo": rng.randint(max(1, hi // 8), hi), "hi": hi}
    if kind == "prompt":
        f32 = rng.random() < 0.2
        hkv = rng.choice([4, 8])
        seq = _log(rng, 17, 1500 if f32 else 4096)
        batch = _log(rng, 1, max(1, min(8, (2000 if f32 else 24000) // seq)))
        return {"kind": kind, "dtype": "f32" if f32 else "bf16", "family": rng.choice(sorted(ORDER)), "batch": batch,
                "seq": seq, "hq": hkv * rng.choice([2, 4, 7] if hkv == 4 else [1, 2, 4]), "hkv": hkv,
                "start": rng.choice([0, 0, rng.randint(1, 3500)])}
    if kind == "attn":
        seq = _log(rng, 17, 1024)
        return {"kind": kind, "model": rng.choice(sorted(MODELS)), "batch": _log(rng, 1, max(1, min(4, 1024 // seq))),
                "seq": seq, "start": rng.choice([0, rng.randint(1, 1500)])}
    if kind == "mlp":
        return {"kind": kind, "model": rng.choice(sorted(MODELS)), "rows": _log(rng, 1, 768)}
    return {"kind": kind, "rows": _log(rng, 1, 96), "vocab": rng.choice([VOCAB, rng.randint(32000, VOCAB)]),
            "k": rng.choice([1, 20, 40, 64, rng.randint(1, 64)])}


# --------------------------------------------------------------------- inputs

def _dev():
    return torch.device("cuda", torch.cuda.current_device())


def _gen(seed):
    return torch.Generator(device=_dev()).manual_seed(seed)


def _randn(shape, gen, dtype, std=1.0):
    x = torch.randn(shape, generator=gen, dtype=dtype, device=_dev())
    return x if std == 1.0 else x.mul_(std)


def _norm_w(n, gen, dtype):
    return (1.0 + 0.1 * torch.randn(n, generator=gen, device=_dev())).to(dtype)


def _lengths(case, seed):
    """batch lengths spread over [lo, hi], their order drawn from the seed."""
    n = np.round(np.linspace(case["lo"], case["hi"], case["batch"])) if case["batch"] > 1 else np.array([case["hi"]])
    return np.random.default_rng(seed).permutation(n.astype(np.int32))


def _starts(case, seed):
    """Cached rows of each sequence before the prompt, up to case["start"]."""
    n = case["start"] - np.arange(case["batch"]) * (case["start"] // (2 * case["batch"]))
    return np.random.default_rng(seed).permutation(n.astype(np.int32))


def _ints(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.int32, device=_dev())


def _tables(dtype, n, narrow=False):
    """cos / sin [n, D / 2] in the model's type; narrow: the angles are formed
    in that type (the Qwen2.5 form)."""
    inv = 1.0 / (torch.tensor(THETA, dtype=torch.float64) ** (torch.arange(0, D, 2, dtype=torch.float64) / D)).float()
    pos = torch.arange(n, dtype=torch.float32)
    angle = (pos.to(dtype)[:, None] * inv.to(dtype)[None, :]).float() if narrow else pos[:, None] * inv[None, :]
    return angle.cos().to(dtype).to(_dev()), angle.sin().to(dtype).to(_dev())


def _layer_weights(model, gen, dtype, layers=1):
    """One layer's weights; a stack's o_proj and down_proj are scaled by
    (2 layers) ** -0.5, so that the residual stream keeps its size."""
    deep = (2 * layers) ** -0.5 if layers > 1 else 1.0
    hidden, hq, hkv, inter, _, family = MODELS[model]
    qkv = (hq + 2 * hkv) * D
    return LayerWeights(
        input_norm=_norm_w(hidden, gen, dtype),
        qkv=_randn((qkv, hidden), gen, dtype, hidden ** -0.5),
        o=_randn((hidden, hq * D), gen, dtype, deep * (hq * D) ** -0.5),
        post_norm=_norm_w(hidden, gen, dtype),
        gate_up=_randn((2 * inter, hidden), gen, dtype, hidden ** -0.5),
        down=_randn((hidden, inter), gen, dtype, deep * inter ** -0.5),
        qkv_bias=_randn((qkv,), gen, dtype, 0.1) if family == "qwen2" else None,
        q_norm=_norm_w(D, gen, dtype) if family != "qwen2" else None,
        k_norm=_norm_w(D, gen, dtype) if family != "qwen2" else None)


def _step_inputs(case, seed):
    gen, dtype = _gen(seed), torch.bfloat16
    hidden, _, hkv, _, _, _ = MODELS[case["model"]]
    cap = case["hi"] + 64
    layers = [_layer_weights(case["model"], gen, dtype, case["layers"]) for _ in range(case["layers"])]
    caches = [(_randn((case["batch"], hkv, cap, D), gen, dtype), _randn((case["batch"], hkv, cap, D), gen, dtype))
              for _ in range(case["layers"])]
    return {"layers": layers, "caches": caches, "cap": cap, "final_norm": _norm_w(hidden, gen, dtype),
            "lm_head": _randn((VOCAB, hidden), gen, dtype, hidden ** -0.5),
            "x": _randn((case["batch"], 1, hidden), gen, dtype), "lens": _lengths(case, seed)}


def _decode_inputs(case, seed):
    gen, dtype = _gen(seed), DTYPES[case["dtype"]]
    lens, hkv, page = _lengths(case, seed), case["hkv"], 256
    q = _randn((case["batch"], case["hq"], D), gen, dtype)
    if not case["paged"]:
        shape = (case["batch"], hkv, int(lens.max()), D)
        return {"q": q, "k": _randn(shape, gen, dtype), "v": _randn(shape, gen, dtype), "lens": lens, "table": None}
    pages = -(-lens // page)
    order = np.random.default_rng(seed).permutation(int(pages.sum())).astype(np.int32)
    table = np.full((case["batch"], int(pages.max())), -1, np.int32)
    at = 0
    for b, n in enumerate(pages):
        table[b, :n] = order[at:at + n]
        at += n
    shape = (int(pages.sum()), hkv, page, D)
    return {"q": q, "k": _randn(shape, gen, dtype), "v": _randn(shape, gen, dtype), "lens": lens, "table": table}


def _prompt_inputs(case, seed):
    gen, dtype = _gen(seed), DTYPES[case["dtype"]]
    B, S, hq, hkv = case["batch"], case["seq"], case["hq"], case["hkv"]
    starts = _starts(case, seed)
    cap = int(starts.max()) + S + 256
    norms = case["family"] != "qwen2"
    cos, sin = _tables(dtype, cap)
    return {"qkv": _randn((B, S, (hq + 2 * hkv) * D), gen, dtype), "k": _randn((B, hkv, cap, D), gen, dtype),
            "v": _randn((B, hkv, cap, D), gen, dtype), "starts": starts, "cos": cos, "sin": sin,
            "q_norm": _norm_w(D, gen, dtype) if norms else None, "k_norm": _norm_w(D, gen, dtype) if norms else None}


def _attn_inputs(case, seed):
    gen, dtype = _gen(seed), torch.bfloat16
    hidden, _, hkv, _, _, _ = MODELS[case["model"]]
    starts = _starts(case, seed)
    cap = int(starts.max()) + case["seq"] + 256
    cos, sin = _tables(dtype, cap)
    return {"w": _layer_weights(case["model"], gen, dtype), "x": _randn((case["batch"], case["seq"], hidden), gen, dtype),
            "k": _randn((case["batch"], hkv, cap, D), gen, dtype), "v": _randn((case["batch"], hkv, cap, D), gen, dtype),
            "starts": starts, "cos": cos, "sin": sin}


def _mlp_inputs(case, seed):
    gen, dtype = _gen(seed), torch.bfloat16
    hidden, _, _, inter, _, _ = MODELS[case["model"]]
    return {"h": _randn((case["rows"], hidden), gen, dtype), "residual": _randn((case["rows"], hidden), gen, dtype),
            "gate_up": _randn((2 * inter, hidden), gen, dtype, hidden ** -0.5),
            "down": _randn((hidden, inter), gen, dtype, inter ** -0.5), "norm": _norm_w(hidden, gen, dtype)}


def _select_inputs(case, seed):
    gen = _gen(seed)
    logits = _randn((case["rows"], case["vocab"]), gen, torch.bfloat16, 2.5)
    return {"logits": logits, "wide": logits.float(), "k": case["k"]}


INPUTS = {"step": _step_inputs, "decode": _decode_inputs, "prompt": _prompt_inputs, "attn": _attn_inputs,
          "mlp": _mlp_inputs, "select": _select_inputs}


def prepare(case, seed):
    s = INPUTS[case["kind"]](case, seed)
    s["kind"] = case["kind"]
    if case["kind"] == "step":
        hidden, hq, hkv, inter, _, family = MODELS[case["model"]]
        cfg = ModelConfig(hidden=hidden, num_heads=hq, num_kv_heads=hkv, intermediate=inter,
                          num_layers=case["layers"], family=family, rope_theta=THETA, rms_norm_eps=EPS,
                          max_position=s["cap"])
        model = DecoderModel(cfg, s["layers"], s["final_norm"], s["lm_head"], case["batch"], s["cap"])
        for i, (k, v) in enumerate(s.pop("caches")):
            model.k[i].copy_(k)
            model.v[i].copy_(v)
        s["start"] = _ints(s["lens"])
        model.lengths.copy_(s["start"])
        model.host_lengths[:] = s["lens"]
        s["model"], s["graph"] = model, DecodeGraph(model)
    elif case["kind"] == "decode":
        s["kv_len"], s["max_kv"] = _ints(s["lens"]), int(s["lens"].max())
        if s["table"] is not None:
            s["table"] = _ints(s["table"])
    elif case["kind"] in ("prompt", "attn"):
        s["start"], s["max_start"] = _ints(s["starts"]), int(s["starts"].max())
        if case["kind"] == "prompt":
            s["hq"], s["hkv"], s["order"] = case["hq"], case["hkv"], ORDER[case["family"]]
        else:
            _, s["hq"], s["hkv"], _, _, family = MODELS[case["model"]]
            s["order"] = ORDER[family]
    return s


def run(s):
    kind = s["kind"]
    if kind == "step":
        # the same step again: the cache goes back to its length before it
        model, graph = s["model"], s["graph"]
        model.lengths.copy_(s["start"])
        model.host_lengths[:] = s["lens"]
        graph.x.copy_(s["x"])
        graph.positions.copy_(s["start"])
        return graph.replay()
    if kind == "decode":
        if s["table"] is not None:
            return ops.attention_decode_paged(s["q"], s["k"], s["v"], s["table"], s["kv_len"], s["max_kv"])
        return ops.attention_decode(s["q"], s["k"], s["v"], s["kv_len"], s["max_kv"])
    if kind == "prompt":
        S = s["qkv"].shape[1]
        q = ops.qk_norm_rope_append(s["qkv"], s["cos"], s["sin"], s["start"], s["k"], s["v"], s["start"],
                                    s["max_start"] + S, s["hq"], s["hkv"], s["q_norm"], s["k_norm"], EPS, s["order"])
        return {"attn": ops.attention_prefill(q, s["k"], s["v"], s["start"], s["max_start"]), "k": s["k"], "v": s["v"]}
    if kind == "attn":
        w, (B, S, H) = s["w"], s["x"].shape
        residual = s["x"].reshape(B * S, H).clone()
        h = ops.rms_norm(residual, w.input_norm, EPS)
        qkv = ops.linear(h, w.qkv, w.qkv_bias).view(B, S, -1)
        q = ops.qk_norm_rope_append(qkv, s["cos"], s["sin"], s["start"], s["k"], s["v"], s["start"],
                                    s["max_start"] + S, s["hq"], s["hkv"], w.q_norm, w.k_norm, EPS, s["order"])
        a = ops.attention_prefill(q, s["k"], s["v"], s["start"], s["max_start"])
        h = ops.add_rms_norm(residual, ops.linear(a.view(B * S, -1), w.o), w.post_norm, EPS)
        return {"h": h, "residual": residual, "k": s["k"], "v": s["v"]}
    if kind == "mlp":
        residual = s["residual"].clone()
        y = ops.linear(ops.linear_silu_mul(s["h"], s["gate_up"]), s["down"])
        return {"h": ops.add_rms_norm(residual, y, s["norm"], EPS), "residual": residual}
    return {"argmax": ops.argmax(s["logits"]), "topk": ops.topk_indices(s["wide"], s["k"])}


def work(case):
    kind = case["kind"]
    if kind == "step":
        hidden, hq, hkv, inter, _, _ = MODELS[case["model"]]
        B, L, lens = case["batch"], case["layers"], _lengths(case, 0)
        weights = L * hidden * ((2 * hq + 2 * hkv) * D + 3 * inter) + VOCAB * hidden
        rows = int(lens.sum()) + B
        return {"bytes": 2 * (weights + L * rows * hkv * D * 2 + B * (hidden + VOCAB)),
                "flops": 2 * B * weights + 4 * L * rows * hq * D}
    if kind == "decode":
        e, rows = 2 if case["dtype"] == "bf16" else 4, int(_lengths(case, 0).sum())
        return {"bytes": e * D * (2 * rows * case["hkv"] + 2 * case["batch"] * case["hq"]),
                "flops": 4 * rows * case["hq"] * D}
    if kind in ("prompt", "attn"):
        B, S, starts = case["batch"], case["seq"], _starts(case, 0)
        if kind == "prompt":
            hq, hkv, e, byt, flops = case["hq"], case["hkv"], 2 if case["dtype"] == "bf16" else 4, 0, 0
            byt = e * B * S * (hq + 2 * hkv) * D + e * B * S * hq * D            # qkv in, attention out
        else:
            hidden, hq, hkv, _, _, _ = MODELS[case["model"]]
            e, weights = 2, hidden * (2 * hq + 2 * hkv) * D
            byt, flops = e * (weights + 3 * B * S * hidden), 2 * B * S * weights  # x in, h and residual out
        byt += e * hkv * D * 2 * (int(starts.sum()) + B * S)                      # cached rows read, new ones written
        keys = sum(int(n) * S + S * (S + 1) // 2 for n in starts)
        return {"bytes": byt, "flops": flops + 4 * keys * hq * D}
    if kind == "mlp":
        hidden, _, _, inter, _, _ = MODELS[case["model"]]
        return {"bytes": 2 * (3 * hidden * inter + 4 * case["rows"] * hidden),
                "flops": 6 * case["rows"] * hidden * inter}
    return {"bytes": case["rows"] * (6 * case["vocab"] + 4 + 4 * case["k"]), "flops": 2 * case["rows"] * case["vocab"]}


def tolerance(case):
    """What another order of the sums shows, with room: a step's bf16 roundings
    travel through its layers (0.004 to 0.01 measured between two ways to sum
    the projections); one layer's outputs lie 0.002 to 0.007 from float64
    (largest difference 0.18 of the rms in attention, whose first rows are far
    larger than its others, and 0.03 elsewhere), f32 attention 4e-7 (6e-6)."""
    kind = case["kind"]
    if kind == "select":
        return "exact"
    if kind == "step":
        return {"rel": 0.03, "max": 0.15}
    if case.get("dtype") == "f32":
        return {"rel": 2e-6, "max": 3e-5}
    return {"rel": 0.015, "max": 0.4 if kind == "prompt" else 0.2 if kind == "decode" else 0.08}


# ---------------------------------------------------------------- in float64

def _rms(x, w):
    y = x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS)
    return y if w is None else y * w.double()


def _rope(x, cos, sin):
    """x [B, S, heads, D]; cos, sin [B, S, D / 2]."""
    c, s, (a, b) = cos.double()[:, :, None], sin.double()[:, :, None], x.split(D // 2, -1)
    return torch.cat((a * c - b * s, b * c + a * s), -1)


def _heads(x, w, cos, sin, family):
    if family == "qwen2":
        return _rope(x, cos, sin)
    return _rope(_rms(x, w), cos, sin) if family == "qwen3" else _rms(_rope(x, cos, sin), w)


def _append(qkv, k, v, starts, cos, sin, hq, hkv, q_norm, k_norm, family):
    """Rotated q [B, S, hq, D]; the new rows go into the float64 caches k, v."""
    B, S, _ = qkv.shape
    rows = torch.stack([torch.arange(int(n), int(n) + S) for n in starts]).to(cos.device)
    cos, sin = cos[rows], sin[rows]
    q, kn, vn = qkv.view(B, S, -1, D).split((hq, hkv, hkv), 2)
    kn = _heads(kn, k_norm, cos, sin, family)
    for b, n in enumerate(starts):
        k[b, :, int(n):int(n) + S] = kn[b].transpose(0, 1)
        v[b, :, int(n):int(n) + S] = vn[b].transpose(0, 1)
    return _heads(q, q_norm, cos, sin, family)


def _attend(q, k, v, start):
    """q [S, hq, D] against k, v [hkv, start + S, D], causal: [S, hq D]."""
    S, hq, _ = q.shape
    n, g = k.shape[1], hq // k.shape[0]
    out = torch.empty((S, hq, D), dtype=torch.float64, device=q.device)
    hide = torch.arange(n, device=q.device)[None, :] > start + torch.arange(S, device=q.device)[:, None]
    for h in range(hq):
        s = (q[:, h] @ k[h // g].T) * D ** -0.5
        out[:, h] = torch.softmax(s.masked_fill_(hide, -math.inf), -1) @ v[h // g]
    return out.reshape(S, hq * D)


def _attend_one(q, k, v):
    """q [hq, D] against every row of k, v [hkv, n, D]: [hq D]."""
    s = torch.softmax(q.view(k.shape[0], -1, D) @ k.transpose(1, 2) * D ** -0.5, -1)
    return (s @ v).reshape(-1)


def _exact_step(case, seed):
    s = _step_inputs(case, seed)
    _, hq, hkv, _, _, family = MODELS[case["model"]]
    B, lens = case["batch"], s["lens"]
    cos, sin = _tables(torch.bfloat16, s["cap"], family == "qwen2")
    at = _ints(lens).long()
    cos, sin = cos[at][:, None], sin[at][:, None]
    x = s["x"].double()[:, 0]
    for w, (kc, vc) in zip(s["layers"], s["caches"]):
        h = _rms(x, w.input_norm) @ w.qkv.double().T
        h = h if w.qkv_bias is None else h + w.qkv_bias.double()
        q, kn, vn = h.view(B, 1, -1, D).split((hq, hkv, hkv), 2)
        q, kn = _heads(q, w.q_norm, cos, sin, family), _heads(kn, w.k_norm, cos, sin, family)
        a = []
        for b in range(B):
            n = int(lens[b])
            k = torch.cat((kc[b, :, :n].double(), kn[b].transpose(0, 1)), 1)
            v = torch.cat((vc[b, :, :n].double(), vn[b].transpose(0, 1)), 1)
            a.append(_attend_one(q[b, 0], k, v))
        x = x + torch.stack(a) @ w.o.double().T
        gate, up = (_rms(x, w.post_norm) @ w.gate_up.double().T).chunk(2, -1)
        x = x + (torch.nn.functional.silu(gate) * up) @ w.down.double().T
    return (_rms(x, s["final_norm"]) @ s["lm_head"].double().T)[:, None]


def _exact_decode(case, seed):
    s, out = _decode_inputs(case, seed), []
    for b, n in enumerate(s["lens"]):
        if s["table"] is None:
            k, v = s["k"][b, :, :n], s["v"][b, :, :n]
        else:
            at = torch.as_tensor(s["table"][b, :-(-n // 256)], device=s["k"].device).long()
            k, v = (p[at].transpose(0, 1).reshape(case["hkv"], -1, D)[:, :n] for p in (s["k"], s["v"]))
        out.append(_attend_one(s["q"][b].double(), k.double(), v.double()))
    return torch.stack(out)[:, None]


def _exact_prompt(case, seed):
    s = _prompt_inputs(case, seed)
    k, v, S = s["k"].double(), s["v"].double(), case["seq"]
    q = _append(s["qkv"].double(), k, v, s["starts"], s["cos"], s["sin"], case["hq"], case["hkv"], s["q_norm"],
                s["k_norm"], case["family"])
    attn = [_attend(q[b], k[b, :, :n + S], v[b, :, :n + S], int(n)) for b, n in enumerate(s["starts"])]
    return {"attn": torch.stack(attn), "k": k, "v": v}


def _exact_attn(case, seed):
    s, (_, hq, hkv, _, _, family) = _attn_inputs(case, seed), MODELS[case["model"]]
    w, k, v, S = s["w"], s["k"].double(), s["v"].double(), case["seq"]
    x = s["x"].double()
    qkv = _rms(x, w.input_norm) @ w.qkv.double().T
    qkv = qkv if w.qkv_bias is None else qkv + w.qkv_bias.double()
    q = _append(qkv, k, v, s["starts"], s["cos"], s["sin"], hq, hkv, w.q_norm, w.k_norm, family)
    attn = [_attend(q[b], k[b, :, :n + S], v[b, :, :n + S], int(n)) for b, n in enumerate(s["starts"])]
    residual = (x + torch.stack(attn) @ w.o.double().T).view(case["batch"] * S, -1)
    return {"h": _rms(residual, w.post_norm), "residual": residual, "k": k, "v": v}


def _exact_mlp(case, seed):
    s = _mlp_inputs(case, seed)
    gate, up = (s["h"].double() @ s["gate_up"].double().T).chunk(2, -1)
    residual = s["residual"].double() + (torch.nn.functional.silu(gate) * up) @ s["down"].double().T
    return {"h": _rms(residual, s["norm"]), "residual": residual}


def _exact_select(case, seed):
    s = _select_inputs(case, seed)
    order = torch.sort(s["wide"].double(), dim=-1, descending=True, stable=True).indices.int()
    return {"argmax": order[:, 0].contiguous(), "topk": order[:, :s["k"]].contiguous()}


EXACT = {"step": _exact_step, "decode": _exact_decode, "prompt": _exact_prompt, "attn": _exact_attn,
         "mlp": _exact_mlp, "select": _exact_select}


def exact(case, seed):
    with torch.no_grad():
        return EXACT[case["kind"]](case, seed)
