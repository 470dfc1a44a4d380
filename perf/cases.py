"""Performance cases of the fused projections and of the modules built on them.

Each case is one pass of work that a program using this package does, through
its public entry points, at the Qwen3-0.6B/4B/8B shapes that the benchmark and
the tests use:

- ``call``: one projection call (``triton_fused_qkv``,
  ``triton_fused_gate_up_silu``, ``fused_linear`` and the int8 and RMSNorm
  forms), as an eager engine issues it.
- ``projections``: the four projections of each decoder layer (QKV, ``o``,
  gate-up, ``down``) on inputs of their own, eagerly (prefill) or from one HIP
  graph (a decode or spec-verify step over several layers' weights).
- ``attention``: ``TritonAttention.forward`` of a swapped model: norm + QKV,
  QK-norm, RoPE, cache write, attention, ``o``.
- ``ffn``: ``TritonFFN.forward`` of a swapped model: norm + gate-up + ``down``.
- ``model``: one decode or verify step of a swapped model from a ``StepGraph``,
  logits out.
- ``quantize``: ``quantize_w8_per_row``, the swap-time packing of one weight.

Activations are N(0, 1), projection weights N(0, 0.02), norm weights near 1,
cached keys and values N(0, 1) (what normalised keys and x.Wv give).
"""

from __future__ import annotations

import math

import torch

from llms_amd import harness
from llms_amd import kernels as fk

DEV = "cuda"
EPS = 1e-6

# (hidden, query heads, key/value heads, head size, FFN width)
SHAPES = {
    "0.6b": (1024, 16, 8, 128, 3072),
    "4b": (2560, 32, 8, 128, 9728),
    "8b": (4096, 32, 8, 128, 12288),
}


def listed():
    return [
        # The smallest call: an eager engine's QKV projection of one token on
        # the smallest model. Launch and host cost count.
        {"name": "qkv-0.6b-one-token", "kind": "call", "op": "qkv", "M": 1, "K": 1024, "n_q": 2048,
         "n_k": 1024, "int8": False, "norm": False},
        # Greedy decoding: one token through every projection of 10 layers,
        # norms fused in, from one HIP graph.
        {"name": "decode-4b", "kind": "projections", "model": "4b", "M": 1, "layers": 10,
         "int8": False, "norm": True, "graph": True},
        # Speculative verification of a 4-token draft on int8 weights.
        {"name": "verify-4b-int8", "kind": "projections", "model": "4b", "M": 4, "layers": 10,
         "int8": True, "norm": True, "graph": True},
        # A batch of 64 sequences decoding together: the FFN of one layer.
        {"name": "ffn-8b-batch64", "kind": "ffn", "model": "8b", "M": 64, "int8": False},
        # One decode step's attention layer of the eager engine, 2047 tokens
        # already in the cache.
        {"name": "attn-4b-decode", "kind": "attention", "model": "4b", "B": 1, "T": 1, "pos": 2047,
         "seq": 4096, "int8": False},
        # A prompt of ordinary length through the attention layer.
        {"name": "attn-4b-prompt", "kind": "attention", "model": "4b", "B": 1, "T": 1000, "pos": 0,
         "seq": 2048, "int8": False},
        # A whole decode step (4 layers, the full vocabulary) from a StepGraph.
        {"name": "model-step", "kind": "model", "model": "4b", "layers": 4, "vocab": 151936, "T": 1,
         "pos": 1500, "seq": 2048, "int8": False},
        # Prefill of a 2048-token prompt: one layer's projections.
        {"name": "prefill-4b", "kind": "projections", "model": "4b", "M": 2048, "layers": 1,
         "int8": False, "norm": True, "graph": False},
        # The same on int8 weights, a prompt length that fills no tile.
        {"name": "prefill-4b-int8", "kind": "projections", "model": "4b", "M": 1500, "layers": 1,
         "int8": True, "norm": True, "graph": False},
        # The largest: 4096 prompt rows on the largest model.
        {"name": "prefill-8b", "kind": "projections", "model": "8b", "M": 4096, "layers": 1,
         "int8": False, "norm": False, "graph": False},
        # Rows that no vector width divides (K = 2541) and a ragged output.
        {"name": "gate-up-ragged", "kind": "call", "op": "gate_up", "M": 300, "K": 2541, "N": 9700,
         "int8": False, "norm": False},
        # Swapping in int8: packing one FFN weight.
        {"name": "quantize-8b-gate", "kind": "quantize", "N": 12288, "K": 4096},
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["call", "call", "ragged", "step", "prefill", "attention", "attention",
                       "ffn", "model", "quantize"])
    model = rng.choice(list(SHAPES))
    hidden, hq, hk, d, inter = SHAPES[model]
    int8 = rng.random() < 0.4
    if kind in ("call", "ragged"):
        op = rng.choice(["qkv", "gate_up", "linear"])
        c = {"kind": "call", "op": op, "M": _log(rng, 1, 2048), "int8": int8,
             "norm": op != "linear" and rng.random() < 0.5}
        if kind == "ragged":
            c["M"] = _log(rng, 1, 1024)
            hidden, inter = rng.randrange(1000, 4097), rng.randrange(1000, 10001)
            nq, nk = 4 * rng.randrange(128, 1025), rng.randrange(64, 1025)
        else:
            nq, nk = hq * d, hk * d
        if op == "qkv":
            return dict(c, K=hidden, n_q=nq, n_k=nk)
        if op == "gate_up":
            return dict(c, K=hidden, N=inter)
        return dict(c, K=inter, N=hidden) if rng.random() < 0.5 else dict(c, K=nq, N=hidden)
    if kind == "step":
        return {"kind": "projections", "model": model, "M": _log(rng, 1, 16),
                "layers": rng.randrange(4, 11), "int8": int8, "norm": rng.random() < 0.5,
                "graph": True}
    if kind == "prefill":
        return {"kind": "projections", "model": model, "M": _log(rng, 17, 4096), "layers": 1,
                "int8": int8, "norm": rng.random() < 0.5, "graph": False}
    if kind == "attention":
        seq = 4096
        if rng.random() < 0.5:  # decode, batched decode, verification
            T, B = rng.choice([1, 1, 1, 2, 4, 5, 9]), _log(rng, 1, 8)
            pos = _log(rng, 16, seq - T)
        else:  # prompts, and later chunks of one
            T, B = _log(rng, 16, 2048), 1
            pos = rng.choice([0, 0, _log(rng, 1, seq - T)])
        return {"kind": "attention", "model": model, "B": B, "T": T, "pos": pos, "seq": seq,
                "int8": int8}
    if kind == "ffn":
        return {"kind": "ffn", "model": model, "M": _log(rng, 1, 2048), "int8": int8}
    if kind == "model":
        T = rng.choice([1, 1, 1, 2, 4, 8])
        return {"kind": "model", "model": model, "layers": rng.randrange(2, 5),
                "vocab": rng.choice([32000, 151936]), "T": T, "pos": _log(rng, 16, 2048 - 2 * T),
                "seq": 2048, "int8": int8}
    return {"kind": "quantize", "N": _log(rng, 512, 12288), "K": _log(rng, 512, 12288)}


# ---------------------------------------------------------------- inputs


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, scale=1.0):
    return (torch.randn(*shape, generator=g, device=DEV) * scale).to(torch.bfloat16)


def _weight(g, n, k):
    return _randn(g, n, k, scale=0.02)


def _norm_weight(g, k):
    return (1.0 + 0.05 * torch.randn(k, generator=g, device=DEV)).to(torch.bfloat16)


def _pack(w):
    """Per-row symmetric int8 and its scales, as ``quantize_w8_per_row`` defines them."""
    s = w.float().abs().amax(dim=1) / 127.0
    q = torch.where(s[:, None] > 0, (w.float() / s[:, None]).round().clamp(-127, 127), 0.0)
    return q.to(torch.int8), s


def _call_inputs(c, seed):
    g = _gen(seed)
    n = {"qkv": lambda: [c["n_q"] + 2 * c["n_k"]], "gate_up": lambda: [c["N"], c["N"]],
         "linear": lambda: [c["N"]]}[c["op"]]()
    d = {"x": _randn(g, c["M"], c["K"]), "w": [_weight(g, i, c["K"]) for i in n]}
    if c["norm"]:
        d["gamma"] = _norm_weight(g, c["K"])
    if c["int8"]:
        d["w"] = [t for w in d["w"] for t in _pack(w)]
    return d


def _layer_calls(c):
    """The projection calls of one layer, as ``call`` cases."""
    hidden, hq, hk, d, inter = SHAPES[c["model"]]
    base = {"M": c["M"], "int8": c["int8"]}
    return [dict(base, op="qkv", K=hidden, n_q=hq * d, n_k=hk * d, norm=c["norm"]),
            dict(base, op="linear", K=hq * d, N=hidden, norm=False),
            dict(base, op="gate_up", K=hidden, N=inter, norm=c["norm"]),
            dict(base, op="linear", K=inter, N=hidden, norm=False)]


def _all_calls(c, seed):
    """(call case, its inputs) of every projection of a ``projections`` case."""
    return [(k, _call_inputs(k, 1000 * seed + 10 * i + j))
            for i in range(c["layers"]) for j, k in enumerate(_layer_calls(c))]


def _cfg(c, layers, vocab):
    hidden, hq, hk, d, inter = SHAPES[c["model"]]
    return harness.Cfg(vocab_size=vocab, hidden_size=hidden, num_hidden_layers=layers,
                       num_attention_heads=hq, num_key_value_heads=hk, head_dim=d,
                       intermediate_size=inter, max_position_embeddings=c.get("seq", 64),
                       rms_norm_eps=EPS, rope_theta=1000000.0)


def _model_state(c, layers, vocab, seed):
    """The bf16 weights of a model of case c, by their names in the engine."""
    hidden, hq, hk, d, inter = SHAPES[c["model"]]
    g = _gen(seed)
    st = {"embed.weight": _weight(g, vocab, hidden), "final_norm.weight": _norm_weight(g, hidden)}
    for i in range(layers):
        p = "layers.%d." % i
        st[p + "norm1.weight"] = _norm_weight(g, hidden)
        st[p + "norm2.weight"] = _norm_weight(g, hidden)
        st[p + "attn.q.weight"] = _weight(g, hq * d, hidden)
        st[p + "attn.k.weight"] = _weight(g, hk * d, hidden)
        st[p + "attn.v.weight"] = _weight(g, hk * d, hidden)
        st[p + "attn.o.weight"] = _weight(g, hidden, hq * d)
        st[p + "attn.q_norm.weight"] = _norm_weight(g, d)
        st[p + "attn.k_norm.weight"] = _norm_weight(g, d)
        st[p + "ffn.gate.weight"] = _weight(g, inter, hidden)
        st[p + "ffn.up.weight"] = _weight(g, inter, hidden)
        st[p + "ffn.down.weight"] = _weight(g, hidden, inter)
    return st


def _model(c, layers, vocab, seed):
    """The engine model with every projection swapped for its fused form."""
    cfg = _cfg(c, layers, vocab)
    with torch.device(DEV):
        m = harness.Qwen3Model(cfg)
    m = m.to(device=DEV, dtype=torch.bfloat16).eval()
    m.load_state_dict(_model_state(c, layers, vocab, seed), strict=False)
    return fk.apply_triton_kernels(m, int8=c["int8"], linear_down_o=True, fuse_norm=True)


def _cache_values(c, layers, B, seed):
    """Keys and values [B, H, pos, D] of the tokens before this pass, by layer."""
    _, _, hk, d, _ = SHAPES[c["model"]]
    g = _gen(seed + 7777)
    return [(_randn(g, B, hk, c["pos"], d), _randn(g, B, hk, c["pos"], d)) for _ in range(layers)]


def _fill(cache, values, pos):
    for i, (k, v) in enumerate(values):
        cache.k[i][:, :, :pos] = k
        cache.v[i][:, :, :pos] = v


def _attention_x(c, seed):
    return _randn(_gen(seed + 5555), c["B"], c["T"], SHAPES[c["model"]][0])


def _ffn_x(c, seed):
    return _randn(_gen(seed + 5555), 1, c["M"], SHAPES[c["model"]][0])


def _tokens(c, seed):
    return torch.randint(0, c["vocab"], (1, c["T"]), generator=_gen(seed + 3333), device=DEV)


# ---------------------------------------------------------------- passes


def _call(c, d):
    x, w = d["x"], d["w"]
    if c["op"] == "linear":
        return (fk.fused_linear_w8 if c["int8"] else fk.fused_linear)(x, *w)
    if c["op"] == "gate_up":
        if c["norm"]:
            fn = fk.fused_rmsnorm_gate_up_silu_w8 if c["int8"] else fk.fused_rmsnorm_gate_up_silu
            return fn(x, d["gamma"], EPS, *w)
        return (fk.fused_gate_up_silu_w8 if c["int8"] else fk.triton_fused_gate_up_silu)(x, *w)
    n = {"n_q": c["n_q"], "n_k": c["n_k"]}
    if c["norm"]:
        fn = fk.fused_rmsnorm_qkv_w8 if c["int8"] else fk.fused_rmsnorm_qkv
        return fn(x, d["gamma"], EPS, *w, **n)
    return (fk.fused_qkv_w8 if c["int8"] else fk.triton_fused_qkv)(x, *w, **n)


def _capture(fn):
    """fn() captured in a HIP graph: the graph and the outputs its replays write."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


def prepare(case, seed):
    c = dict(case)
    kind = c["kind"]
    if kind == "call":
        return {"case": c, "in": _call_inputs(c, seed)}
    if kind == "projections":
        calls = _all_calls(c, seed)
        state = {"case": c, "calls": calls}
        if c["graph"]:
            with torch.inference_mode():
                state["graph"], state["out"] = _capture(lambda: [_call(k, d) for k, d in calls])
        return state
    if kind == "attention":
        m = _model(c, 1, 32, seed)
        cache = m.alloc_cache(c["seq"], max_batch=c["B"])
        _fill(cache, _cache_values(c, 1, c["B"], seed), c["pos"])
        cos = m.rope_cos[c["pos"]:c["pos"] + c["T"]]
        sin = m.rope_sin[c["pos"]:c["pos"] + c["T"]]
        return {"case": c, "attn": m.layers[0].attn, "cache": cache, "cos": cos, "sin": sin,
                "x": _attention_x(c, seed)}
    if kind == "ffn":
        return {"case": c, "ffn": _model(c, 1, 32, seed).layers[0].ffn, "x": _ffn_x(c, seed)}
    if kind == "model":
        m = _model(c, c["layers"], c["vocab"], seed)
        cache = m.alloc_cache(c["seq"])
        step = harness.StepGraph(m, cache, T=c["T"])
        _fill(cache, _cache_values(c, c["layers"], 1, seed), c["pos"])
        return {"case": c, "step": step, "cache": cache, "ids": _tokens(c, seed)}
    return {"case": c, "w": _weight(_gen(seed), c["N"], c["K"])}


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "model":
        logits = state["step"](state["ids"], c["pos"])
        # the keys and values this step wrote
        t = slice(c["pos"], c["pos"] + c["T"])
        return [logits] + [kv[i][:, :, t] for i in range(c["layers"])
                           for kv in (state["cache"].k, state["cache"].v)]
    if kind == "projections" and c["graph"]:
        state["graph"].replay()
        return state["out"]
    with torch.inference_mode():
        if kind == "call":
            return _call(c, state["in"])
        if kind == "projections":
            return [_call(k, d) for k, d in state["calls"]]
        if kind == "attention":
            cache = state["cache"]
            y = state["attn"](state["x"], kv_cache=cache, layer_idx=0, cos=state["cos"],
                              sin=state["sin"], start_pos=c["pos"])
            return [y, cache.k[0], cache.v[0]]
        if kind == "ffn":
            return state["ffn"](state["x"])
        return fk.quantize_w8_per_row(state["w"])


# ---------------------------------------------------------------- work


def _call_work(c):
    cols = {"qkv": lambda: c["n_q"] + 2 * c["n_k"], "gate_up": lambda: 2 * c["N"],
            "linear": lambda: c["N"]}[c["op"]]()
    out = c["N"] if c["op"] == "gate_up" else cols
    wb = cols * (c["K"] + 4) if c["int8"] else 2 * cols * c["K"]
    return {"bytes": wb + 2 * c["M"] * (c["K"] + out) + (2 * c["K"] if c["norm"] else 0),
            "flops": 2 * c["M"] * c["K"] * cols}


def _sum(parts):
    parts = list(parts)
    return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}


def _attention_core_work(c, B, T):
    """Keys and values read and written, and the visible query-key pairs."""
    _, hq, hk, d, _ = SHAPES[c["model"]]
    pairs = T * c["pos"] + T * (T + 1) // 2
    return {"bytes": 2 * 2 * B * hk * d * (c["pos"] + 2 * T), "flops": 4 * B * hq * d * pairs}


def _module_calls(c, M, which):
    calls = _layer_calls({"model": c["model"], "M": M, "int8": c["int8"], "norm": True})
    return [_call_work(k) for k in calls[which]]


def work(case):
    c = case
    if c["kind"] == "call":
        return _call_work(c)
    if c["kind"] == "projections":
        one = _sum(_call_work(k) for k in _layer_calls(c))
        return {k: v * c["layers"] for k, v in one.items()}
    if c["kind"] == "attention":
        # in and out once: x and y of the two projections, but not the
        # intermediate q, k, v and attention rows
        hidden, hq, hk, d, _ = SHAPES[c["model"]]
        M = c["B"] * c["T"]
        w = _sum(_module_calls(c, M, slice(0, 2)) + [_attention_core_work(c, c["B"], c["T"])])
        w["bytes"] -= 2 * M * (2 * hq + 2 * hk) * d
        return w
    if c["kind"] == "ffn":
        w = _sum(_module_calls(c, c["M"], slice(2, 4)))
        w["bytes"] -= 2 * 2 * c["M"] * SHAPES[c["model"]][4]
        return w
    if c["kind"] == "model":
        hidden = SHAPES[c["model"]][0]
        parts = _module_calls(c, c["T"], slice(0, 4)) + [_attention_core_work(c, 1, c["T"])]
        w = {k: v * c["layers"] for k, v in _sum(parts).items()}
        w["bytes"] += 2 * c["vocab"] * (hidden + c["T"])
        w["flops"] += 2 * c["T"] * c["vocab"] * hidden
        return w
    return {"bytes": c["N"] * (3 * c["K"] + 4), "flops": 3 * c["N"] * c["K"]}


# ---------------------------------------------------------------- correctness


def tolerance(case):
    """bf16 outputs: the last rounding alone is 1.7e-3 (rel. 2-norm); a
    projection sums in fp32, the gate-up epilogue rounds four times, the
    attention layer about eight, and a model step carries every layer's
    roundings into its logits."""
    c = case
    if c["kind"] == "quantize":
        # whole values: q of a tie may fall either way with another division
        return {"rel": 1e-6, "max": 1e-6, "differ": 1e-4}
    if c["kind"] == "model":
        return {"rel": 3e-2, "max": 0.25}
    if c["kind"] in ("attention", "ffn"):
        return {"rel": 1.5e-2, "max": 0.12}
    return {"rel": 1e-2, "max": 0.08}


def _f64(t):
    return t.to(torch.float64)


def _norm64(x, gamma):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * _f64(gamma)


def _silu64(g):
    return g / (1.0 + torch.exp(-g))


def _w64(c, w):
    """The weights of a call in 64 bits: bf16 as they are, int8 times their scales."""
    if not c["int8"]:
        return [_f64(t) for t in w]
    return [_f64(q) * _f64(s)[:, None] for q, s in zip(w[::2], w[1::2])]


def _call64(c, d):
    x, w = _f64(d["x"]), _w64(c, d["w"])
    if c["norm"]:
        x = _norm64(x, d["gamma"])
    if c["op"] == "gate_up":
        return _silu64(x @ w[0].T) * (x @ w[1].T)
    y = x @ w[0].T
    return tuple(y.split([c["n_q"], c["n_k"], c["n_k"]], dim=-1)) if c["op"] == "qkv" else y


def _rope64(t, pos, theta=1000000.0):
    """Rotate-half RoPE of t [B, H, T, D] at positions pos .., with the tables
    rounded to bf16 as the engine holds them."""
    T, d = t.shape[2], t.shape[3]
    inv = theta ** (-torch.arange(0, d, 2, dtype=torch.float32) / d)
    ang = torch.arange(pos + T, dtype=torch.float32)[pos:, None] * inv[None, :]
    ang = torch.cat([ang, ang], dim=-1)
    cos = _f64(ang.cos().to(torch.bfloat16)).to(t.device)
    sin = _f64(ang.sin().to(torch.bfloat16)).to(t.device)
    h = d // 2
    return t * cos + torch.cat((-t[..., h:], t[..., :h]), dim=-1) * sin


def _proj64(c, x, w):
    return x @ _w64(c, list(_pack(w)) if c["int8"] else [w])[0].T


def _attention64(c, st, p, x, kv, pos):
    """The attention layer of x [B, T, hidden] (64 bits); its new keys and values too."""
    _, hq, hk, d, _ = SHAPES[c["model"]]
    B, T, _ = x.shape
    xn = _norm64(x, st[p + "norm1.weight"])
    heads = lambda n, h: _proj64(c, xn, st[p + "attn.%s.weight" % n]).view(B, T, h, d)  # noqa: E731
    q = _rope64(_norm64(heads("q", hq), st[p + "attn.q_norm.weight"]).transpose(1, 2), pos)
    k = _rope64(_norm64(heads("k", hk), st[p + "attn.k_norm.weight"]).transpose(1, 2), pos)
    v = heads("v", hk).transpose(1, 2)
    fullk, fullv = torch.cat([_f64(kv[0]), k], dim=2), torch.cat([_f64(kv[1]), v], dim=2)
    rows = torch.arange(pos, pos + T, device=x.device)[:, None]
    hide = torch.arange(pos + T, device=x.device)[None, :] > rows
    out = torch.empty(B, T, hq * d, dtype=torch.float64, device=x.device)
    for b in range(B):
        for h in range(hq):
            s = (q[b, h] @ fullk[b, h * hk // hq].T) * d ** -0.5
            s = s.masked_fill(hide, float("-inf"))
            out[b, :, h * d:(h + 1) * d] = torch.softmax(s, dim=-1) @ fullv[b, h * hk // hq]
    return _proj64(c, out, st[p + "attn.o.weight"]), k, v


def _ffn64(c, st, p, x):
    xn = _norm64(x, st[p + "norm2.weight"])
    h = _silu64(_proj64(c, xn, st[p + "ffn.gate.weight"])) * _proj64(c, xn, st[p + "ffn.up.weight"])
    return _proj64(c, h, st[p + "ffn.down.weight"])


def exact(case, seed):
    c = dict(case)
    with torch.inference_mode():
        if c["kind"] == "call":
            return _call64(c, _call_inputs(c, seed))
        if c["kind"] == "projections":
            return [_call64(k, d) for k, d in _all_calls(c, seed)]
        if c["kind"] == "ffn":
            return _ffn64(c, _model_state(c, 1, 32, seed), "layers.0.", _f64(_ffn_x(c, seed)))
        if c["kind"] == "attention":
            _, _, hk, d, _ = SHAPES[c["model"]]
            kv = _cache_values(c, 1, c["B"], seed)[0]
            y, k, v = _attention64(c, _model_state(c, 1, 32, seed), "layers.0.",
                                   _f64(_attention_x(c, seed)), kv, c["pos"])
            caches = []
            for old, new in zip(kv, (k, v)):
                t = torch.zeros(c["B"], hk, c["seq"], d, dtype=torch.float64, device=DEV)
                t[:, :, :c["pos"]] = _f64(old)
                t[:, :, c["pos"]:c["pos"] + c["T"]] = new
                caches.append(t)
            return [y] + caches
        if c["kind"] == "model":
            st = _model_state(c, c["layers"], c["vocab"], seed)
            h = _f64(st["embed.weight"][_tokens(c, seed)])
            written = []
            for i, kv in enumerate(_cache_values(c, c["layers"], 1, seed)):
                p = "layers.%d." % i
                y, k, v = _attention64(c, st, p, h, kv, c["pos"])
                h = h + y
                h = h + _ffn64(c, st, p, h)
                written += [k, v]
            h = _norm64(h, st["final_norm.weight"])
            return [h @ _f64(st["embed.weight"]).T] + written
        q, s = _pack(_weight(_gen(seed), c["N"], c["K"]))
        return q, _f64(s)
