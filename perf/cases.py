"""The work that a serving program has this package do, as cases that can be timed and checked.

Every case calls the public entry points (leanstack_amd.dispatch, .kernels, .stack, .kv_cache) on the
Qwen3-4B geometry, with weights in the packed layout and all inputs on the GPU.  Kinds:

  token         one greedy decode token of the whole model, replayed as one HIP graph (stack.DecodeStep):
                what a decode loop runs for every token it generates.
  decode_layer  one decode token through one layer, called eagerly (semantic_qwen_decode_layer_forward):
                a decode loop that keeps the reference runtime's per-layer calls.
  vector_layer  the same token through the reference's narrower per-layer names (QKV vector, cache append,
                attention + o_proj, MLP epilogue): a runtime that only swaps its dispatch table.
  layer         rows of one sequence through one layer's norm, QKV heads, o_proj and MLP, with the attention
                output given (the caller's causal attention runs between the calls).  2..16 rows are a
                speculative verify, more are a prefill; the small, repeated row counts are captured as a
                graph, prompts of any length are called eagerly.
  head          the greedy lm_head over 1..16 normed rows, with its fp32 scores.
"""

from __future__ import annotations

import math
from types import SimpleNamespace

import torch

from leanstack_amd import _lib, dispatch, kernels
from leanstack_amd.geometry import QWEN3_4B as G
from leanstack_amd.kv_cache import ArenaKVCache
from leanstack_amd.layout import PackedWeight
from leanstack_amd.stack import DecodeStep, LayerProjections

DEV = "cuda"
H, I, D, V = G.hidden_size, G.intermediate_size, G.head_dim, G.vocab_size
NQ, NKV = G.num_attention_heads, G.num_key_value_heads
EPS = G.rms_norm_eps
SCALE = D ** -0.5
SHAPES = {"qkv": (G.qkv_dim, H), "o": (H, G.q_dim), "gate_up": (2 * I, H), "down": (H, I)}
LAYOUTS = {"qkv": _lib.LAYOUT_MFMA16X32, "o": _lib.LAYOUT_MFMA16X32, "gate_up": _lib.LAYOUT_MFMA16X32_GATEUP,
           "down": _lib.LAYOUT_MFMA16X32}
BUCKETS = (320, 576, 1088)  # prompt + new tokens of the decode_64_256, decode_64_512 and prefill_1024_64 profiles
GRAPH_ROWS = 64             # largest row count that a serving loop repeats often enough to keep a graph of


def listed() -> list[dict]:
    return [
        # the last token of a 1024-token prompt's 64 new ones: the model's step with a usual context
        {"name": "token_1088", "kind": "token", "rows": 1087, "capacity": 1088},
        # the longest context that the caches hold
        {"name": "token_16384", "kind": "token", "rows": 16383, "capacity": 16384},
        # the first tokens after a 64-token prompt, per-layer calls: the smallest call
        {"name": "decode_layer_64", "kind": "decode_layer", "rows": 64, "capacity": 320},
        # the same step through the narrower names, in the middle of a long answer
        {"name": "vector_layer_700", "kind": "vector_layer", "rows": 700, "capacity": 1088},
        # verify of four drafted tokens and the current one
        {"name": "verify_5", "kind": "layer", "m": 5, "graph": True},
        # verify of a longer draft
        {"name": "verify_12", "kind": "layer", "m": 12, "graph": True},
        # the shortest prompt bucket
        {"name": "prefill_64", "kind": "layer", "m": 64, "graph": True},
        # a ragged prompt
        {"name": "prefill_301", "kind": "layer", "m": 301, "graph": False},
        # the longest prompt bucket
        {"name": "prefill_1024", "kind": "layer", "m": 1024, "graph": False},
        {"name": "prefill_2048", "kind": "layer", "m": 2048, "graph": False},
        # a long prompt in one piece
        {"name": "prefill_8192", "kind": "layer", "m": 8192, "graph": False},
        # greedy tokens of a verify block, with their scores
        {"name": "head_5", "kind": "head", "m": 5},
    ]


def _spread(rng, low: int, high: int) -> int:
    """A whole number of [low, high], even over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng) -> dict:
    kind = rng.choice(("token", "decode_layer", "vector_layer", "layer", "layer", "layer", "layer", "layer", "head"))
    if kind == "token":
        capacity = rng.choice(BUCKETS + (4096, 16384))
        return {"kind": kind, "rows": _spread(rng, 1, capacity - 1), "capacity": capacity}
    if kind in ("decode_layer", "vector_layer"):
        capacity = rng.choice(BUCKETS + (4096,))
        return {"kind": kind, "rows": _spread(rng, 1, capacity - 1), "capacity": capacity}
    if kind == "head":
        return {"kind": kind, "m": rng.randint(1, 16), "bf16_logits": rng.random() < 0.3}
    m = _spread(rng, 2, 8192)
    return {"kind": kind, "m": m, "graph": m <= GRAPH_ROWS and rng.random() < 0.7}


# ------------------------------------------------------------------ inputs


def _normal(gen, shape, std=1.0, mean=0.0):
    return torch.empty(shape, device=DEV, dtype=torch.bfloat16).normal_(mean, std, generator=gen)


def _weights(gen, residual_std=0.02) -> dict[str, PackedWeight]:
    """One layer's projections, N(0, 0.02); the packed order of independent values is any order.
    residual_std: of the two that add to the residual stream."""
    out = {}
    for name, (n, k) in SHAPES.items():
        std = residual_std if name in ("o", "down") else 0.02
        out[name] = PackedWeight(_normal(gen, (n * k,), std), n, k, LAYOUTS[name])
    return out


def _rope_tables(positions: torch.Tensor):
    inv = 1.0 / (G.rope_theta ** (torch.arange(0, D, 2, device=DEV, dtype=torch.float32) / D))
    freqs = torch.outer(positions.float(), inv)
    return freqs.cos().to(torch.bfloat16), freqs.sin().to(torch.bfloat16)


def _layer_inputs(gen) -> SimpleNamespace:
    w = _weights(gen)
    return SimpleNamespace(w=w, ln_in=_normal(gen, (H,), 0.1, 1.0), ln_post=_normal(gen, (H,), 0.1, 1.0),
                           q_norm=_normal(gen, (D,), 0.1, 1.0), k_norm=_normal(gen, (D,), 0.1, 1.0))


def _token_inputs(case, seed) -> SimpleNamespace:
    """36 layers as a freshly initialised tied model has them: embeddings N(0, 1), the projections into the
    residual stream scaled by 1/sqrt(2 * layers).  Such a model's best next token is its input token by a wide
    margin, so the token does not hang on a rounding."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    n, cap = G.num_hidden_layers, case["capacity"]
    s = SimpleNamespace()
    s.layers = [_weights(gen, 0.02 / math.sqrt(2 * n)) for _ in range(n)]
    s.norms = _normal(gen, (n, 2, H), 0.1, 1.0)
    s.qk_norms = _normal(gen, (n, 2, D), 0.1, 1.0)
    s.final_norm = _normal(gen, (H,), 0.1, 1.0)
    s.embedding = _normal(gen, (V, H))
    s.k = torch.zeros((n, NKV, cap, D), device=DEV, dtype=torch.bfloat16)
    s.v = torch.zeros((n, NKV, cap, D), device=DEV, dtype=torch.bfloat16)
    for l in range(n):
        s.k[l, :, : case["rows"]] = _normal(gen, (NKV, case["rows"], D))
        s.v[l, :, : case["rows"]] = _normal(gen, (NKV, case["rows"], D))
    s.first = torch.randint(0, V, (1,), device=DEV, generator=gen)
    return s


def _step_inputs(case, seed) -> SimpleNamespace:
    gen = torch.Generator(device=DEV).manual_seed(seed)
    s = _layer_inputs(gen)
    s.hidden = _normal(gen, (1, 1, H))
    s.k = _normal(gen, (1, NKV, case["rows"], D))
    s.v = _normal(gen, (1, NKV, case["rows"], D))
    s.cos, s.sin = _rope_tables(torch.tensor([case["rows"]], device=DEV))
    return s


def _rows_inputs(case, seed) -> SimpleNamespace:
    gen = torch.Generator(device=DEV).manual_seed(seed)
    s = _layer_inputs(gen)
    s.hidden = _normal(gen, (1, case["m"], H))
    s.attn = _normal(gen, (1, case["m"], G.q_dim), 0.5)
    s.cos, s.sin = (t[None] for t in _rope_tables(torch.arange(case["m"], device=DEV)))
    return s


def _head_inputs(case, seed) -> SimpleNamespace:
    gen = torch.Generator(device=DEV).manual_seed(seed)
    return SimpleNamespace(w=PackedWeight(_normal(gen, (V * H,), 0.02), V, H), hidden=_normal(gen, (case["m"], H)))


# ------------------------------------------------------------------ what a program keeps, and its calls


def _graph(fn):
    """fn() as a graph, warmed on the stream that it is captured on."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = fn()
    return graph, out


def prepare(case: dict, seed: int):
    kind = case["kind"]
    if kind == "token":
        s = _token_inputs(case, seed)
        lm = PackedWeight.from_rowmajor(s.embedding)
        layers = [LayerProjections(w["qkv"], w["o"], w["gate_up"], w["down"]) for w in s.layers]
        step = DecodeStep(layers, s.norms, s.qk_norms, s.final_norm, lm, G, s.k, s.v, torch.device(DEV, 0))
        step.set_position(case["rows"])
        step.token.copy_(s.first)
        graph, _ = _graph(lambda: step.launch_next(s.embedding))
        return SimpleNamespace(kind=kind, step=step, graph=graph, first=s.first, rows=case["rows"], keep=s)
    if kind in ("decode_layer", "vector_layer"):
        s = _step_inputs(case, seed)
        cache = ArenaKVCache(1, NKV, D, case["capacity"], device=DEV)
        cache.write_rows(0, s.k, s.v)
        attention = SimpleNamespace(
            layer_idx=0, qkv_proj_weight=s.w["qkv"], o_proj_weight=s.w["o"], q_proj_out_dim=G.q_dim,
            k_proj_out_dim=G.kv_dim, num_attention_heads=NQ, num_key_value_heads=NKV,
            num_key_value_groups=NQ // NKV, head_dim=D, attention_scale=SCALE, q_norm_weight=s.q_norm,
            k_norm_weight=s.k_norm)
        layer = SimpleNamespace(attention=attention, input_layernorm_weight=s.ln_in,
                                post_attention_layernorm_weight=s.ln_post,
                                mlp=SimpleNamespace(gate_up_proj_weight=s.w["gate_up"], gate_proj_out_dim=I,
                                                    down_proj_weight=s.w["down"]))
        return SimpleNamespace(kind=kind, layer=layer, cache=cache, mark=cache.mark(), rows=case["rows"],
                               hidden=s.hidden, rope=(s.cos, s.sin))
    if kind == "layer":
        s = _rows_inputs(case, seed)
        s.kind = kind
        s.graph = None
        if case["graph"]:
            s.graph, s.out = _graph(lambda: _layer(s))
        return s
    s = _head_inputs(case, seed)
    s.kind = kind
    s.logits = torch.empty((case["m"], V), device=DEV, dtype=torch.float32)
    s.tokens = torch.empty((case["m"],), device=DEV, dtype=torch.long)
    s.ws = kernels.LmHeadWorkspace(case["m"], V, H, DEV)
    s.mode = _lib.LOGITS_BF16 if case.get("bf16_logits") else _lib.LOGITS_FP32
    return s


def _layer(s):
    normed = dispatch.qwen_rmsnorm(s.hidden, s.ln_in, EPS)
    q, k, v = dispatch._semantic_attention_qkv(normed, s.w["qkv"], G.q_dim, G.kv_dim, NQ, NKV, D, s.q_norm, s.k_norm,
                                               s.cos, s.sin, EPS)
    out = dispatch._semantic_post_attention_mlp(s.attn, s.hidden, s.w["o"], s.ln_post, s.w["gate_up"], I, s.w["down"],
                                                EPS)
    return {"q": q, "k": k, "v": v, "hidden": out}


def run(s):
    if s.kind == "token":
        s.step.set_position(s.rows)
        s.step.token.copy_(s.first)
        s.graph.replay()
        return {"token": s.step.token, "hidden": s.step.hidden[G.num_hidden_layers % 2],
                "k": s.step.k_cache[:, :, s.rows], "v": s.step.v_cache[:, :, s.rows]}
    if s.kind == "decode_layer":
        s.cache.rewind(s.mark)
        out = dispatch.semantic_qwen_decode_layer_forward(s.layer, s.hidden, s.cache, s.rope, EPS)
        k, v = s.cache.layer_tensors(0)
        return {"hidden": out, "k": k[:, s.rows], "v": v[:, s.rows]}
    if s.kind == "vector_layer":
        s.cache.rewind(s.mark)
        a = s.layer.attention
        residual = s.hidden.view(-1)
        q, k, v = dispatch._semantic_input_norm_attention_qkv_vector(
            residual, s.layer.input_layernorm_weight, a.qkv_proj_weight, a.q_proj_out_dim, a.k_proj_out_dim, NQ, NKV,
            D, a.q_norm_weight, a.k_norm_weight, s.rope[0][None], s.rope[1][None], EPS)
        s.cache.write_rows(0, k, v)
        keys, values = s.cache.attended(0)
        attn = dispatch._semantic_decode_attention_output_vector(q, keys, values, a.o_proj_weight, SCALE, NQ // NKV)
        m = s.layer.mlp
        out = dispatch._semantic_mlp_epilogue_vector(residual + attn, s.layer.post_attention_layernorm_weight,
                                                     m.gate_up_proj_weight, m.gate_proj_out_dim, m.down_proj_weight,
                                                     EPS)
        return {"hidden": out.view(1, 1, -1), "attn": attn, "q": q, "k": k, "v": v}
    if s.kind == "layer":
        if s.graph is None:
            return _layer(s)
        s.graph.replay()
        return s.out
    kernels.lm_head_argmax(s.hidden, s.w, logits_mode=s.mode, logits_out=s.logits, workspace=s.ws, out=s.tokens)
    return {"logits": s.logits, "tokens": s.tokens}


# ------------------------------------------------------------------ what a pass cannot do without


def work(case: dict) -> dict:
    kind = case["kind"]
    row = 2 * NKV * D * 2  # one cached key and value row
    if kind == "token":
        n, s = G.num_hidden_layers, case["rows"]
        return {"bytes": n * (G.layer_weight_bytes() + (s + 1) * row) + G.lm_head_bytes() + 4 * H,
                "flops": 2 * (n * (G.layer_params() + 2 * (s + 1) * NQ * D) + V * H)}
    if kind in ("decode_layer", "vector_layer"):
        s = case["rows"]
        return {"bytes": G.layer_weight_bytes() + (s + 1) * row + 4 * H,
                "flops": 2 * (G.layer_params() + 2 * (s + 1) * NQ * D)}
    m = case["m"]
    if kind == "head":
        return {"bytes": G.lm_head_call_bytes(m), "flops": 2 * m * V * H}
    # hidden and attention rows in, q / k / v and the layer's output rows out
    return {"bytes": G.layer_weight_bytes() + 2 * m * (2 * H + G.q_dim + G.qkv_dim), "flops": G.layer_flops(m)}


def tolerance(case: dict):
    kind = case["kind"]
    if kind == "head":  # fp32 sums of 2560 exact products; bf16_logits rounds them to bf16
        return {"rel": 4e-3, "max": 2e-2} if case.get("bf16_logits") else {"rel": 1e-5, "max": 1e-4}
    if kind == "token":  # 72 bf16 roundings of the residual stream, 0.017 off 64 bits in each of two paths
        return {"rel": 3e-2, "max": 0.5}
    # the projections' and norms' bf16 roundings are 0.0045 off 64 bits
    return {"rel": 1e-2, "max": 0.2}


# ------------------------------------------------------------------ the same in 64 bits


def _rows64(w: PackedWeight) -> torch.Tensor:
    """W[N, K] of a packed weight (16 x 32 tiles, lane l holding row l % 16 and 8 columns from 8 * (l // 16);
    gate and up row-blocks alternate), in 64 bits."""
    t = w.data.view(w.n // 16, w.k // 32, 4, 16, 8).permute(0, 3, 1, 2, 4).reshape(w.n, w.k)
    if w.layout == _lib.LAYOUT_MFMA16X32_GATEUP:
        t = t.view(-1, 2, 16, w.k).transpose(0, 1).reshape(w.n, w.k)
    return t.double()


def _linear64(x, w):
    return x @ _rows64(w).t()


def _norm64(x, weight):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * weight.double()


def _rope64(t, cos, sin):
    a, b = t.chunk(2, dim=-1)
    c, s = cos.double(), sin.double()
    return torch.cat((a * c - b * s, b * c + a * s), dim=-1)


def _heads64(x, p, cos, sin):
    """q, k, v heads [heads, T, d] of normed rows [T, H]; cos, sin [T, d/2]."""
    q, k, v = torch.split(_linear64(x, p["w"]["qkv"]), (G.q_dim, G.kv_dim, G.kv_dim), dim=-1)
    q = _rope64(_norm64(q.view(-1, NQ, D), p["q_norm"]).transpose(0, 1), cos, sin)
    k = _rope64(_norm64(k.view(-1, NKV, D), p["k_norm"]).transpose(0, 1), cos, sin)
    return q, k, v.view(-1, NKV, D).transpose(0, 1)


def _mlp64(hidden, p):
    gate, up = _linear64(_norm64(hidden, p["ln_post"]), p["w"]["gate_up"]).chunk(2, dim=-1)
    return hidden + _linear64(gate * torch.sigmoid(gate) * up, p["w"]["down"])


def _step64(hidden, p, keys, values, cos, sin):
    """One decode token [1, H] over keys, values [n_kv, rows, d]: the layer's output, the attention's part of the
    residual, and the new heads."""
    q, k, v = _heads64(_norm64(hidden, p["ln_in"]), p, cos, sin)
    keys, values = torch.cat((keys.double(), k), 1), torch.cat((values.double(), v), 1)
    scores = (q.view(NKV, NQ // NKV, D) @ keys.transpose(1, 2)) * SCALE
    attn = _linear64((torch.softmax(scores, -1) @ values).reshape(1, -1), p["w"]["o"])
    return _mlp64(hidden + attn, p), attn, q, k, v


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "token":
        s = _token_inputs(case, seed)
        cos, sin = _rope_tables(torch.tensor([case["rows"]], device=DEV))
        hidden = s.embedding[s.first].double()
        ks, vs = [], []
        for l, w in enumerate(s.layers):
            p = {"w": w, "ln_in": s.norms[l, 0], "ln_post": s.norms[l, 1], "q_norm": s.qk_norms[l, 0],
                 "k_norm": s.qk_norms[l, 1]}
            hidden, _, _, k, v = _step64(hidden, p, s.k[l, :, : case["rows"]], s.v[l, :, : case["rows"]], cos, sin)
            ks.append(k[:, 0])
            vs.append(v[:, 0])
        logits = torch.cat([_norm64(hidden, s.final_norm) @ e.double().t() for e in s.embedding.chunk(8)], 1)
        return {"token": logits.argmax(1), "hidden": hidden, "k": torch.stack(ks), "v": torch.stack(vs)}
    if kind in ("decode_layer", "vector_layer"):
        s = _step_inputs(case, seed)
        out, attn, q, k, v = _step64(s.hidden.view(1, -1).double(), vars(s), s.k[0], s.v[0], s.cos, s.sin)
        if kind == "decode_layer":
            return {"hidden": out.view(1, 1, -1), "k": k[:, 0], "v": v[:, 0]}
        return {"hidden": out.view(1, 1, -1), "attn": attn.view(-1), "q": q[None], "k": k[None], "v": v[None]}
    if kind == "layer":
        s = _rows_inputs(case, seed)
        p = vars(s)
        hidden = s.hidden[0].double()
        q, k, v = _heads64(_norm64(hidden, s.ln_in), p, s.cos[0], s.sin[0])
        out = _mlp64(hidden + _linear64(s.attn[0].double(), s.w["o"]), p)
        return {"q": q[None], "k": k[None], "v": v[None], "hidden": out[None]}
    s = _head_inputs(case, seed)
    logits = _linear64(s.hidden.double(), s.w)
    return {"logits": logits, "tokens": None if case.get("bf16_logits") else logits.argmax(1)}
