"""Timed cases of the int4 decode path: what a program using this package
calls, with sizes from its own configurations and tests.

Families (key "kind"):
  gemv     one packed-int4 projection of one token (quant_int4_gemv)
  gemm     the same projection for m tokens (quant_int4_gemm): concurrent
           sequences, or a prompt's tokens
  gqa      grouped-query attention of one token over an fp16 cache (gqa_decode)
  sample   one token drawn from the logits by the runner's policy (sample_token)
  prefill  a prompt through the whole model to its next-token logits
  decode   greedy decoding of one sequence (decode_greedy)
  batch    one decode step of several independent sequences (forward_tokens)
The first four are single operators, the last three whole-model calls over
random-init weights of the Qwen3-4B shape (or a smaller one in drawn cases).
"""
from __future__ import annotations

import math

import numpy as np
import torch

from harsh4b_amd.config import QWEN3_4B
from harsh4b_amd.lightspark import (LiteSparkProjection, gqa_decode, quant_int4_gemm, quant_int4_gemv,
                                    sample_token)
from harsh4b_amd.synthetic import random_model, random_packed

# A smaller model of the same architecture, for drawn cases only.
SMALL = dict(QWEN3_4B, hidden_size=1024, intermediate_size=3072, num_attention_heads=16, num_hidden_layers=8,
             vocab_size=32000, max_position_embeddings=8192)


def _config(case: dict) -> dict:
    return SMALL if case["model"] == "small" else QWEN3_4B


# --------------------------------------------------------------------------- the cases
def listed() -> list[dict]:
    return [
        # one token's k (or v) projection: the smallest call of the path
        dict(name="gemv_kv", kind="gemv", rows=1024, width=2560),
        # one token's gate projection: the package's headline GEMV
        dict(name="gemv_gate", kind="gemv", rows=9728, width=2560),
        # gate_up of 32 sequences decoding together
        dict(name="gemm_m32_gate_up", kind="gemm", m=32, rows=19456, width=2560),
        # down projection of a prompt of odd length
        dict(name="gemm_m501_down", kind="gemm", m=501, rows=2560, width=9728),
        # attention early in a chat
        dict(name="gqa_300", kind="gqa", context=300, kv_heads=8, groups=4, head_dim=128),
        # attention at the long-context benchmark's length
        dict(name="gqa_4096", kind="gqa", context=4096, kv_heads=8, groups=4, head_dim=128),
        # attention over a long document
        dict(name="gqa_32767", kind="gqa", context=32767, kv_heads=8, groups=4, head_dim=128),
        # the runner's default policy over the full vocabulary
        dict(name="sample_k40", kind="sample", n=151936, top_k=40, history=100, top_p=0.9, temperature=0.7,
             penalty=1.08),
        # a chat message to its first logits
        dict(name="prefill_64", kind="prefill", model="4b", tokens=64, start=0),
        # a document to its first logits
        dict(name="prefill_2000", kind="prefill", model="4b", tokens=2000, start=0),
        # a few tokens of a reply, 600 tokens into a chat
        dict(name="decode_600", kind="decode", model="4b", context=600, steps=4),
        # one step of 16 chats of different lengths around 256 tokens
        dict(name="batch_16", kind="batch", model="4b", sequences=16, context=256),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng) -> dict:
    kind = rng.choice(["gemv", "gemm", "gemm", "gqa", "gqa", "sample", "prefill", "prefill", "decode", "batch"])
    if kind == "gemv":
        return dict(kind=kind, rows=_log_int(rng, 64, 151936), width=32 * _log_int(rng, 8, 320))
    if kind == "gemm":
        rows, width = rng.choice([(6144, 2560), (2560, 4096), (19456, 2560), (2560, 9728),
                                  (_log_int(rng, 100, 20000), 32 * _log_int(rng, 4, 320))])
        return dict(kind=kind, m=_log_int(rng, 2, 2000), rows=rows, width=width)
    if kind == "gqa":
        kv, g, d = rng.choice([(8, 4, 128), (8, 4, 128), (8, 2, 128), (4, 8, 128), (2, 3, 64), (8, 5, 64)])
        return dict(kind=kind, context=_log_int(rng, 1, 40960), kv_heads=kv, groups=g, head_dim=d)
    if kind == "sample":
        return dict(kind=kind, n=rng.choice([151936, _log_int(rng, 2048, 151936)]), top_k=_log_int(rng, 1, 2048),
                    history=_log_int(rng, 1, 2000), top_p=rng.choice([0.8, 0.9, 0.95, 1.0]),
                    temperature=rng.choice([0.3, 0.7, 1.0]), penalty=rng.choice([1.0, 1.08, 1.15]))
    model = rng.choice(["4b", "4b", "small"])
    if kind == "prefill":
        tokens = _log_int(rng, 2, 2000)
        return dict(kind=kind, model=model, tokens=tokens,
                    start=0 if rng.random() < 0.5 else _log_int(rng, 1, 2000 - tokens) if tokens < 2000 else 0)
    if kind == "decode":
        return dict(kind=kind, model=model, context=_log_int(rng, 1, 6000), steps=4)
    return dict(kind=kind, model=model, sequences=rng.randint(2, 31), context=_log_int(rng, 8, 1500))


# --------------------------------------------------------------------------- inputs
def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(shape, gen, dtype=torch.float32) -> torch.Tensor:
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32).to(dtype)


def _projection(rows: int, width: int, gen) -> LiteSparkProjection:
    # integers uniform in [-7, 7], row scales U(0.005, 0.02), as the benchmark configurations state
    scales = torch.rand(rows, generator=gen, device="cuda") * 0.015 + 0.005
    return LiteSparkProjection(random_packed(rows, width, gen, torch.device("cuda")), scales)


def _fill_cache(state, positions: int, gen) -> None:
    """A history of `positions` tokens: N(0,1) keys and values, as the long-context configuration states."""
    for layer in range(state.keys.shape[0]):
        state.keys[layer, :positions] = _normal(state.keys[layer, :positions].shape, gen, torch.float16)
        state.values[layer, :positions] = _normal(state.values[layer, :positions].shape, gen, torch.float16)


def _tokens(count: int, vocab: int, seed: int) -> list[int]:
    return np.random.default_rng(seed).integers(0, vocab, count).tolist()


def _contexts(case: dict) -> list[int]:
    """Ragged histories around case["context"]: 3/4 to 5/4 of it."""
    c = case["context"]
    return np.random.default_rng(c).integers(max(1, 3 * c // 4), 5 * c // 4 + 2, case["sequences"]).tolist()


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    gen = _gen(seed)
    s = {"case": case, "kind": kind}
    if kind in ("gemv", "gemm"):
        s["projection"] = _projection(case["rows"], case["width"], gen)
        if kind == "gemv":
            s["x"] = _normal(case["width"], gen)
            s["out"] = torch.empty(case["rows"], device="cuda")
        else:
            s["x"] = _normal((case["m"], case["width"]), gen)
            s["out"] = torch.empty((case["m"], case["rows"]), device="cuda")
    elif kind == "gqa":
        heads, d = case["kv_heads"] * case["groups"], case["head_dim"]
        s["query"] = _normal((heads, d), gen)
        s["keys"] = _normal((case["context"], case["kv_heads"], d), gen, torch.float16)
        s["values"] = _normal((case["context"], case["kv_heads"], d), gen, torch.float16)
        s["out"] = torch.empty((heads, d), device="cuda")
    elif kind == "sample":
        s["logits"] = 3.0 * _normal(case["n"], gen)
        s["generated"] = _tokens(case["history"], case["n"], seed)
        s["u"] = float(np.random.default_rng(seed + 2).random())
    else:
        config = _config(case)
        model = random_model(config, seed)
        vocab = config["vocab_size"]
        s["model"] = model
        if kind == "batch":
            s["contexts"] = _contexts(case)
            s["states"] = [model.new_state(c + 8) for c in s["contexts"]]
            for state, c in zip(s["states"], s["contexts"]):
                _fill_cache(state, c, gen)
            s["positions"] = [st.device_position for st in s["states"]]
            s["rewound"] = [torch.tensor([c], dtype=torch.int32, device="cuda") for c in s["contexts"]]
            s["tokens"] = _tokens(case["sequences"], vocab, seed)
        else:
            start = case["start"] if kind == "prefill" else case["context"]
            count = case["tokens"] if kind == "prefill" else case["steps"]
            s["start"] = start
            s["state"] = model.new_state(start + count)
            _fill_cache(s["state"], start, gen)
            s["tokens"] = _tokens(count if kind == "prefill" else 1, vocab, seed)
        # the histories were written on torch's stream; the steps run on the model's
        model.stream.wait_stream(torch.cuda.current_stream())
    return s


# --------------------------------------------------------------------------- one pass
def run(s: dict):
    kind = s["kind"]
    case = s["case"]
    if kind == "gemv":
        return quant_int4_gemv(s["x"], s["projection"], out=s["out"])
    if kind == "gemm":
        return quant_int4_gemm(s["x"], s["projection"], out=s["out"])
    if kind == "gqa":
        return gqa_decode(s["query"], s["keys"], s["values"], s["out"], case["context"], case["kv_heads"],
                          case["groups"], case["head_dim"])
    if kind == "sample":
        return sample_token(s["logits"], s["generated"], case["penalty"], case["temperature"], case["top_k"],
                            case["top_p"], s["u"])
    model = s["model"]
    if kind == "batch":
        # back to where the histories end (the reply is drawn again)
        with torch.cuda.stream(model.stream):
            torch._foreach_copy_(s["positions"], s["rewound"])
        for state, c in zip(s["states"], s["contexts"]):
            state.position = c
        logits = model.forward_tokens(s["tokens"], s["states"])
        # (stacked, as the next step's batched sampling takes them)
        return [torch.stack(logits), [st.keys for st in s["states"]], [st.values for st in s["states"]]]
    state = s["state"]
    state.position = s["start"]
    if kind == "prefill":
        logits = model.prefill(s["tokens"], state)
        return [logits, *_first_and_rest(state.keys), *_first_and_rest(state.values)]
    with torch.cuda.stream(state.stream):
        state.device_position.fill_(s["start"])
        state.token.fill_(s["tokens"][0])
    model.decode_greedy(state, case["steps"])
    return [state.logits, state.token, state.keys, state.values]


EXACT_LAYERS = 4


def _first_and_rest(cache: torch.Tensor):
    """The whole cache in two parts: the layers that exact() computes, and the others.  Past a few layers of
    random weights a 64-bit run has no comparable value: one int8 rounding that falls the other way moves
    every later layer by a few percent."""
    return cache[:EXACT_LAYERS], cache[EXACT_LAYERS:]


# --------------------------------------------------------------------------- what a pass cannot do without
def _model_sizes(c: dict):
    h, i, d = c["hidden_size"], c["intermediate_size"], c["head_dim"]
    q, kv = c["num_attention_heads"] * d, c["num_key_value_heads"] * d
    per_layer = (q + 2 * kv) * h + h * q + 2 * i * h + h * i            # weights of one layer
    rows = q + 2 * kv + h + 2 * i + h
    layers = c["num_hidden_layers"]
    body = layers * (per_layer // 2 + 4 * rows + 4 * (2 * h + 2 * d))   # bytes
    head = c["vocab_size"] * (h // 2 + 4)
    return h, q, kv, layers, per_layer, body, head


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        m, rows, width = case.get("m", 1), case["rows"], case["width"]
        return {"bytes": rows * width // 2 + 4 * rows + 4 * m * (width + rows), "flops": 2 * m * rows * width}
    if kind == "gqa":
        kv, heads, d = case["kv_heads"], case["kv_heads"] * case["groups"], case["head_dim"]
        return {"bytes": case["context"] * kv * d * 4 + heads * d * 8, "flops": 4 * case["context"] * heads * d}
    if kind == "sample":
        return {"bytes": 4 * case["n"] + 4 * case["history"] + 8 * case["top_k"], "flops": 2 * case["n"]}
    h, q, kv, layers, per_layer, body, head = _model_sizes(_config(case))
    vocab = _config(case)["vocab_size"]
    if kind == "prefill":
        t, start = case["tokens"], case["start"]
        pairs = t * start + t * (t + 1) // 2                            # (query, key) pairs of a head
        return {"bytes": body + head + layers * kv * 4 * (start + t) + t * h // 2 + 4 * vocab,
                "flops": 2 * t * layers * per_layer + 2 * vocab * h + 4 * layers * pairs * q}
    if kind == "decode":
        n, c = case["steps"], case["context"]
        return {"bytes": n * (body + head + layers * kv * 4 * (c + 1) + 4 * vocab),
                "flops": n * (2 * layers * per_layer + 2 * vocab * h + 4 * layers * (c + 1) * q)}
    m, c = case["sequences"], case["context"]
    return {"bytes": body + head + m * (layers * kv * 4 * (c + 1) + 4 * vocab),
            "flops": m * (2 * layers * per_layer + 2 * vocab * h + 4 * layers * (c + 1) * q)}


def tolerance(case: dict):
    # the package fixes the order of every operation (its CPU oracle restates it): the same bits every time
    return "exact"


# --------------------------------------------------------------------------- 64-bit results
def _unpack(w: torch.Tensor) -> torch.Tensor:
    lo = ((w & 15).to(torch.int8) ^ 8) - 8
    hi = ((w >> 4).to(torch.int8) ^ 8) - 8
    return torch.stack((lo, hi), dim=-1).reshape(w.shape[0], -1).double()


def _quantize(x: torch.Tensor):
    """int8 activations and scale per row, as the path defines them: q = rint(127 x / max|x|)."""
    amax = x.abs().amax(dim=-1, keepdim=True).clamp_min(1e-5)
    return torch.round(x * (127.0 / amax)).clamp(-127, 127), amax / 127.0


def _linear(x: torch.Tensor, p: LiteSparkProjection) -> torch.Tensor:
    q, scale = _quantize(x)
    out = torch.empty((x.shape[0], p.weights.shape[0]), dtype=torch.float64, device=x.device)
    for r in range(0, out.shape[1], 16384):
        out[:, r:r + 16384] = q @ _unpack(p.weights[r:r + 16384]).t().contiguous()
    return out * scale * p.scales.double()


def _rms(x: torch.Tensor, gamma: torch.Tensor, eps: float) -> torch.Tensor:
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps) * gamma.double()


def _rope(config: dict, positions: torch.Tensor):
    """The path's float32 rotation tables at the given positions."""
    d = config["head_dim"]
    inv = np.float32(1.0) / np.float32(config["rope_theta"]) ** (np.arange(0, d, 2, dtype=np.float32) / np.float32(d))
    angles = positions.cpu().numpy().astype(np.float32)[:, None] * inv[None, :]
    cos, sin = np.cos(angles).astype(np.float32), np.sin(angles).astype(np.float32)
    return torch.from_numpy(cos).to(positions.device).double(), torch.from_numpy(sin).to(positions.device).double()


def _attend(q, keys, values, first: int, kv_heads: int):
    """q [t, heads, d]; query i sees the cache's first + i + 1 positions."""
    t, heads, d = q.shape
    n = first + t
    g = heads // kv_heads
    out = torch.empty_like(q)
    seen = torch.arange(n, device=q.device)[None, :] <= first + torch.arange(t, device=q.device)[:, None]
    for kv in range(kv_heads):
        k, v = keys[:n, kv].double(), values[:n, kv].double()
        for h in range(kv * g, kv * g + g):
            s = (q[:, h] @ k.t().contiguous()) / math.sqrt(d)
            p = torch.softmax(s.masked_fill(~seen, -math.inf), dim=-1)
            out[:, h] = p @ v
    return out


def _forward(model, config: dict, ids: list[int], keys, values, first: int) -> None:
    """The K/V rows of the first layers in float64 for a run of tokens at positions first.., written into
    the caches."""
    dev = model.embedding.device
    eps, d = config["rms_norm_eps"], config["head_dim"]
    heads, kvh = config["num_attention_heads"], config["num_key_value_heads"]
    inter = config["intermediate_size"]
    idx = torch.tensor(ids, device=dev)
    x = _unpack(model.embedding[idx]) * model.embedding_scales[idx].double()[:, None]
    n = len(ids)
    cos, sin = (a[:, None, :] for a in _rope(config, first + torch.arange(n, device=dev)))

    def rotate(a):
        lo, hi = a[..., :d // 2], a[..., d // 2:]
        return torch.cat((lo * cos - hi * sin, hi * cos + lo * sin), dim=-1)

    for l, layer in enumerate(model.layers[:EXACT_LAYERS]):
        qkv = _linear(_rms(x, layer.input_norm, eps), layer.qkv).view(n, heads + 2 * kvh, d)
        q = rotate(_rms(qkv[:, :heads], layer.q_norm, eps))
        k = rotate(_rms(qkv[:, heads:heads + kvh], layer.k_norm, eps))
        keys[l, first:first + n] = k.float().half()
        values[l, first:first + n] = qkv[:, heads + kvh:].float().half()
        att = _attend(q, keys[l], values[l], first, kvh)
        x = x + _linear(att.reshape(n, -1), layer.o)
        gu = _linear(_rms(x, layer.post_norm, eps), layer.gate_up)
        g, u = gu[:, :inter], gu[:, inter:]
        x = x + _linear(g / (1.0 + torch.exp(-g)) * u, layer.down)


def _exact_sample(case: dict, s: dict):
    v = s["logits"].cpu().numpy().astype(np.float64)
    for i in set(s["generated"]):
        v[i] = v[i] / np.float32(case["penalty"]) if v[i] > 0 else v[i] * np.float32(case["penalty"])
    v = v / np.float32(case["temperature"])
    ids = np.argsort(-v, kind="stable")[:case["top_k"]]
    p = np.exp(v[ids] - v[ids[0]])
    p /= p.sum()
    if case["top_p"] < 1.0:
        p[np.cumsum(p) - p >= np.float32(case["top_p"])] = 0.0
        p /= p.sum()
    cdf = np.cumsum(p)
    token = int(ids[min(len(ids) - 1, int(np.searchsorted(cdf / cdf[-1], s["u"], side="right")))])
    return token, ids.astype(np.int32), p


def exact(case: dict, seed: int):
    kind = case["kind"]
    s = prepare(case, seed)
    if kind == "gemv":
        return _linear(s["x"].double()[None, :], s["projection"])[0]
    if kind == "gemm":
        return _linear(s["x"].double(), s["projection"])
    if kind == "gqa":
        q = s["query"].double()[None]
        return _attend(q, s["keys"], s["values"], case["context"] - 1, case["kv_heads"])[0]
    if kind == "sample":
        return _exact_sample(case, s)
    if kind in ("decode", "batch"):
        return None            # every output but the first rows of a cache follows from all the layers
    state = s["state"]
    _forward(s["model"], _config(case), s["tokens"], state.keys, state.values, s["start"])
    return [None, state.keys[:EXACT_LAYERS], None, state.values[:EXACT_LAYERS], None]
