"""Performance cases of the deterministic integer transformer path.

Each case is one piece of work that a program does through ``rasterdet``: the
primitive operators on device buffers, the layer-level operators an executor
calls, whole requests through sessions, batched serving, and the committed
checkpoint trace. Inputs are synthetic: weights from the counter-hash
generators the benchmark uses (int8 with a row scale, or i16 bits that do not
factor), activations ``f32_to_act`` of seeded normals. The widths are those of
the E4B-shaped configuration (hidden 2560, 8/2 heads of 256, FF 10240,
vocabulary 262144) and of the two-layer tiny configuration.

Every result is a whole number defined bit for bit by the fixed-point
arithmetic, so every comparison is exact.
"""
from __future__ import annotations

import math
import pathlib
import sys

import numpy as np
import torch

_ROOT = pathlib.Path(__file__).resolve().parents[1]
if str(_ROOT / "raster-inference_amd") not in sys.path:
    sys.path.insert(0, str(_ROOT / "raster-inference_amd"))

import rasterdet as rd  # noqa: E402
from rasterdet import synthetic  # noqa: E402

SCALE_MAX = 256  # row scales in [1, 256], as the benchmark's E4B model
_CTX = None


def _ctx() -> "rd.Context":
    """The program's one context (device 0, one stream)."""
    global _CTX
    if _CTX is None:
        _CTX = rd.Context(0)
    return _CTX


class _Buf:
    """A torch tensor as a device buffer of the operator API."""

    def __init__(self, t: torch.Tensor):
        self.t = t
        self.ptr = t.data_ptr()


def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFFFFFF)
    return g


def _acts(g: torch.Generator, *shape, std: float = 1.0, outliers: bool = False) -> torch.Tensor:
    """Q16.16 rows: f32_to_act of normals; `outliers` scales one column in 512 by 16
    (the few large channels of a residual stream)."""
    x = torch.randn(*shape, generator=g, device="cuda") * std
    if outliers:
        x[..., ::512] *= 16.0
    return torch.clamp(torch.round(x.double() * 65536.0), -2.0**31, 2.0**31 - 1).to(torch.int32)


def _out(*shape) -> _Buf:
    return _Buf(torch.zeros(*shape, dtype=torch.int32, device="cuda"))


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------
def _projections(c: dict) -> list[tuple[int, int]]:
    """The four matrices of one layer as the layer runs them: stacked q/k/v, o, stacked gate/up, down."""
    h, q, kv, ff = c["hidden"], c["q_width"], c["kv_width"], c["ff"]
    return [(q + 2 * kv, h), (h, q), (2 * ff, h), (h, ff)]


_E4B = {"hidden": 2560, "q_width": 2048, "kv_width": 512, "ff": 10240}


def listed() -> list[dict]:
    return [
        # the smallest whole call: a short request to the two-layer tiny model, bound by launches
        {"name": "tiny_request", "kind": "request", "model": "tiny", "layers": 2, "vocab": 512, "window": 128, "ple": 0,
         "storage": "int8", "prompt": 16, "new": 16},
        # one token through a layer's projections, operator by operator (single-stream decode)
        {"name": "linear_1", "kind": "linear", "m": 1, "storage": "int8", **_E4B},
        # final norm and vocabulary projection of one decoded token
        {"name": "head", "kind": "head", "hidden": 2560, "vocab": 262144, "storage": "int8"},
        # a short prompt, or a few dozen tokens batched over requests
        {"name": "linear_37", "kind": "linear", "m": 37, "storage": "int8", **_E4B},
        # a prompt chunk over weights as the reference stores them (i16 bits that do not factor)
        {"name": "linear_512_i16", "kind": "linear", "m": 512, "storage": "i16", **_E4B},
        # a long prompt's projections
        {"name": "linear_2048", "kind": "linear", "m": 2048, "storage": "int8", **_E4B},
        # causal attention of a long prompt in a full-attention layer
        {"name": "attention_5000", "kind": "attention", "n": 5000, "heads": 8, "kv_heads": 2, "head_dim": 256,
         "window": 0},
        # an executor's prefill of one sliding and one full layer, at a ragged prompt length
        {"name": "layers_1643", "kind": "layers", "n": 1643, "window": 512, "storage": "int8"},
        # an executor's decode of one token in one sliding layer whose window is full
        {"name": "layer_decode", "kind": "layer_decode", "window": 512, "storage": "int8"},
        # a request end to end: session, 512-token prompt, greedy decode
        {"name": "request_512", "kind": "request", "model": "e4b", "layers": 4, "vocab": 32768, "window": 512, "ple": 0,
         "storage": "int8", "prompt": 512, "new": 64},
        # sixteen ragged requests prefilled and decoded together
        {"name": "serve_16", "kind": "serve", "layers": 4, "vocab": 32768, "window": 512, "storage": "int8",
         "sequences": 16, "shortest": 91, "longest": 811, "new": 48},
        # a claimer's run: a request with every checkpoint committed
        {"name": "claim", "kind": "claim", "layers": 2, "vocab": 8192, "window": 512, "storage": "int8", "prompt": 200,
         "new": 16},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    """One more case of the ranges above."""
    kind = rng.choice(["linear", "linear", "linear", "linear", "head", "attention", "attention", "layers", "layers",
                       "layer_decode", "request", "request", "serve", "claim"])
    storage = rng.choice(["int8", "int8", "i16"])
    window = _log_int(rng, 16, 1024)
    if kind == "linear":
        if rng.random() < 0.5:
            widths = dict(_E4B)
        else:
            hidden = rng.randint(300, 2560)
            widths = {"hidden": hidden, "q_width": 16 * rng.randint(16, 128), "kv_width": 16 * rng.randint(4, 32),
                      "ff": hidden * rng.randint(2, 4)}
        return {"kind": kind, "m": _log_int(rng, 1, 1800 if storage == "int8" else 900), "storage": storage, **widths}
    if kind == "head":
        return {"kind": kind, "hidden": 2560, "vocab": _log_int(rng, 2048, 262144 if storage == "int8" else 131072),
                "storage": storage}
    if kind == "attention":
        heads, kv_heads, head_dim = rng.choice([(8, 2, 256), (8, 2, 256), (16, 4, 128), (4, 1, 64)])
        return {"kind": kind, "n": _log_int(rng, 16, 4900), "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim,
                "window": rng.choice([0, window])}
    if kind == "layers":
        return {"kind": kind, "n": _log_int(rng, 16, 1600 if storage == "int8" else 800), "window": window,
                "storage": storage}
    if kind == "layer_decode":
        return {"kind": kind, "window": window, "storage": storage}
    if kind == "request":
        return {"kind": kind, "model": "e4b", "layers": rng.randint(2, 4), "vocab": _log_int(rng, 4096, 32768),
                "window": window, "ple": rng.choice([0, 0, 256]), "storage": "int8", "prompt": _log_int(rng, 8, 900),
                "new": _log_int(rng, 8, 60)}
    if kind == "serve":
        shortest = _log_int(rng, 8, 200)
        return {"kind": kind, "layers": rng.randint(2, 4), "vocab": _log_int(rng, 4096, 32768), "window": window,
                "storage": "int8", "sequences": rng.randint(2, 15), "shortest": shortest,
                "longest": shortest + _log_int(rng, 16, 600), "new": _log_int(rng, 8, 44)}
    return {"kind": kind, "layers": 2, "vocab": _log_int(rng, 2048, 8192), "window": window, "storage": "int8",
            "prompt": _log_int(rng, 8, 200), "new": _log_int(rng, 4, 16)}


# ---------------------------------------------------------------------------
# What the program holds before the call
# ---------------------------------------------------------------------------
def _values(seed: int, rows: int, cols: int, storage: str):
    if storage == "int8":
        return rd.synthetic_int8(seed, rows, cols, SCALE_MAX)
    return rd.synthetic_i16(seed, rows, cols, 4096), None


def _model(cfg: dict, seed: int, storage: str) -> "rd.Model":
    model = rd.Model(_ctx(), cfg)
    make = synthetic.synthetic_model_i16 if storage == "i16" else synthetic.synthetic_model_fast
    for name, v, s in make(cfg, seed) if storage == "i16" else make(cfg, seed, scale_max=SCALE_MAX):
        model.set_tensor(name, v, s)
    return model.finalize()


def _request_model(c: dict, seed: int) -> "rd.Model":
    if c.get("model") == "tiny":
        cfg, tensors = synthetic.tiny_model(seed=0x5EED + seed)
        model = rd.Model(_ctx(), cfg)
        for name, v, s in tensors:
            model.set_tensor(name, v, s)
        return model.finalize()
    return _model(synthetic.e4b_config(layers=c["layers"], vocab=c["vocab"], sliding_window=c["window"],
                                       ple=c.get("ple", 0)), seed, c["storage"])


def _prompts(c: dict) -> list[int]:
    """Prompt lengths of a serving batch: spread evenly from the shortest to the longest."""
    n, lo, hi = c["sequences"], c["shortest"], c["longest"]
    return [lo + (hi - lo) * i // max(n - 1, 1) for i in range(n)]


def prepare(case: dict, seed: int) -> dict:
    c, kind = dict(case), case["kind"]
    g, ids = _gen(seed), np.random.default_rng(seed)
    state = {"case": c}
    if kind == "linear":
        state["w"], state["x"], state["out"] = [], [], []
        for i, (rows, cols) in enumerate(_projections(c)):
            v, s = _values(seed * 16 + i, rows, cols, c["storage"])
            state["w"].append(_ctx().upload_matrix(v, s))
            state["x"].append(_Buf(_acts(g, c["m"], cols)))
            state["out"].append(_out(c["m"], rows))
    elif kind == "head":
        state["model"] = _model(synthetic.e4b_config(layers=1, vocab=c["vocab"]), seed, c["storage"])
        state["ops"] = rd.LayerOps(state["model"])
        state["x"], state["out"] = _Buf(_acts(g, c["hidden"], std=4.0, outliers=True)), _out(c["vocab"])
    elif kind == "attention":
        n, hd = c["n"], c["head_dim"]
        # head-normalised rows: unit RMS
        state["q"] = _Buf(_acts(g, n, c["heads"] * hd))
        state["k"] = _Buf(_acts(g, n, c["kv_heads"] * hd))
        state["v"] = _Buf(_acts(g, n, c["kv_heads"] * hd))
        state["out"] = _out(n, c["heads"] * hd)
    elif kind in ("layers", "layer_decode"):
        cfg = synthetic.e4b_config(layers=2, vocab=512, sliding_window=c["window"])
        model = state["model"] = _model(cfg, seed, c["storage"])
        ops = state["ops"] = rd.LayerOps(model)
        rows = c["n"] if kind == "layers" else c["window"]
        state["x"] = _Buf(_acts(g, rows, 2560, std=4.0, outliers=True))
        state["caches"] = [rd.KvCache(model, l, max(rows, c["window"])) for l in range(2)]
        state["out"] = [_out(rows, 2560) for _ in range(2)]
        if kind == "layer_decode":
            ops.layer_prefill(0, state["x"], rows, None, None, state["caches"][0], state["out"][0])
            state["x"], state["out"] = _Buf(_acts(g, 2560, std=4.0, outliers=True)), _out(2560)
            state["position"] = rows
    elif kind == "request":
        state["model"] = _request_model(c, seed)
        state["prompt"] = ids.integers(0, c["vocab"], size=c["prompt"]).tolist()
    elif kind == "serve":
        state["model"] = _request_model(c, seed)
        state["prompts"] = [ids.integers(0, c["vocab"], size=n).tolist() for n in _prompts(c)]
    elif kind == "claim":
        state["model"] = _request_model(c, seed)
        state["prompt"] = ids.integers(0, c["vocab"], size=c["prompt"]).tolist()
    else:
        raise ValueError(kind)
    return state


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(state: dict):
    c, ctx = state["case"], _ctx()
    kind = c["kind"]
    if kind == "linear":
        for w, x, out in zip(state["w"], state["x"], state["out"]):
            if c["m"] == 1:
                ctx.det_linear_into(w, x, out)
            else:
                ctx.det_linear_slab(w, c["m"], x, out)
        return [o.t for o in state["out"]]
    if kind == "head":
        state["ops"].hidden_to_logits(state["x"], state["out"])
        return state["out"].t
    if kind == "attention":
        ctx.attention(state["q"], state["k"], state["v"], c["n"], c["n"], c["heads"], c["kv_heads"], c["head_dim"],
                      c["window"], state["out"])
        return state["out"].t
    if kind == "layers":
        ops, x = state["ops"], state["x"]
        for l in range(2):
            ops.layer_prefill(l, x, c["n"], None, None, state["caches"][l], state["out"][l])
            x = state["out"][l]
        return [o.t for o in state["out"]]
    if kind == "layer_decode":
        state["ops"].layer_decode(0, state["x"], None, state["caches"][0], None, state["position"], state["out"])
        state["position"] += 1
        return state["out"].t
    if kind == "request":
        sess = state["model"].session(c["prompt"] + c["new"])
        tokens = [sess.prefill(state["prompt"], rd.DET_COMMIT_NONE).next_token]
        while len(tokens) < c["new"]:
            tokens.append(sess.decode(tokens[-1], rd.DET_COMMIT_NONE).next_token)
        return {"tokens": np.asarray(tokens, dtype=np.int64), "logits": sess.logits(c["vocab"])}
    if kind == "serve":
        sessions = [state["model"].session(len(p) + c["new"]) for p in state["prompts"]]
        tokens = [[s.prefill(p, rd.DET_COMMIT_NONE).next_token for s, p in zip(sessions, state["prompts"])]]
        while len(tokens) < c["new"]:
            tokens.append([r.next_token for r in rd.decode_batch(sessions, tokens[-1], rd.DET_COMMIT_NONE)])
        return {"tokens": np.asarray(tokens, dtype=np.int64),
                "logits": np.stack([s.logits(c["vocab"]) for s in sessions])}
    text, _ = state["model"].trace("a prompt", state["prompt"], max_new_tokens=c["new"],
                                   detokenize=lambda ids: " ".join(map(str, ids)))
    return np.frombuffer(text, dtype=np.uint8)


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _pairs(n: int, window: int) -> int:
    """(query, key) pairs of causal attention over n rows."""
    if window == 0 or window >= n:
        return n * (n + 1) // 2
    return window * (window + 1) // 2 + (n - window) * window


def _layer_work(c: dict, n: int, pairs: int, keys: int) -> tuple[float, float]:
    """Bytes and operations of one E4B-width layer over n tokens that attend to `pairs` keys, `keys` of them distinct."""
    width = 1 if c["storage"] == "int8" else 2
    weights = sum(r * k for r, k in _projections(_E4B))
    ple = c.get("ple", 0)
    weights += 3 * ple * 2560  # gate, projection and this layer's rows of the model projection
    return (weights * width + 4.0 * n * 2560 * 2 + 4.0 * keys * 1024,
            2.0 * n * weights + 4.0 * 256 * 8 * pairs)


def _stack_work(c: dict, spans: list[tuple[int, int]]) -> tuple[float, float]:
    """All layers (sliding and full in turn) over tokens [start, end) of each span in one pass over the weights."""
    total_b = total_f = 0.0
    for l in range(c["layers"]):
        w = c["window"] if l % 2 == 0 else 0
        n = sum(e - s for s, e in spans)
        pairs = sum(_pairs(e, w) - _pairs(s, w) for s, e in spans)
        keys = sum(min(e, w + e - s) if w else e for s, e in spans)
        b, f = _layer_work(c, n, pairs, keys)
        total_b, total_f = total_b + b, total_f + f
    return total_b, total_f


def _head_work(c: dict, m: int, hidden: int = 2560) -> tuple[float, float]:
    width = 1 if c["storage"] == "int8" else 2
    return c["vocab"] * hidden * width + 4.0 * m * (hidden + c["vocab"]), 2.0 * m * c["vocab"] * hidden


def _tiny_work(c: dict) -> tuple[float, float]:
    weights = 2 * (96 * 64 + 64 * 64 + 256 * 64 + 64 * 128) + 512 * 64
    tokens = c["prompt"] + c["new"] - 1
    return float(weights * c["new"] + 4 * tokens * 2 * 32), 2.0 * weights * tokens


def work(case: dict) -> dict:
    c, kind = case, case["kind"]
    b = f = 0.0
    if kind == "linear":
        width = 1 if c["storage"] == "int8" else 2
        for rows, cols in _projections(c):
            b += rows * cols * width + 4 * rows + 4 * c["m"] * (rows + cols)
            f += 2.0 * c["m"] * rows * cols
    elif kind == "head":
        b, f = _head_work(c, 1)
    elif kind == "attention":
        b = 4.0 * c["n"] * c["head_dim"] * 2 * (c["heads"] + c["kv_heads"])
        f = 4.0 * c["head_dim"] * c["heads"] * _pairs(c["n"], c["window"])
    elif kind == "layers":
        b, f = _stack_work({**c, "layers": 2}, [(0, c["n"])])
    elif kind == "layer_decode":
        b, f = _layer_work(c, 1, c["window"], c["window"])
    elif c.get("model") == "tiny":
        b, f = _tiny_work(c)
    else:
        prompts = _prompts(c) if kind == "serve" else [c["prompt"]]
        steps = c["new"] - (0 if kind == "claim" else 1)
        parts = [_stack_work(c, [(0, n)]) for n in prompts] + [_head_work(c, 1) for _ in prompts]
        for t in range(steps):
            parts += [_stack_work(c, [(n + t, n + t + 1) for n in prompts]), _head_work(c, len(prompts))]
        b, f = (sum(p[i] for p in parts) for i in range(2))
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case: dict):
    return "exact"


def exact(case: dict, seed: int):
    """The linear operators in 64 bits: the activation's high and low halves times the integer weights in float64
    (every partial sum below 2^53), then the rounding to Q16.16. None for the others: their results are whole
    numbers of a fixed-point recipe (integer softmax, norms and rotations) that plain real arithmetic only
    approximates, and they are compared bit for bit."""
    c = case
    if c["kind"] != "linear":
        return None
    g, outs = _gen(seed), []
    for i, (rows, cols) in enumerate(_projections(c)):
        v, s = _values(seed * 16 + i, rows, cols, c["storage"])
        x = _acts(g, c["m"], cols).to(torch.int64)
        w = torch.from_numpy(v).cuda().double()
        hi, lo = x >> 16, x & 0xFFFF
        acc = (hi.double() @ w.T).to(torch.int64) * 65536 + (lo.double() @ w.T).to(torch.int64)
        if s is not None:
            acc = acc * torch.from_numpy(s).cuda().to(torch.int64)
        half = acc >> 16
        rem = acc & 0xFFFF
        up = (rem > 0x8000) | ((rem == 0x8000) & ((half & 1) == 1))
        outs.append(torch.clamp(half + up.to(torch.int64), -2**31, 2**31 - 1).to(torch.int32))
    return outs
