"""GPU parity of the layer-level operators (det_layer_prefill,
det_layer_decode, det_decode_ple_input, det_hidden_to_logits, KV handles).

The routines call these per layer (prefill_range/native/deterministic_tiles.rs
:69-199, decode_layer_range/native/tiles.rs:133-197). Here a host loop
restates the det_goldens capture protocol (src/runtime/det_goldens.rs:90-236)
on top of them, every call going through the C ABI, and must reproduce the
reference's goldens (tests/golden/det_commitment_goldens.det.json, both PLE
fixtures, one with a KV-sharing donor layer) and the oracle's capture of an
E4B-shaped model.
"""
import hashlib
import struct

import numpy as np
import pytest

import fixtures
import oracle_lib

pytestmark = pytest.mark.gpu
rd = pytest.importorskip("rasterdet")
from rasterdet import synthetic  # noqa: E402


@pytest.fixture(scope="module")
def ctx():
    c = rd.Context(0)
    yield c
    c.close()


def act_commitment(rows: np.ndarray) -> str:
    # build_det_activation_commitment (transformer_kernels.rs:1395-1430)
    rows = np.atleast_2d(rows).astype("<i4")
    h = hashlib.sha256(b"raster-det-num-act-v1" + struct.pack("<Q", rows.shape[0]))
    for r in rows:
        h.update(struct.pack("<Q", r.size) + r.tobytes())
    return h.hexdigest()


def vector_commitment(v: np.ndarray) -> str:
    # build_det_vector_commitment (transformer_kernels.rs:1432-1438)
    v = np.asarray(v).astype("<i4")
    return hashlib.sha256(b"raster-det-num-act-vector-v1" + struct.pack("<Q", v.size) + v.tobytes()).hexdigest()


def donor_of(tc: dict, layer: int):
    # kv_shared_layer_index (gemma/io.rs:165-190): the last layer before the
    # shared block with the same attention type
    shared = tc.get("num_kv_shared_layers") or 0
    first = tc["num_hidden_layers"] - shared
    if not shared or layer < first:
        return None
    return max(i for i in range(first) if tc["layer_types"][i] == tc["layer_types"][layer])


class LayerLoop:
    """det_goldens capture through the layer-level entry points."""

    def __init__(self, ctx, model, config, max_tokens):
        self.ctx, self.model, self.ops = ctx, model, rd.LayerOps(model)
        self.tc = config.get("text_config", config)
        self.H, self.L = self.tc["hidden_size"], self.tc["num_hidden_layers"]
        self.ple = self.tc.get("hidden_size_per_layer_input") or 0
        self.max_tokens = max_tokens

    def buf(self, rows, width):
        return self.ctx.empty((max(rows, 1), max(width, 1)))

    def ple_rows(self, ids, emb, n):
        out = []
        for layer in range(self.L):
            b = self.buf(n, self.ple)
            made = (self.ops.prefill_ple_inputs(layer, ids, emb, b) if n > 1
                    else self.ops.decode_ple_input(ids[0], emb, layer, b))
            out.append(b if made else None)
        return out

    def logits(self, hidden_row):
        out = self.ctx.empty(self.tc["vocab_size"])
        self.ops.hidden_to_logits(hidden_row, out)
        return out.numpy()

    def prefill(self, ids):
        n, H = len(ids), self.H
        emb = self.buf(n, H)
        self.ops.embed(ids, emb)
        ple = self.ple_rows(ids, emb, n)
        caches, x = [], self.buf(n, H)
        self.ctx.check(self.ctx.lib.det_memcpy_d2d(self.ctx.handle, rd.C.c_void_p(x.ptr), rd.C.c_void_p(emb.ptr),
                                                   n * H * 4))
        for layer in range(self.L):
            d = donor_of(self.tc, layer)
            cache = rd.KvCache(self.model, layer, self.max_tokens)
            self.ops.layer_prefill(layer, x, n, ple[layer], caches[d] if d is not None else None,
                                   None if d is not None else cache, x)
            caches.append(cache)
        hidden = x.numpy().reshape(n, H)
        last = self.ctx.to_device(np.ascontiguousarray(hidden[-1]))
        lg = self.logits(last)
        return caches, lg, {"embedding": act_commitment(emb.numpy().reshape(n, H)),
                            "final_hidden": act_commitment(hidden), "logits": vector_commitment(lg),
                            "kv": rd.kv_commitment(caches)}

    def decode(self, caches, token, position, per_layer=None):
        """One step on `caches` in place; per_layer collects (layer output,
        effective-cache commitment) with the untouched `original` caches."""
        emb = self.buf(1, self.H)
        self.ops.embed([token], emb)
        ple = self.ple_rows([token], emb, 1)
        x = self.ctx.to_device(emb.numpy().reshape(-1))
        for layer in range(self.L):
            d = donor_of(self.tc, layer)
            self.ops.layer_decode(layer, x, ple[layer], None if d is not None else caches[layer],
                                  caches[d] if d is not None else None, position, x)
            if per_layer is not None:
                original = per_layer["original"]
                eff = caches[:layer + 1] + original[layer + 1:]
                per_layer["layers"].append({"layer_output": act_commitment(x.numpy()),
                                            "kv": rd.kv_commitment(eff)})
        return x.numpy()

    def capture(self, ids, steps):
        caches, lg, pre = self.prefill(ids)
        out = {"prefill": pre}
        tok = int(np.argmax(lg))
        first = {"original": caches, "layers": []}
        copies = [c.clone() for c in caches]
        self.decode(copies, tok, len(ids), first)
        out["first_step_layers"] = first["layers"]
        out["decode_steps"], gen = [], []
        for i in range(steps):
            tok = int(np.argmax(lg))
            gen.append(tok)
            act = self.decode(caches, tok, len(ids) + i)
            lg = self.logits(self.ctx.to_device(act))
            out["decode_steps"].append({"token": tok, "activation": act_commitment(act),
                                        "logits": vector_commitment(lg), "kv": rd.kv_commitment(caches)})
        text = "[" + ",".join(map(str, gen)) + "]"
        out["end_to_end"] = {"generated_token_ids": gen,
                             "generated_token_ids_sha256": hashlib.sha256(text.encode()).hexdigest()}
        return out


@pytest.mark.parametrize("name", ["donor_ple", "no_donor_ple"])
def test_layer_loop_reproduces_reference_goldens(ctx, name):
    cfg, wgt, prompt, _ = fixtures.golden_fixture(name)
    steps = 16
    model = rd.Model(ctx, cfg).load_detwgt(wgt).finalize()
    got = LayerLoop(ctx, model, cfg, len(prompt) + steps + 1).capture(prompt, steps)
    exp = fixtures.golden_expected(name)
    assert got["prefill"] == exp["prefill"]
    assert got["first_step_layers"] == exp["first_step_layers"]
    assert got["decode_steps"] == exp["decode_steps"][:steps]


def test_layer_loop_e4b_shaped_matches_oracle(ctx):
    # int8 GEMM prefill, sliding ring wrapped (window 8 < 21 tokens)
    cfg = synthetic.e4b_config(layers=2, vocab=4096, sliding_window=8)
    om, gm = fixtures.load_both(cfg, synthetic.synthetic_model_fast(cfg, seed=7, scale_max=256), ctx,
                                threads=oracle_lib.cpu_count())
    prompt = list(range(3, 3 + 21))
    exp = om.capture(prompt, 5)
    got = LayerLoop(ctx, gm, cfg, len(prompt) + 6).capture(prompt, 5)
    assert got["prefill"] == exp["prefill"]
    assert got["first_step_layers"] == exp["first_step_layers"]
    assert got["decode_steps"] == exp["decode_steps"]
    assert got["end_to_end"] == exp["end_to_end"]


def test_kv_handles_read_logical_rows_and_reject_misuse(ctx):
    cfg = synthetic.e4b_config(layers=2, vocab=512, sliding_window=4)
    cfg["text_config"].update({"hidden_size": 128, "intermediate_size": 256, "head_dim": 32,
                               "num_attention_heads": 4, "num_key_value_heads": 2})
    gm = rd.Model(ctx, cfg)
    for name, v, s in fixtures.custom_model(cfg, seed=5):
        gm.set_tensor(name, v, s)
    gm.finalize()
    loop = LayerLoop(ctx, gm, cfg, 16)
    caches, _, _ = loop.prefill([1, 2, 3, 4, 5, 6])
    n0, heads, hd, has = caches[0].info()
    assert (n0, heads, hd, has) == (4, 2, 32, True)  # sliding window 4 keeps the last 4 rows
    assert caches[1].info()[0] == 6
    k0, v0 = caches[0].read_logical()
    k1, _ = caches[1].read_logical()
    assert k0.shape == (2, 4, 32) and k1.shape == (2, 6, 32)
    # one decode step appends one row; the ring drops its oldest
    loop.decode(caches, 7, 6)
    k0b, v0b = caches[0].read_logical()
    assert caches[0].info()[0] == 4
    assert np.array_equal(k0b[:, :3], k0[:, 1:]) and np.array_equal(v0b[:, :3], v0[:, 1:])
    k1b, _ = caches[1].read_logical()
    assert np.array_equal(k1b[:, :6], k1)
    empty = rd.KvCache(gm, 0, 8)
    assert empty.info()[3] is False
    assert rd.kv_commitment([empty, caches[1]]) is None  # a cache without det data
    x = ctx.empty((1, 128))
    with pytest.raises(rd.DetError):  # a layer-1 handle given to layer 0
        loop.ops.layer_decode(0, x, None, caches[1], None, 7, x)
    with pytest.raises(rd.DetError):  # neither a cache nor a donor
        loop.ops.layer_decode(0, x, None, None, None, 7, x)
    with pytest.raises(rd.DetError):
        rd.KvCache(gm, 2, 8)  # no such layer


def test_kv_handle_smaller_than_window_fails_closed(ctx):
    # a sliding-window cache created for fewer tokens than its window holds
    # max_tokens rows: a prefill or append past max_tokens must fail (the
    # reference's cache would still hold the last `window` rows) instead of
    # overwriting rows the window reads; a linear cache fails the same way,
    # and a ring sized at its window keeps taking tokens
    cfg = synthetic.e4b_config(layers=2, vocab=512, sliding_window=8)
    cfg["text_config"].update({"hidden_size": 128, "intermediate_size": 256, "head_dim": 32,
                               "num_attention_heads": 4, "num_key_value_heads": 2})
    gm = rd.Model(ctx, cfg)
    for name, v, s in fixtures.custom_model(cfg, seed=6):
        gm.set_tensor(name, v, s)
    gm.finalize()
    ops = rd.LayerOps(gm)
    x = ctx.to_device(np.zeros((6, 128), dtype=np.int32))
    small = rd.KvCache(gm, 0, 5)  # layer 0 is sliding (window 8), room for 5 tokens
    with pytest.raises(rd.DetError, match="KV cache capacity exceeded"):
        ops.layer_prefill(0, x, 6, None, None, small, x)
    small = rd.KvCache(gm, 0, 5)
    ops.layer_prefill(0, x, 5, None, None, small, x)
    assert small.info()[0] == 5
    row = ctx.to_device(np.zeros(128, dtype=np.int32))
    with pytest.raises(rd.DetError, match="KV cache capacity exceeded"):
        ops.layer_decode(0, row, None, small, None, 5, row)
    linear = rd.KvCache(gm, 1, 5)  # layer 1 is full attention
    ops.layer_prefill(1, x, 5, None, None, linear, x)
    with pytest.raises(rd.DetError, match="KV cache capacity exceeded"):
        ops.layer_decode(1, row, None, linear, None, 5, row)
    ring = rd.KvCache(gm, 0, 8)  # sized at the window: the trim keeps it going
    ops.layer_prefill(0, x, 5, None, None, ring, x)
    for pos in range(5, 12):
        ops.layer_decode(0, row, None, ring, None, pos, row)
    assert ring.info()[0] == 8


class _Shifted:
    """A device buffer's view `words` int32 past its start (not 16-byte aligned)."""

    def __init__(self, buf, words=1):
        self.buf, self.ptr = buf, buf.ptr + 4 * words


@pytest.mark.parametrize("prompt,window,donor", [(1, 24, False), (40, 24, False), (70, 512, False), (700, 40, True)])
def test_layer_decode_routes_agree(ctx, prompt, window, donor):
    """det_layer_decode on the fused step's kernels (aligned rows, the cache's next position) against the
    per-op form (rows off alignment), for sliding rings past their wrap, full and donor caches: the same
    rows and the same cache contents, step after step; a position other than the cache's length takes the
    per-op form and the next fused step still agrees."""
    cfg = synthetic.e4b_config(layers=4, vocab=512, sliding_window=window)
    if donor:
        cfg["text_config"]["num_kv_shared_layers"] = 2
    model = rd.Model(ctx, cfg)
    for name, v, s in synthetic.synthetic_model_fast(cfg, 3, scale_max=256):
        model.set_tensor(name, v, s)
    model.finalize()
    H, tc = 2560, cfg["text_config"]
    rng = np.random.default_rng(prompt)
    rows = np.rint(rng.normal(size=(prompt, H)) * 4 * 65536).astype(np.int32)
    steps = [np.rint(rng.normal(size=H) * 4 * 65536).astype(np.int32) for _ in range(5)]

    def play(shift: bool):
        ops = rd.LayerOps(model)
        caches = {l: rd.KvCache(model, l, prompt + 8) for l in range(4) if donor_of(tc, l) is None}
        x, out = ctx.to_device(rows), ctx.empty((prompt, H))
        for l in caches:
            ops.layer_prefill(l, x, prompt, None, None, caches[l], out)
        got = []
        for i, row in enumerate(steps):
            pos = prompt + i
            buf, res = ctx.empty(H + 1), ctx.empty(H + 1)
            src, dst = (_Shifted(buf), _Shifted(res)) if shift else (buf, res)
            buf.upload(np.concatenate([np.zeros(int(shift), np.int32), row, np.zeros(1 - int(shift), np.int32)]))
            for l in range(4):
                d = donor_of(tc, l)
                rope = pos + (7 if i == 2 and d is None and l == 0 else 0)
                ops.layer_decode(l, src, None, caches.get(l), None if d is None else caches[d], rope, dst)
                got.append(res.numpy()[int(shift):H + int(shift)].copy())
            if i == 3:  # in place
                ops.layer_decode(3 if not donor else 1, src, None, caches.get(3 if not donor else 1), None,
                                 pos + 1, src)
                got.append(buf.numpy()[int(shift):H + int(shift)].copy())
                break
        return got, [c.read_logical() for c in caches.values()]

    a, b = play(False), play(True)
    assert len(a[0]) == len(b[0]) and all(np.array_equal(p, q) for p, q in zip(a[0], b[0]))
    for (k0, v0), (k1, v1) in zip(a[1], b[1]):
        assert np.array_equal(k0, k1) and np.array_equal(v0, v1)


def test_recorded_layer_calls_keep_their_scratch():
    """A graph of layer calls replays correctly after later calls on the same scratch and context have replaced
    every scratch buffer it uses with a larger one: the decode buffers (a larger cache), the row buffers and the
    GEMM, GEMV and attention areas (more rows, a wider matrix)."""
    cfg = synthetic.e4b_config(layers=2, vocab=512, sliding_window=64)
    cfg["text_config"].update({"hidden_size": 128, "intermediate_size": 256, "head_dim": 64,
                               "num_attention_heads": 4, "num_key_value_heads": 1})
    own = rd.Context(0)  # (scratch of its own, so that it starts small)
    model = rd.Model(own, cfg)
    for name, v, s in fixtures.custom_model(cfg, seed=9):
        model.set_tensor(name, v, s)
    model.finalize()
    assert model.fused_decode
    rng = np.random.default_rng(4)
    acts = lambda *shape: np.rint(rng.normal(size=shape) * 65536).astype(np.int32)  # noqa: E731
    ops, n = rd.LayerOps(model), 20
    prompt, row = own.to_device(acts(n, 128)), own.to_device(acts(128))
    mid, out, wide = own.empty((n, 128)), own.empty(128), own.empty(1000)
    cache = rd.KvCache(model, 0, 64)
    q, s = synthetic.fast_int8_matrix(3, 1000, 128, 16)
    mat = own.upload_matrix(q, s)

    def calls():
        ops.layer_prefill(0, prompt, n, None, None, cache, mid)  # GEMM, attention and row scratch
        ops.layer_decode(0, row, None, cache, None, n, out)      # decode scratch
        own.det_linear_into(mat, out, wide)                      # GEMV scratch

    calls()  # (their scratch exists now)
    want = [b.numpy().copy() for b in (mid, out, wide)]
    graph = own.capture(calls)
    big, rows = rd.KvCache(model, 1, 3000), 700
    many, more = own.to_device(acts(rows, 128)), own.empty((rows, 128))
    wq, ws = synthetic.fast_int8_matrix(4, 32, 40000, 16)
    filler = []
    for i in range(3):
        ops.layer_prefill(1, many, rows, None, None, big, more)
        ops.layer_decode(1, row, None, big, None, rows, more)
        own.upload_matrix(wq, ws)
        filler.append(own.to_device(acts(1 << 20)))  # takes freed memory, if any was freed
        for b in (mid, out, wide):
            b.upload(np.zeros(b.shape, np.int32))
        graph.launch()
        assert all(np.array_equal(w, b.numpy()) for w, b in zip(want, (mid, out, wide))), i


def free_memory() -> int:
    """Free bytes of the device, from the HIP runtime that the library is linked against."""
    free, total = rd.C.c_size_t(), rd.C.c_size_t()
    assert rd.lib().hipMemGetInfo(rd.C.byref(free), rd.C.byref(total)) == 0
    return free.value


def test_session_memory_is_its_buffers():
    """A session takes its caches and step buffers and no more, also where the vocabulary row alone is a MiB."""
    cfg = synthetic.e4b_config(layers=2, vocab=262144, sliding_window=64)
    cfg["text_config"].update({"hidden_size": 128, "intermediate_size": 256, "head_dim": 64, "num_attention_heads": 4,
                               "num_key_value_heads": 2, "layer_types": ["full_attention"] * 2})
    own = rd.Context(0)
    model = rd.Model(own, cfg)
    for name, v, s in fixtures.custom_model(cfg, seed=2):
        model.set_tensor(name, v, s)
    model.finalize()
    tokens = 200_000
    kv = 2 * 2 * tokens * 2 * 64 * 4  # layers, keys and values, rows, KV heads x head dim, int32
    rest = 4 * tokens * 4 + 262144 * 4  # score rows, logits
    before = free_memory()
    session = model.session(tokens)
    used = before - free_memory()
    assert kv <= used <= kv + rest + (8 << 20), (used, kv)
    del session


@pytest.mark.parametrize("tokens", [2**37, 2**54, 2**60, 2**62, 2**64 - 1])
@pytest.mark.parametrize("sliding", [False, True])
def test_session_too_large_for_any_device_is_refused(ctx, tokens, sliding):
    """Sizes that wrap around 64 bits (2^54 rows of 256 words, 2^60 score rows of 4 heads) are refused like any
    other session that does not fit, with and without caches that grow with it."""
    cfg = synthetic.e4b_config(layers=2, vocab=512, sliding_window=16)
    cfg["text_config"].update({"hidden_size": 128, "intermediate_size": 256, "head_dim": 64, "num_attention_heads": 4,
                               "num_key_value_heads": 4})
    if sliding:
        cfg["text_config"]["layer_types"] = ["sliding_attention"] * 2
    model = rd.Model(ctx, cfg)
    for name, v, s in fixtures.custom_model(cfg, seed=2):
        model.set_tensor(name, v, s)
    model.finalize()
    with pytest.raises(rd.DetError, match="out of memory"):
        model.session(tokens)
    model.session(64).prefill([1, 2, 3])


def test_layer_decode_scratch_is_bounded_by_the_window():
    """A decode in a cache of millions of rows takes scratch for the longest window there is, not for the cache, and
    gives what a small cache gives."""
    cfg = synthetic.e4b_config(layers=2, vocab=512, sliding_window=64)
    cfg["text_config"].update({"hidden_size": 128, "intermediate_size": 256, "head_dim": 64, "num_attention_heads": 4,
                               "num_key_value_heads": 1})
    own = rd.Context(0)
    model = rd.Model(own, cfg)
    for name, v, s in fixtures.custom_model(cfg, seed=3):
        model.set_tensor(name, v, s)
    model.finalize()
    rng = np.random.default_rng(6)
    rows, row = (own.to_device(np.rint(rng.normal(size=(n, 128)) * 65536).astype(np.int32)) for n in (30, 1))
    got = []
    for cap in (64, 4_000_000):
        ops, cache, out = rd.LayerOps(model), rd.KvCache(model, 1, cap), own.empty((30, 128))
        ops.layer_prefill(1, rows, 30, None, None, cache, out)
        before = free_memory()
        for pos in range(30, 34):
            ops.layer_decode(1, row, None, cache, None, pos, out)
            got.append(out.numpy()[0].copy())
        assert before - free_memory() <= 8 << 20, cap
    assert all(np.array_equal(a, b) for a, b in zip(got[:4], got[4:]))
