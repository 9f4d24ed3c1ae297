"""The Nulunex decoder through the engine, against ``plain_nulunex``: whole prompts, decoding token by token, prompts in
pieces down to two tokens, batches of unequal requests, slots and pages used again, long decoding across page, window and
chunk borders, a key made to stand out just inside and just outside every window and chunk, the first tokens of a
sequence and their sinks, faults planted in the plain implementation that must show, other sizes (also ones where the
usual sizes coincide or are 1), the residual after every layer run, greedy generation through the engine's entry point,
the command line and the trace replay tool."""
import copy
import json
import os
import random
import subprocess
import sys

import numpy as np
import pytest
import torch

import engine_utils as U
import plain_nulunex as P

pytestmark = pytest.mark.gpu

CONFIGS = {
    # both mixers, a layer run twice with its own keys each time, one without a feed-forward, sizes that are no multiples
    # of 16, a window and a chunk that are no multiples of a page
    "mixed": lambda: P.config([
        P.latent_layer(3, 12, 6, 20, 40, 37, base=500.0, mlp=P.dense(56, limit=0.8)),
        P.attention_layer(6, 3, 16, 50, 8, base=900.0, mlp=P.dense(24, limit=2.5)),
        P.latent_layer(2, 8, 2, 4, 16, 90, mlp=None),
        P.attention_layer(6, 3, 16, 50, 8, base=900.0, mlp=P.dense(24, limit=2.5), weights_of=1),
        P.latent_layer(3, 12, 6, 20, 40, 37, base=500.0, mlp=P.dense(56, limit=0.8), weights_of=0)],
        vocab=131, width=40, eps=2e-6),
    # a width that is no multiple of 8 (no matrix-core packing), one head, one latent element, a window of one position, a
    # chunk shorter than a page, one pair turned, no chunk at all
    "odd": lambda: P.config([
        P.attention_layer(1, 1, 10, 7, 2, base=3.0, mlp=P.dense(30, limit=0.4)),
        P.latent_layer(1, 5, 2, 3, 1, 1, mlp=None),
        P.latent_layer(5, 1, 4, 7, 19, 150, base=77.0, mlp=P.dense(18, limit=6.0)),
        P.attention_layer(6, 2, 4, None, 4, scale=0.9, mlp=P.dense(30, limit=0.4))], vocab=97, width=60, eps=1e-3),
    # sizes the matrix cores take everywhere, the prompt form with every head's own keys, a window and a chunk of exactly
    # a page and two
    "even": lambda: P.config([
        P.latent_layer(8, 16, 8, 32, 48, 64, mlp=P.dense(256, limit=2.0)),
        P.attention_layer(4, 2, 32, 128, 32, mlp=P.dense(192, limit=1.0)),
        P.latent_layer(20, 32, 16, 16, 64, 128, base=100.0, mlp=P.dense(64, limit=1.5)),
        P.latent_layer(8, 16, 8, 32, 48, 64, mlp=P.dense(256, limit=2.0), weights_of=0),
        P.attention_layer(4, 2, 32, 128, 32, mlp=P.dense(192, limit=1.0), weights_of=1)], vocab=256, width=128),
    # cached rows as wide as the kernels take, no window
    "wide": lambda: P.config([
        P.latent_layer(3, 64, 64, 80, 512, None, mlp=P.dense(40, limit=3.0)),
        P.latent_layer(2, 24, 16, 16, 272, 100, mlp=None)], vocab=61, width=72),
}


@pytest.fixture(scope="module")
def models(tmp_path_factory):
    made = {}

    def get(name):
        if name not in made:
            cfg = CONFIGS[name]()
            w = P.random_weights(cfg, seed=len(name))
            folder = U.write_model(str(tmp_path_factory.mktemp(name)), cfg, w)
            made[name] = (cfg, w, folder)
        return made[name]
    return get


def engine(folder, dtype, **kw):
    from agave_amd.engine import Engine
    kw.setdefault("max_slots", 4)
    kw.setdefault("max_context", 512)
    return Engine.from_folder(folder, dtype=dtype, **kw)


def close(got, ref, dtype, what):
    """32-bit: every row within 3e-5 of the largest logit.  bfloat16: 4 % of the largest logit for all rows but one
    in twenty, twice that for those."""
    scale = float(ref.abs().max())
    err = (got.double() - ref).abs().max(dim=-1).values
    where = f"{what}: error {float(err.max()):.3e} of {scale:.3e} at row {int(err.argmax())}"
    if dtype == "float32":
        assert float(err.max()) <= 3e-5 * scale, where
    else:
        assert float(err.max()) <= 0.08 * scale, where
        assert int((err > 0.04 * scale).sum()) <= max(1, len(err) // 20), where


@pytest.mark.parametrize("name", list(CONFIGS))
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_whole_tail_and_pieces(models, name, dtype):
    cfg, w, folder = models(name)
    eng = engine(folder, dtype)
    toks = U.random_tokens(200, cfg["vocab"], 1)
    ref = P.forward(cfg, w, toks)
    close(U.run_whole(eng, toks), ref, dtype, "whole")
    close(U.run_tail(eng, toks, 150), ref, dtype, "the last 150 one by one, across page, window and chunk borders")
    close(U.run_tail(eng, toks, 199), ref, dtype, "token by token from the first")
    for piece in (2, 7, 64, 100):                 # the prompt enters in pieces of this many tokens
        eng.prefill_chunk = piece
        close(U.run_whole(eng, toks[:170]), ref[:170], dtype, f"pieces of {piece}")
    eng.prefill_chunk = 0
    assert eng.cache.slots.n_free == eng.cache.max_slots
    assert all(g.pool.n_free == g.pool.n_pages for g in eng.cache.groups)


@pytest.mark.parametrize("name", list(CONFIGS))
def test_32_bit_products_in_slices(models, name, monkeypatch):
    """What reads a product's rows adds up its slices, or gets them added up."""
    made = U.products_in_slices(monkeypatch)
    test_whole_tail_and_pieces(models, name, "float32")
    assert made


def test_residual_after_every_layer_run(models):
    """The residual stream after each run of a layer (one that runs another layer's tensors counts as itself), read off
    the engine between its blocks."""
    from agave_amd.parts.norm import add_branch
    cfg, w, folder = models("mixed")
    eng = engine(folder, "float32")
    eng.use_graphs = False
    toks = U.random_tokens(90, cfg["vocab"], 4)
    want, seen = [], []
    P.forward(cfg, w, toks, layers_out=want)
    for b in eng.model.blocks:
        def wrapped(h, pending, step, memory, writes, inner=b.forward):
            if pending is not None:
                stream = h.clone()
                add_branch(stream, pending)
                seen.append(stream.cpu())
            return inner(h, pending, step, memory, writes)
        b.forward = wrapped
    U.run_whole(eng, toks)
    assert len(eng.model.blocks) == 3 and len(seen) == len(want) - 1 == 4
    for i, (got, ref) in enumerate(zip(seen, want)):
        assert float((got.double() - ref).abs().max()) < 3e-5 * float(ref.abs().max()), f"after layer run {i}"


@pytest.mark.parametrize("name, dtype", [("mixed", "float32"), ("mixed", "bfloat16"), ("even", "bfloat16")])
def test_batches_of_unequal_requests_and_slots_used_again(models, name, dtype):
    """Three batches one after another over the same three slots, through pools of pages that only hold them because
    pages come back."""
    cfg, w, folder = models(name)
    eng = engine(folder, dtype, max_slots=3, max_context=256, cache_tokens=448)
    for b, (lens, first) in enumerate([((50, 1, 130), (30, 1, 2)), ((70, 33), (69, 1)), ((90, 9, 140), (5, 9, 101))]):
        reqs = [U.random_tokens(n, cfg["vocab"], 10 * b + i) for i, n in enumerate(lens)]
        outs = U.run_batched(eng, reqs, first)
        for i, (r, o) in enumerate(zip(reqs, outs)):
            close(o, P.forward(cfg, w, r), dtype, f"batch {b} request {i}")
    assert eng.cache.slots.n_free == eng.cache.max_slots
    assert all(g.pool.n_free == g.pool.n_pages for g in eng.cache.groups)


def test_a_batch_of_more_than_sixteen(models):
    """Eighteen sequences decoded together (more than the decode step's joint kernels take at a time)."""
    cfg, w, folder = models("even")
    eng = engine(folder, "bfloat16", max_slots=18, max_context=192)
    reqs = [U.random_tokens(70 + 3 * i, cfg["vocab"], 300 + i) for i in range(18)]
    for r, o in zip(reqs, U.run_batched(eng, reqs, [len(r) - 12 for r in reqs])):
        close(o, P.forward(cfg, w, r), "bfloat16", f"{len(r)} tokens in a batch of eighteen")


def test_prompts_from_their_first_position_make_every_heads_keys(models):
    """In bfloat16, with head sizes the matrix cores take, a step of prompts that all start at position 0 runs the latent
    attention over every head's own keys and values; its pieces and the decoding after it read the latent rows."""
    cfg, w, folder = models("even")
    eng = engine(folder, "bfloat16", max_slots=3, max_context=512)
    latent = [b.mixer for b in eng.model.blocks if hasattr(b.mixer, "fresh_prompt")]
    assert len(latent) == 2 and all(m.fresh_ok and m.decode_ok for m in latent)
    calls = []
    for m in latent:
        def counted(*a, inner=m.fresh_prompt, **k):
            calls.append(1)
            return inner(*a, **k)
        m.fresh_prompt = counted
    reqs = [U.random_tokens(n, cfg["vocab"], 40 + n) for n in (150, 40, 128)]
    refs = [P.forward(cfg, w, r) for r in reqs]
    for r, o in zip(refs, U.run_batched(eng, reqs, (141, 33, 128))):
        close(o, r, "bfloat16", "prompts together, then decoded")
    assert len(calls) == 3                                  # three latent runs of two layers' tensors
    eng.prefill_chunk = 70                                  # the first piece from position 0, the others behind it
    close(U.run_whole(eng, reqs[0]), refs[0], "bfloat16", "pieces of 70")
    assert len(calls) == 6
    eng.prefill_chunk = 0
    close(U.run_tail(eng, reqs[2], 100), refs[2], "bfloat16", "28 tokens (the latent rows' form), then decoded")
    assert len(calls) == 6


def test_the_cache_as_the_mixers_asked(models):
    cfg, w, folder = models("mixed")
    eng = engine(folder, "bfloat16")
    keys = {m: eng.cache.group_keys[g] for m, g in eng.cache.group_of_memory.items()}
    assert set(keys) == {0, 1, 2, 3, 4} and not eng.cache.state
    assert keys[0] == keys[4] and (keys[0].window, keys[0].n_kv_heads, keys[0].head_dim, keys[0].v_head_dim) == (37, 1, 46, 40)
    assert keys[1] == keys[3] and (keys[1].chunk, keys[1].window, keys[1].n_kv_heads, keys[1].head_dim) == (50, None, 3, 16)
    from agave_amd.ops import library
    slot = eng.alloc_slot()
    eng.step([slot], [[1, 2]])
    eng.free_slot(slot)
    loaded = library.loaded_paths()
    for name in ("latent.so", "attention_latent.so", "attention_biased.so"):
        assert any(p.endswith(name) for p in loaded), name


@pytest.mark.parametrize("name, dtype", [("even", "float32"), ("even", "bfloat16"), ("mixed", "float32")])
def test_long_decoding(models, name, dtype):
    cfg, w, folder = models(name)
    eng = engine(folder, dtype, max_slots=1, max_context=1024, cache_tokens=64 * 11)
    toks = U.random_tokens(700, cfg["vocab"], 9)
    close(U.run_tail(eng, toks, 500), P.forward(cfg, w, toks), dtype, "500 tokens decoded")


# ---------------------------------------------------------------- a key that stands out
VOCAB_NEEDLE = 40


def needle_model(kind: str, size, boost=30.0, value=25.0):
    """One layer whose head 0 is made to look for one token: token ``A``'s key is turned towards token ``Q``'s query in
    the elements that are not rotated and its value is made large, so that the logits at a ``Q`` change much with whether
    ``A`` is seen.  A layer's input is a function of the token alone in a model of one layer, and there are fewer tokens
    than the rows are long: the matrices are changed along the part of ``A``'s row that is orthogonal to every other
    token's, so no other token's key or value moves."""
    A, Q = 0, 1
    if kind == "attention":
        cfg = P.config([P.attention_layer(2, 1, 16, size, 8, scale=1.0)], vocab=VOCAB_NEEDLE, width=64)
    else:
        cfg = P.config([P.latent_layer(2, 8, 8, 12, 64, size, base=100.0)], vocab=VOCAB_NEEDLE, width=64)
    w = P.random_weights(cfg, 3)
    eps, m, p = cfg["norm"]["eps"], cfg["layers"][0]["mixer"], "l0.mix."
    h = P.rms(w["embed"], eps) * w["l0.norm1"]                               # [vocab, width]: every token's input

    def only_for_a(rows):
        coef = torch.linalg.lstsq(rows[1:].T, rows[A][:, None]).solution[:, 0]
        d = rows[A] - rows[1:].T @ coef                                     # orthogonal to every other token's row
        return d / float(d @ rows[A])
    if kind == "attention":
        q0 = P.rms((h[Q] @ w[p + "q"].T).view(2, 16), eps)[0].clone()
        q0[:8] = 0.0
        d = only_for_a(h)
        w[p + "k"] = w[p + "k"] + boost * torch.outer(q0 / q0.norm(), d)     # (a key is its value too: the value moves by as much)
        names = [p + "k"]
    else:
        c = P.rms((h @ w[p + "dkv"].T)[:, :m["kv_rank"]], eps) * w[p + "dkv.norm"]
        q0 = (h[Q] @ w[p + "q"].T).view(2, 16)[0, :8]
        d = only_for_a(c)
        uk, uv = w[p + "uk"].clone(), w[p + "uv"].clone()
        uk[:8] += boost * torch.outer(q0 / (q0.norm() ** 2), d) / m["scale"]
        uv[:12] += value * torch.outer(torch.ones(12, dtype=P.F), d)
        w[p + "uk"], w[p + "uv"] = uk, uv
        names = [p + "uk", p + "uv"]
    for n in names:
        w[n] = w[n].to(torch.float32).to(P.F)
    return cfg, w, A, Q


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("kind, size", [("latent", 70), ("latent", 64), ("latent", 300), ("latent", None), ("attention", 96),
                                        ("attention", 64), ("attention", 50), ("attention", None)])
def test_a_key_at_the_edges_of_windows_and_chunks(dtype, kind, size):
    """The key that the last queries look for stands just inside and just outside what the last query sees (the window's
    far end; the chunk's first position and the one before it), at the query's own side, at page borders, and at the
    sequence's first positions; the queries come in the prompt, in pieces of it, and decoded one by one."""
    from agave_amd.engine import Engine
    cfg, w, A, Q = needle_model(kind, size)
    # (the changed matrices are handed over in 32-bit, so that the orthogonal direction survives; a bfloat16 engine casts them)
    eng = Engine.from_tensors(cfg, {k: v.float() for k, v in w.items()}, dtype=dtype, max_slots=2, max_context=512,
                              keep_stored_precision=False)
    T = 430
    last = T - 1
    if size is None:
        places = {0: True, 1: True, 63: True, 64: True, 300: True, last - 1: True}
    else:
        inside = last - size + 1 if kind == "latent" else last // size * size
        places = {inside: True, inside - 1: False, last - 1: True, 0: False, 1: False, 63: False, 64: False}
        if size == 300:
            places.update({191: True, 192: True, 255: True, 256: True})
    for at, seen in places.items():
        toks = [2 + t % (VOCAB_NEEDLE - 2) for t in U.random_tokens(T, 1000, at + 5)]
        toks[-1] = Q
        toks[at] = A
        without = list(toks)
        without[at] = 7
        ref, ref_without = P.forward(cfg, w, toks), P.forward(cfg, w, without)
        scale = float(ref.abs().max())
        moved = float((ref[-1] - ref_without[-1]).abs().max())
        if seen:
            assert moved > 0.1 * scale, (at, moved, scale)
        else:
            assert moved < 1e-9 * scale, (at, moved, scale)
        eng.prefill_chunk = 0
        runs = {"whole": U.run_whole(eng, toks), "decoded": U.run_tail(eng, toks, 100 if at < 200 else T - at + 3)}
        eng.prefill_chunk = 50
        runs["pieces"] = U.run_whole(eng, toks)
        for what, got in runs.items():
            if dtype == "float32":
                close(got, ref, dtype, f"key at {at}, {what}")
            if seen:
                assert float((got[-1].double() - ref[-1]).abs().max()) < (0.002 if dtype == "float32" else 0.25) * moved, (at, what)
            else:
                # what the key would do if it were seen is as large as where it is seen
                assert float((got[-1].double() - ref[-1]).abs().max()) < (3e-5 if dtype == "float32" else 0.08) * scale, (at, what)


# ---------------------------------------------------------------- faults planted in the plain implementation
def planted(monkeypatch, fault):
    """The plain implementation with one mistake."""
    if fault == "attention without its sink":
        inner = P.softmax_with_sink
        monkeypatch.setattr(P, "softmax_with_sink", lambda s, see, sink: inner(s, see, -1e9 if sink == 0.0 else sink))
    elif fault == "latent attention without its sink":
        inner = P.softmax_with_sink
        monkeypatch.setattr(P, "softmax_with_sink", lambda s, see, sink: inner(s, see, sink if sink == 0.0 else -1e9))
    elif fault == "a window one longer":
        inner = P.sees_window
        monkeypatch.setattr(P, "sees_window", lambda T, size: inner(T, None if size is None else size + 1))
    elif fault == "chunks one later":
        def shifted(T, size):
            i, j = torch.arange(T)[:, None], torch.arange(T)[None, :]
            return (j <= i) if size is None else (j <= i) & ((i - 1) // size == (j - 1) // size)
        monkeypatch.setattr(P, "sees_chunk", shifted)
    elif fault == "the other pairs turned":
        monkeypatch.setattr(P, "turn_neighbours", P.turn_halves)
    elif fault == "values after norm and rotation":
        def attention(h, w, p, m, eps, inner=P.attention):
            T, H, G, d = h.shape[0], m["heads"], m["kv_heads"], m["dim"]
            pos = torch.arange(T)
            q, k = (h @ w[p + "q"].T).view(T, H, d), (h @ w[p + "k"].T).view(T, G, d)
            q, k = (P.rms(P.turn_halves(x, pos, m["rot"]["dims"], m["rot"]["base"]), eps) for x in (q, k))
            see = P.sees_chunk(T, m["mask"]["size"] if m.get("mask") else None)
            out = torch.stack([P.softmax_with_sink((q[:, n] @ k[:, n // (H // G)].T) * m["scale"], see, 0.0) @ k[:, n // (H // G)] for n in range(H)], 1)
            return out.reshape(T, H * d) @ w[p + "o"].T
        monkeypatch.setattr(P, "attention", attention)
    elif fault == "an up value without its one":
        monkeypatch.setattr(P, "clamped_swish", lambda g, u, L: torch.clamp(g, max=L) * torch.sigmoid(1.702 * torch.clamp(g, max=L)) * torch.clamp(u, -L, L))
    elif fault == "an up value clamped on one side":
        monkeypatch.setattr(P, "clamped_swish", lambda g, u, L: torch.clamp(g, max=L) * torch.sigmoid(1.702 * torch.clamp(g, max=L)) * (torch.clamp(u, max=L) + 1))
    elif fault == "a shared layer with its owner's keys":
        # the second run of layer 1's tensors reads the keys of the first (its queries are its own)
        inner, kept = P.attention, {}

        def attention(h, w, p, m, eps):
            if p in kept:
                return _with_keys_of(h, kept[p], w, p, m, eps)
            kept[p] = h
            return inner(h, w, p, m, eps)
        monkeypatch.setattr(P, "attention", attention)
    else:
        raise AssertionError(fault)


def _with_keys_of(h, h_keys, w, p, m, eps):
    T, H, G, d = h.shape[0], m["heads"], m["kv_heads"], m["dim"]
    pos = torch.arange(T)
    q, k = (h @ w[p + "q"].T).view(T, H, d), (h_keys @ w[p + "k"].T).view(T, G, d)
    v = k
    q, k = (P.rms(P.turn_halves(x, pos, m["rot"]["dims"], m["rot"]["base"]), eps) for x in (q, k))
    see = P.sees_chunk(T, m["mask"]["size"] if m.get("mask") else None)
    out = torch.stack([P.softmax_with_sink((q[:, n] @ k[:, n // (H // G)].T) * m["scale"], see, 0.0) @ v[:, n // (H // G)] for n in range(H)], 1)
    return out.reshape(T, H * d) @ w[p + "o"].T


FAULTS = ["attention without its sink", "latent attention without its sink", "a window one longer", "chunks one later",
          "the other pairs turned", "values after norm and rotation", "an up value without its one",
          "an up value clamped on one side", "a shared layer with its owner's keys"]


def test_planted_faults_show(models, monkeypatch):
    """The engine's logits are far (a hundred times the tolerance) from what each mistake would give, and near what the
    plain implementation gives without it: the comparisons of this file would show every one of these."""
    cfg, w, folder = models("mixed")
    eng = engine(folder, "float32")
    toks = U.random_tokens(120, cfg["vocab"], 31)
    got = U.run_tail(eng, toks, 40)
    ref = P.forward(cfg, w, toks)
    close(got, ref, "float32", "no fault")
    scale = float(ref.abs().max())
    for fault in FAULTS:
        with monkeypatch.context() as mp:
            planted(mp, fault)
            wrong = P.forward(cfg, w, toks)
        assert float((got.double() - wrong).abs().max()) > 3e-3 * scale, fault
    close(got, P.forward(cfg, w, toks), "float32", "the mistakes are gone again")


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_the_first_tokens_and_their_sinks(models, dtype):
    """Sequences of one, two and three tokens, alone and together: at the first position a sink takes its share beside a
    single key."""
    cfg, w, folder = models("even")
    eng = engine(folder, dtype, max_slots=3)
    reqs = [U.random_tokens(n, cfg["vocab"], 60 + n) for n in (1, 2, 3)]
    refs = [P.forward(cfg, w, r) for r in reqs]
    for r, ref in zip(reqs, refs):
        close(U.run_whole(eng, r), ref, dtype, f"{len(r)} tokens")
    for o, ref in zip(U.run_batched(eng, reqs, (1, 1, 1)), refs):
        close(o, ref, dtype, "together, one by one")


# ---------------------------------------------------------------- other sizes
def random_config(seed: int) -> dict:
    """A configuration drawn from a seed: two to six layers of either kind in any order, head counts and sizes that the
    matrix cores take and ones they do not, windows and chunks around page borders, layers that run an earlier one's
    tensors."""
    rng = random.Random(seed)
    layers = []
    for i in range(rng.randint(2, 6)):
        own = [j for j, layer in enumerate(layers) if "weights_of" not in layer]
        if own and rng.random() < 0.3:
            j = rng.choice(own)
            layers.append(dict(copy.deepcopy(layers[j]), weights_of=j))
            continue
        mlp = None if rng.random() < 0.2 else P.dense(rng.choice([64, 96, 200, 50]), limit=rng.choice([0.5, 1.5, 7.0]))
        size = rng.choice([1, 2, 7, 31, 63, 64, 65, 72, 100, 127, 128, 129, 200, 400, None])
        base = rng.choice([100.0, 1e4, 1e6])
        if rng.random() < 0.4:
            kv = rng.choice([1, 1, 2, 3])
            dim = rng.choice([8, 16, 24, 48, 64, 80, 128, 20, 36])
            layers.append(P.attention_layer(kv * rng.choice([1, 2, 4, 8]), kv, dim, size, rng.choice([dim, dim // 2 // 2 * 2, 2, 0]),
                                            base=base, scale=rng.choice([dim ** -0.5, 1.7 * dim ** -0.5]), mlp=mlp))
        else:
            layers.append(P.latent_layer(rng.choice([1, 2, 3, 4, 8, 17]), rng.choice([8, 16, 24, 32, 64, 12, 128]),
                                         rng.choice([2, 8, 16, 32, 64, 6]), rng.choice([16, 32, 48, 128, 20]),
                                         rng.choice([16, 48, 64, 96, 160, 256, 20, 30]), size, base=base, mlp=mlp))
    return P.config(layers, vocab=rng.choice([97, 256, 1000]), width=rng.choice([64, 96, 128, 160, 320, 72, 100]),
                    eps=rng.choice([1e-6, 1e-5]))


@pytest.mark.parametrize("seed", list(range(21, 31)))
def test_configurations_drawn_at_random(seed):
    from agave_amd.engine import Engine
    cfg = random_config(seed)
    w = P.random_weights(cfg, seed)
    toks = U.random_tokens(330, cfg["vocab"], seed)
    others = [U.random_tokens(n, cfg["vocab"], seed + 100 + n) for n in (1, 150)]
    refs = [P.forward(cfg, w, t) for t in [toks] + others]
    for dtype in ("float32", "bfloat16"):
        eng = Engine.from_tensors(cfg, {k: v.bfloat16() for k, v in w.items()}, dtype=dtype, max_slots=3, max_context=512)
        close(U.run_tail(eng, toks, 140), refs[0], dtype, f"{cfg}: tail")
        for o, r in zip(U.run_batched(eng, [toks] + others, (300, 1, 100)), refs):
            close(o, r, dtype, f"{cfg}: in a batch")


# ---------------------------------------------------------------- the ways in
@pytest.mark.parametrize("name, dtype", [("mixed", "float32"), ("wide", "float32")])
def test_greedy_generation_through_the_entry_point(models, name, dtype):
    from agave_amd.sampling import SamplingParams
    cfg, w, folder = models(name)
    eng = engine(folder, dtype, max_slots=2, max_context=128)
    prompts = [U.random_tokens(7, cfg["vocab"], 50), U.random_tokens(45, cfg["vocab"], 51), U.random_tokens(1, cfg["vocab"], 52)]
    res = eng.generate(prompts, SamplingParams(temperature=0.0, max_tokens=8))      # three requests, two slots: a slot is used again
    for p, r in zip(prompts, res):
        seq = list(p)
        for _ in range(8):
            seq.append(P.argmax_first(P.forward(cfg, w, seq)[-1]))
        assert list(r.tokens) == seq[len(p):]


def test_decode_steps_replayed_as_graphs_match_eager_ones(models):
    """The recorded decode step, replayed many times with other steps between, against the same steps run eagerly."""
    cfg, w, folder = models("even")
    toks = [U.random_tokens(n, cfg["vocab"], 400 + n) for n in (100, 66)]
    outs = []
    for graphs in (True, False):
        eng = engine(folder, "bfloat16", max_slots=3, max_context=256)
        eng.use_graphs = graphs
        a = U.run_batched(eng, toks, (40, 30))
        U.run_tail(eng, toks[0], 20)                     # a step of another kind between
        b = U.run_batched(eng, toks, (40, 30))
        for x, y in zip(a, b):
            assert torch.equal(x, y)
        outs.append(b)
    for x, y in zip(*outs):
        assert float((x - y).abs().max()) <= 0.02 * float(y.abs().max())


def test_command_line_and_trace_replay(models, tmp_path):
    cfg, w, folder = models("odd")
    root = U.ROOT
    out = subprocess.run([sys.executable, os.path.join(root, "bin", "agave_amd"), folder, "3 17 5 80 2", "-n", "5", "--dtype", "float32",
                          "--json"], capture_output=True, text=True, timeout=600)
    assert out.returncode == 0, out.stderr[-2000:]
    seq = [3, 17, 5, 80, 2]
    for _ in range(5):
        seq.append(P.argmax_first(P.forward(cfg, w, seq)[-1]))
    got = json.loads(out.stdout.strip().splitlines()[-1])
    assert got["outputs"][0]["tokens"] == seq[5:] and got["outputs"][0]["prompt_tokens"] == 5
    batches = [[U.random_tokens(n, cfg["vocab"], 70 + n) for n in (40, 3, 110)], [U.random_tokens(n, cfg["vocab"], 90 + n) for n in (25, 60)]]
    firsts = [(8, 3, 78), (1, 59)]
    records, where = U.trace_steps_batched(batches, firsts)
    for dtype in ("float32", "bfloat16"):
        steps = U.run_trace_tool(folder, dtype, records, str(tmp_path / dtype), 153, cfg["vocab"])
        for bi, reqs in enumerate(batches):
            for i, r in enumerate(reqs):
                got = torch.from_numpy(np.stack([steps[s][row] for s, row in where[(bi, i)]]))
                close(got, P.forward(cfg, w, r), dtype, f"replay {dtype} batch {bi} request {i}")
