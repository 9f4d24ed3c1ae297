"""What users of this library wait for, as cases that can be timed and checked.

A pass serves one batch of requests through :class:`agave_amd.engine.Engine` as a caller does who brings the tokens (trace
replay, scoring, a draft that is verified): a slot for every sequence, the prompts as one step, then ``steps`` steps of one
given token per sequence, and the slots are given back.  The tokens are given and not drawn from the logits, so that two
correct implementations stay on the same sequences.  A pass returns the logits behind the prompts and behind the last token.

The engine and its weights are made once per model and kept while cases of that model follow one another, as a server keeps
them; the tokens come from the seed.  Weights are random, with the spread that the models' norms and gates need to stay in
the range they work in (activations of order one, forget gates that remember, queries that resemble keys where a read-out is
normed).

``exact`` states the three decoders again in 64 bits, whole sequences at once and without a cache.
"""
from __future__ import annotations

import math

import torch

F = torch.float64

# ---------------------------------------------------------------- the models
# The layer sizes of the published Gemma 3 4B text configuration.
GEMMA3_4B = dict(
    architectures=["Gemma3ForCausalLM"], model_type="gemma3_text", vocab_size=262208, hidden_size=2560, num_hidden_layers=34,
    num_attention_heads=8, num_key_value_heads=4, head_dim=256, query_pre_attn_scalar=256, intermediate_size=10240,
    sliding_window=1024, sliding_window_pattern=6, rope_theta=1e6, rope_local_base_freq=1e4,
    rope_scaling={"rope_type": "linear", "factor": 8.0}, rms_norm_eps=1e-6, tie_word_embeddings=True,
    hidden_activation="gelu_pytorch_tanh", max_position_embeddings=131072, bos_token_id=2, eos_token_id=1)

# A Gemma 3 decoder of a middle size for the 32-bit engine, which serves checks of a checkpoint rather than traffic.
GEMMA3_MEDIUM = dict(
    GEMMA3_4B, vocab_size=32768, hidden_size=2048, num_hidden_layers=8, num_attention_heads=16, num_key_value_heads=4, head_dim=128,
    query_pre_attn_scalar=128, intermediate_size=5376, tie_word_embeddings=False)


def _batasun(width=2048, heads=16, layers=8, kv_rank=512, expert=2048):
    """Latent attention and state-space mixers in turn, a routed feed-forward behind each."""
    moe = {"kind": "moe", "expert": {"ff": expert, "limit": 7.0}, "shared": {"ff": expert, "limit": 7.0}, "router": {"experts": 16, "top": 4}}
    def latent(source):
        m = {"heads": heads, "dim": 128, "rot_dim": 64, "vdim": 128, "q_rank": 3 * width // 4, "kv_rank": kv_rank, "scale": 192 ** -0.5,
             "rot": {"base": 10000.0, "dims": 64}}
        return {"type": "latent_attention", "mixer": m if source is None else dict(m, kv_from=source), "mlp": moe}
    ssm = {"type": "mamba2", "mlp": moe,
           "mixer": {"heads": 2 * width // 64, "vdim": 64, "state": 128, "groups": 1, "conv": 4, "norm_groups": 1}}
    return {"architecture": "Batasun", "vocab": 32768, "width": width, "norm": {"eps": 1e-5},
            "layers": [latent(None) if i % 4 == 0 else latent(i - 3) if i % 4 == 3 else ssm for i in range(layers)]}


def _derosun(width=2048, heads=16, kv_heads=4, layers=8, kv_rank=512, ff=5376):
    """Matrix memories, attention with capped scores and latent attention in turn, dense feed-forwards."""
    memory = {"type": "mlstm", "mixer": {"heads": width // 512, "dim": 256, "vdim": 512, "gate_cap": 15.0}}
    attention = {"type": "attention",
                 "mixer": {"heads": heads, "kv_heads": kv_heads, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "softcap": 30.0,
                           "rot": {"dims": 128, "base": 500000.0, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}}}
    latent = {"type": "latent_attention",
              "mixer": {"heads": heads, "dim": 128, "rot_dim": 64, "vdim": 128, "q_rank": 3 * width // 4, "kv_rank": kv_rank, "scale": 192 ** -0.5,
                        "rot": {"base": 10000.0, "dims": 64, "scaling": {"factor": 40.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}}
    return {"architecture": "Derosun", "vocab": 32768, "width": width, "norm": {"eps": 1e-5}, "postln_alpha": 2.0, "embedding": {"scale": 1.0},
            "layers": [dict((memory, attention, memory, latent)[i % 4], mlp={"kind": "dense", "ff": ff}) for i in range(layers)]}


# name -> (configuration, the engine's element type, slots, longest sequence, positions the cache holds)
MODELS = {
    "gemma3-4b": (GEMMA3_4B, "bfloat16", 64, 16384, 32768),
    "gemma3-medium-f32": (GEMMA3_MEDIUM, "float32", 8, 4096, 8192),
    "batasun-medium": (_batasun(), "bfloat16", 32, 8192, 24576),
    "derosun-medium": (_derosun(), "bfloat16", 32, 8192, 24576),
}


# ---------------------------------------------------------------- the cases
def listed():
    def case(name, model, batch, shortest, longest, steps):
        return {"name": name, "model": model, "batch": batch, "shortest": shortest, "longest": longest, "steps": steps}
    return [
        # one short turn of a chat: the time to its first token is launches and the weights' way from memory
        case("4b prompt 37", "gemma3-4b", 1, 37, 37, 0),
        # an ordinary question, and a page of text
        case("4b prompt 509", "gemma3-4b", 1, 509, 509, 0),
        case("4b prompt 2048", "gemma3-4b", 1, 2048, 2048, 0),
        # a long document, which enters in pieces
        case("4b prompt 10007", "gemma3-4b", 1, 10007, 10007, 0),
        # a batch starts: unequal prompts in one step
        case("4b prompts 8 unequal", "gemma3-4b", 8, 61, 1637, 0),
        # one user's answer
        case("4b decode b1", "gemma3-4b", 1, 150, 150, 48),
        # a small batch in the middle of long sequences, and a full one in the middle of short ones
        case("4b decode b8", "gemma3-4b", 8, 1024, 1024, 96),
        case("4b decode b64", "gemma3-4b", 64, 40, 161, 48),
        # a checkpoint is checked in 32 bits: prompts and a few tokens
        case("f32 check", "gemma3-medium-f32", 3, 97, 421, 12),
        # the other designs: a long prompt, and a batch that decodes
        case("batasun prompt 3001", "batasun-medium", 1, 3001, 3001, 0),
        case("batasun decode b6", "batasun-medium", 6, 130, 1030, 64),
        case("derosun serve b4", "derosun-medium", 4, 300, 1900, 48),
    ]


def _between(rng, lo, hi):
    """A whole number from lo to hi, even over the logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """A request or a batch of the same kinds: single prompts, batches of unequal prompts, batches that decode."""
    model = rng.choice(["gemma3-4b", "gemma3-4b", "gemma3-4b", "gemma3-medium-f32", "batasun-medium", "derosun-medium"])
    most, slots = {"gemma3-4b": (10000, 64), "gemma3-medium-f32": (700, 8), "batasun-medium": (6000, 32), "derosun-medium": (6000, 32)}[model]
    kind = rng.choice(["prompt", "batch", "decode"])
    if kind == "prompt":
        n = _between(rng, 5, most)
        return {"model": model, "batch": 1, "shortest": n, "longest": n, "steps": 0}
    batch = _between(rng, 2 if kind == "batch" else 1, 8 if kind == "batch" else slots)
    longest = _between(rng, 16, min(most, max(32, (most if model == "gemma3-medium-f32" else 9000) // batch)))
    shortest = _between(rng, max(2, longest // 16), longest)
    return {"model": model, "batch": batch, "shortest": shortest, "longest": longest,
            "steps": 0 if kind == "batch" else _between(rng, 8, 16 if model == "gemma3-medium-f32" else 64)}


def _lengths(case):
    b, lo, hi = int(case["batch"]), int(case["shortest"]), int(case["longest"])
    return [hi] if b == 1 else [lo + (hi - lo) * i // (b - 1) for i in range(b)]


# ---------------------------------------------------------------- weights
def _gemma_shapes(c):
    e, hd, ff = c["hidden_size"], c["head_dim"], c["intermediate_size"]
    qd, kvd = c["num_attention_heads"] * hd, c["num_key_value_heads"] * hd
    out = {"model.embed_tokens.weight": (c["vocab_size"], e), "model.norm.weight": (e,)}
    for i in range(c["num_hidden_layers"]):
        p = f"model.layers.{i}."
        out.update({p + "input_layernorm.weight": (e,), p + "post_attention_layernorm.weight": (e,),
                    p + "pre_feedforward_layernorm.weight": (e,), p + "post_feedforward_layernorm.weight": (e,),
                    p + "self_attn.q_proj.weight": (qd, e), p + "self_attn.k_proj.weight": (kvd, e), p + "self_attn.v_proj.weight": (kvd, e),
                    p + "self_attn.q_norm.weight": (hd,), p + "self_attn.k_norm.weight": (hd,), p + "self_attn.o_proj.weight": (e, qd),
                    p + "mlp.gate_proj.weight": (ff, e), p + "mlp.up_proj.weight": (ff, e), p + "mlp.down_proj.weight": (e, ff)})
    if not c["tie_word_embeddings"]:
        out["lm_head.weight"] = (c["vocab_size"], e)
    return out


def _design_shapes(c):
    e, out = c["width"], {"embed": (c["vocab"], c["width"])}
    if c["architecture"] == "Batasun":
        out["embed.norm"] = (e,)
    for i, layer in enumerate(c["layers"]):
        p, x, m, f = f"l{i}.", f"l{i}.mix.", layer["mixer"], layer["mlp"]
        H = m["heads"]
        out[p + "norm1"], out[p + "norm2"] = (e,), (e,)
        if layer["type"] == "attention":
            G = m["kv_heads"]
            out.update({x + "q": (H * m["dim"], e), x + "k": (G * m["dim"], e), x + "v": (G * m["vdim"], e),
                        x + "q.norm": (H * m["dim"],), x + "k.norm": (G * m["dim"],)})
        elif layer["type"] == "latent_attention":
            out.update({x + "dq": (m["q_rank"], e), x + "dq.norm": (m["q_rank"],), x + "uq": (H * (m["dim"] + m["rot_dim"]), m["q_rank"]),
                        x + "uk": (H * m["dim"], m["kv_rank"]), x + "uv": (H * m["vdim"], m["kv_rank"])})
            if m.get("kv_from") is None:
                out.update({x + "dkv": (m["kv_rank"] + m["rot_dim"], e), x + "dkv.norm": (m["kv_rank"],)})
            if c["architecture"] == "Batasun":
                out[x + "g"] = (H * m["vdim"], e)
        elif layer["type"] == "mamba2":
            inner, gn = H * m["vdim"], m["groups"] * m["state"]
            out.update({x + "in": (2 * inner + 2 * gn + H, e), x + "conv": (inner + 2 * gn, m["conv"]), x + "conv.b": (inner + 2 * gn,),
                        x + "dt_bias": (H,), x + "A_log": (H,), x + "D": (H,), x + "norm": (inner,)})
        else:
            out.update({x + "q": (H * m["dim"], e), x + "k": (H * m["dim"], e), x + "v": (H * m["vdim"], e), x + "g": (H * m["vdim"], e),
                        x + "norm": (H * m["vdim"],), x + "i": (H, e), x + "i.b": (H,), x + "f": (H, e), x + "f.b": (H,)})
        out[x + "o"] = (e, H * m["vdim"])
        if f["kind"] == "dense":
            for n, shape in (("gate", (f["ff"], e)), ("up", (f["ff"], e)), ("down", (e, f["ff"]))):
                out[p + "mlp." + n], out[p + "mlp." + n + ".b"] = shape, shape[:1]
        else:
            for q in [f"{p}mlp.e{k}." for k in range(f["router"]["experts"])] + [p + "mlp.shared."]:
                ff = f["expert"]["ff"] if ".e" in q else f["shared"]["ff"]
                out.update({q + "gate": (ff, e), q + "up": (ff, e), q + "down": (e, ff)})
            out.update({p + "mlp.router": (f["router"]["experts"], e), p + "mlp.router.b": (f["router"]["experts"],), p + "mlp.shared.sg": (1, e)})
    out["final.norm"], out["head"] = (e,), (c["vocab"], e)
    return out


def _spread(name, shape, design):
    """(mean, standard deviation) of a tensor's values; ``design``: the architecture where it is not Gemma 3."""
    last = name.rsplit(".", 1)[-1]
    if not design:
        return (0.0, 0.1) if len(shape) == 1 else (0.0, 0.02)
    if name == "embed":
        return 0.0, 1.0
    if last == "conv":
        return 0.0, 0.5
    if len(shape) == 2:
        return 0.0, shape[1] ** -0.5
    if last in ("dt_bias", "A_log", "D"):
        return {"dt_bias": (-2.0, 0.7), "A_log": (-0.3, 0.7), "D": (1.0, 0.5)}[last]
    if last == "b":
        return (3.0, 2.0) if name.endswith("mix.f.b") else (0.0, 1.0) if name.endswith("mix.i.b") else (0.0, 0.2)
    # norms: Batasun stores a layer's and the model's around zero (they act as 1 + w), all others around one
    return (0.0 if design == "Batasun" and ".mix." not in name else 1.0), 0.1


def _weights(model):
    """The model's tensors on the GPU, in bfloat16 values (the 32-bit engine reads the same numbers)."""
    config, dtype = MODELS[model][:2]
    design = config.get("architecture", "")
    shapes = _design_shapes(config) if design else _gemma_shapes(config)
    g = torch.Generator(device="cuda").manual_seed(20240)
    out = {}
    for name, shape in shapes.items():
        mean, std = _spread(name, shape, design)
        out[name] = torch.empty(shape, dtype=torch.bfloat16, device="cuda").normal_(mean, std, generator=g)
    for i, layer in enumerate(config.get("layers", [])):
        if layer["type"] == "mlstm":        # a read-out is normed, so queries that have nothing of the keys would be all rounding
            p = f"l{i}.mix."
            out[p + "q"] = (0.9 * out[p + "k"].float() + 0.45 * out[p + "q"].float()).bfloat16()
        if layer["mlp"]["kind"] == "moe":
            _clear_choice(out, f"l{i}.", layer["mlp"]["router"], g)
    return {k: v.float() for k, v in out.items()} if dtype == "float32" else out


def _clear_choice(out, p, router, g):
    """Routers that are as sure as trained ones: every token's embedding says, in one element per expert, which experts it is
    for (as many tokens for each), no sublayer writes to these elements, and a router reads little else.  With plain noise in
    their place a choice hangs on rounding for every thirtieth token and layer, and no two implementations would agree."""
    n, top = router["experts"], router["top"]
    for norm in ("norm1", "norm2"):
        out[p + norm][:n] = -1.0                     # (these norms act as 1 + w)
    out[p + "mlp.router"] *= 0.3
    out[p + "mlp.router"][:, :n] = torch.eye(n, device="cuda", dtype=torch.bfloat16)
    if p == "l0.":
        out["embed.norm"][:n] = 0.0
        chosen = torch.rand(out["embed"].shape[0], n, device="cuda", generator=g).argsort(-1).argsort(-1) < top
        out["embed"][:, :n] = torch.where(chosen, 6.0, -6.0).bfloat16()


_kept = {}          # the engine of the model that was asked for last


def _engine(model):
    if model not in _kept:
        from agave_amd.engine import Engine
        _kept.clear()
        torch.cuda.empty_cache()
        config, dtype, slots, context, held = MODELS[model]
        _kept[model] = Engine.from_tensors(config, _weights(model), dtype=dtype, max_slots=slots, max_context=context, cache_tokens=held,
                                           device="cuda:0")
    return _kept[model]


# ---------------------------------------------------------------- a pass
def _tokens(case, seed):
    """Every sequence's tokens: its prompt and the ``steps`` that follow."""
    config = MODELS[case["model"]][0]
    vocab = config.get("vocab_size") or config["vocab"]
    g = torch.Generator().manual_seed(int(seed))
    return [torch.randint(0, vocab, (n + int(case["steps"]),), generator=g).tolist() for n in _lengths(case)]


def prepare(case, seed):
    tokens, lengths, steps = _tokens(case, seed), _lengths(case), int(case["steps"])
    return {"engine": _engine(case["model"]), "prompts": [t[:n] for t, n in zip(tokens, lengths)],
            "following": [[[t[n + s]] for t, n in zip(tokens, lengths)] for s in range(steps)]}


def run(state):
    engine, following = state["engine"], state["following"]
    slots = [engine.alloc_slot() for _ in state["prompts"]]
    try:
        first = engine.step(slots, state["prompts"], "last").clone()        # (a step's logits last until the next one)
        last = first
        for tokens in following:
            last = engine.step(slots, tokens, "last")
        return {"prompt": first, "last": last.clone()} if following else {"prompt": first}
    finally:
        for s in slots:
            engine.free_slot(s)


# ---------------------------------------------------------------- what a pass cannot do without
def _layer_costs(config):
    """Per layer: (multiply-adds of its matrices per token, bytes of all its weights per element's byte, keys a token can see,
    numbers cached per position, multiply-adds per visible key, numbers of fixed state per sequence)."""
    if "layers" not in config:
        e, hd, ff = config["hidden_size"], config["head_dim"], config["intermediate_size"]
        qd, kvd = config["num_attention_heads"] * hd, config["num_key_value_heads"] * hd
        n = e * (2 * qd + 2 * kvd) + 3 * e * ff
        return [(n, n, config["sliding_window"] if (i + 1) % config["sliding_window_pattern"] else None, 2 * kvd, 2 * qd, 0)
                for i in range(config["num_hidden_layers"])]
    out, shapes = [], _design_shapes(config)
    for i, layer in enumerate(config["layers"]):
        sizes = {k: math.prod(s) for k, s in shapes.items() if k.startswith(f"l{i}.") and len(s) == 2}
        held, m, f = sum(sizes.values()), layer["mixer"], layer["mlp"]
        used = held
        if f["kind"] == "moe":
            experts = sum(v for k, v in sizes.items() if ".mlp.e" in k)
            used = held - experts + experts * f["router"]["top"] // f["router"]["experts"]
        if layer["type"] == "attention":
            out.append((used, held, None, m["kv_heads"] * (m["dim"] + m["vdim"]), m["heads"] * (m["dim"] + m["vdim"]), 0))
        elif layer["type"] == "latent_attention":
            out.append((used, held, None, m["kv_rank"] + m["rot_dim"], m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"]), 0))
        else:
            state = m["heads"] * m["vdim"] * (m["state"] if layer["type"] == "mamba2" else m["dim"])
            out.append((used + 2 * state, held, 0, 0, 0, state))
    return out


def work(case):
    config, dtype = MODELS[case["model"]][:2]
    size = 4 if dtype == "float32" else 2
    e, vocab = config.get("hidden_size") or config["width"], config.get("vocab_size") or config["vocab"]
    layers, lengths, steps = _layer_costs(config), _lengths(case), int(case["steps"])
    total, b = sum(lengths), len(lengths)
    flops = 2.0 * sum(x[0] for x in layers) * (total + b * steps) + 2.0 * vocab * e * b * (1 + steps)
    nbytes = float(size * vocab * e + size * e * total) + 8.0 * vocab * b          # the output matrix, the tokens' rows, the logits
    for used, held, reach, cached, per_key, state in layers:
        # (of the experts no more is needed than the tokens choose: all of them as soon as there are a few)
        share = min(1.0, used * total / held) if used < held else 1.0
        nbytes += size * held * share + size * cached * total + 4.0 * state * b
        for n in lengths:
            if reach != 0:
                seen = n * (n + 1) / 2 if reach is None or n <= reach else reach * (reach + 1) / 2 + (n - reach) * reach
                flops += 2.0 * per_key * seen
        for s in range(steps):
            share = min(1.0, used * b / held) if used < held else 1.0
            keys = sum(min(n + s + 1, reach) if reach else n + s + 1 for n in lengths) if reach != 0 else 0
            nbytes += size * held * share + size * cached * keys + 8.0 * state * b
            flops += 2.0 * per_key * keys
    nbytes += steps * (size * vocab * e)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times what the engine's logits are off those of :func:`exact`; bfloat16 rounds every sublayer's input, and
    the error grows with the number of layers."""
    return {"gemma3-4b": {"rel": 0.03, "max": 0.2}, "gemma3-medium-f32": {"rel": 1.2e-5, "max": 1e-4},
            "batasun-medium": {"rel": 0.03, "max": 0.2}, "derosun-medium": {"rel": 0.015, "max": 0.1}}[case["model"]]


# ---------------------------------------------------------------- the same in 64 bits
def _rms(x, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _turn(x, freq, neighbours=False, magnitude=1.0):
    """x [B, T, heads, n]: position t's first 2 len(freq) elements turn by t * freq, in pairs of halves or of neighbours."""
    n = len(freq)
    a = torch.arange(x.shape[1], dtype=F, device=x.device)[:, None, None] * torch.tensor(freq, dtype=F, device=x.device)
    c, s = torch.cos(a) * magnitude, torch.sin(a) * magnitude
    u, v = (x[..., 0:2 * n:2], x[..., 1:2 * n:2]) if neighbours else (x[..., :n], x[..., n:2 * n])
    u, v = u * c - v * s, v * c + u * s
    return torch.cat([torch.stack([u, v], -1).flatten(-2) if neighbours else torch.cat([u, v], -1), x[..., 2 * n:]], -1)


def _attend(q, k, v, scale, window=None, cap=None):
    """q [B, T, H, d], k and v [B, T, G, .]: softmax over the positions up to the query's own (and within the window)."""
    B, T, H, _ = q.shape
    at = torch.arange(T, device=q.device)
    hidden = at[None, :] > at[:, None]
    if window is not None:
        hidden = hidden | (at[None, :] < at[:, None] - window + 1)
    out = torch.empty(B, T, H, v.shape[-1], dtype=F, device=q.device)
    for b in range(B):
        for h in range(H):
            g = h // (H // k.shape[2])
            s = (q[b, :, h] @ k[b, :, g].T) * scale
            s = cap * torch.tanh(s / cap) if cap is not None else s
            out[b, :, h] = torch.softmax(s.masked_fill_(hidden, -math.inf), -1) @ v[b, :, g]
    return out.flatten(2)


def _exact_gemma(c, w, ids):
    e, hd, eps = c["hidden_size"], c["head_dim"], c["rms_norm_eps"]
    H, G, B, T = c["num_attention_heads"], c["num_key_value_heads"], *ids.shape
    x = w("model.embed_tokens.weight", ids) * math.sqrt(e)
    for i in range(c["num_hidden_layers"]):
        p = f"model.layers.{i}."
        local = (i + 1) % c["sliding_window_pattern"] != 0
        base, factor = (c["rope_local_base_freq"], 1.0) if local else (c["rope_theta"], c["rope_scaling"]["factor"])
        freq = [base ** (-2.0 * j / hd) / factor for j in range(hd // 2)]
        n = _rms(x, eps) * (1 + w(p + "input_layernorm.weight"))
        q = _rms((n @ w(p + "self_attn.q_proj.weight").T).view(B, T, H, hd), eps) * (1 + w(p + "self_attn.q_norm.weight"))
        k = _rms((n @ w(p + "self_attn.k_proj.weight").T).view(B, T, G, hd), eps) * (1 + w(p + "self_attn.k_norm.weight"))
        v = (n @ w(p + "self_attn.v_proj.weight").T).view(B, T, G, hd)
        a = _attend(_turn(q, freq), _turn(k, freq), v, c["query_pre_attn_scalar"] ** -0.5, c["sliding_window"] if local else None)
        x = x + _rms(a @ w(p + "self_attn.o_proj.weight").T, eps) * (1 + w(p + "post_attention_layernorm.weight"))
        n = _rms(x, eps) * (1 + w(p + "pre_feedforward_layernorm.weight"))
        f = torch.nn.functional.gelu(n @ w(p + "mlp.gate_proj.weight").T, approximate="tanh") * (n @ w(p + "mlp.up_proj.weight").T)
        x = x + _rms(f @ w(p + "mlp.down_proj.weight").T, eps) * (1 + w(p + "post_feedforward_layernorm.weight"))
    return _rms(x, eps) * (1 + w("model.norm.weight")), "model.embed_tokens.weight" if c["tie_word_embeddings"] else "lm_head.weight"


def _frequencies(rot):
    """(the rotation's frequencies, the factor on sine and cosine)."""
    d, s = rot["dims"], rot.get("scaling")
    plain = [rot["base"] ** (-2.0 * j / d) for j in range(d // 2)]
    if s is None:
        return plain, 1.0
    if "fast" in s:                                  # YaRN: blended by how often a pair turns within the original context
        def where(turns):
            return d * math.log(s["original"] / (2 * math.pi * turns)) / (2 * math.log(rot["base"]))
        lo, hi = max(math.floor(where(s["fast"])), 0), min(math.ceil(where(s["slow"])), d - 1)
        ramp = [min(max((j - lo) / max(hi - lo, 0.001), 0.0), 1.0) for j in range(d // 2)]
        return [f / s["factor"] * r + f * (1 - r) for f, r in zip(plain, ramp)], 0.1 * math.log(s["factor"]) + 1.0
    out = []
    for f in plain:                                  # blended by wavelength
        t = (s["original"] * f / (2 * math.pi) - s["low"]) / (s["high"] - s["low"])
        out.append(f if t > 1 else f / s["factor"] if t < 0 else (1 - t) * f / s["factor"] + t * f)
    return out, 1.0


def _latent(m, w, p, x, eps, rows, neighbours):
    B, T, _ = x.shape
    H, d, rd = m["heads"], m["dim"], m["rot_dim"]
    freq, magnitude = _frequencies(m["rot"])
    q = ((_rms(x @ w(p + "dq").T, eps) * w(p + "dq.norm")) @ w(p + "uq").T).view(B, T, H, d + rd)
    q = torch.cat([q[..., :d], _turn(q[..., d:], freq, neighbours, magnitude)], -1)
    if rows is None:
        raw = x @ w(p + "dkv").T
        rows = _rms(raw[..., :m["kv_rank"]], eps) * w(p + "dkv.norm"), _turn(raw[..., None, m["kv_rank"]:], freq, neighbours, magnitude)
    c, r = rows
    k = torch.cat([(c @ w(p + "uk").T).view(B, T, H, d), r.expand(B, T, H, rd)], -1)
    return _attend(q, k, (c @ w(p + "uv").T).view(B, T, H, m["vdim"]), m["scale"]), rows


def _lower(T, device):
    return torch.ones(T, T, dtype=torch.bool, device=device).tril()


def _mamba2(m, w, p, x, eps):
    B, T, _ = x.shape
    H, P, N = m["heads"], m["vdim"], m["state"]
    inner = H * P
    proj = x @ w(p + "in").T
    z, u, dt = proj[..., :inner], proj[..., inner:2 * inner + 2 * N], proj[..., 2 * inner + 2 * N:]
    taps = w(p + "conv")
    padded = torch.nn.functional.pad(u, (0, 0, taps.shape[1] - 1, 0))
    u = torch.nn.functional.silu(sum(padded[:, j:j + T] * taps[:, j] for j in range(taps.shape[1])) + w(p + "conv.b"))
    dt = torch.nn.functional.softplus(dt + w(p + "dt_bias"), threshold=1e9)
    since = torch.cumsum(-torch.exp(w(p + "A_log")) * dt, 1)                        # the logarithm of what is left of the start
    y = torch.empty(B, T, H, P, dtype=F, device=x.device)
    for b in range(B):
        xs, scores = u[b, :, :inner].view(T, H, P), u[b, :, inner + N:] @ u[b, :, inner:inner + N].T
        for h in range(H):
            left = torch.exp((since[b, :, h, None] - since[b, None, :, h]).masked_fill_(~_lower(T, x.device), -math.inf))
            y[b, :, h] = (scores * left * dt[b, None, :, h]) @ xs[:, h] + w(p + "D")[h] * xs[:, h]
    return _rms(y.flatten(2) * torch.nn.functional.silu(z), eps) * w(p + "norm")


def _mlstm(m, w, p, x, eps):
    B, T, _ = x.shape
    H, d, vd, cap = m["heads"], m["dim"], m["vdim"], m["gate_cap"]
    q, k = (x @ w(p + "q").T).view(B, T, H, d) * d ** -0.5, (x @ w(p + "k").T).view(B, T, H, d)
    v = (x @ w(p + "v").T).view(B, T, H, vd)
    i = cap * torch.tanh((x @ w(p + "i").T + w(p + "i.b")) / cap)
    since = torch.cumsum(torch.nn.functional.logsigmoid(cap * torch.tanh((x @ w(p + "f").T + w(p + "f.b")) / cap)), 1)
    o = torch.empty(B, T, H, vd, dtype=F, device=x.device)
    for b in range(B):
        for h in range(H):
            logs = (since[b, :, h, None] - since[b, None, :, h] + i[b, None, :, h]).masked_fill_(~_lower(T, x.device), -math.inf)
            most = torch.maximum(logs.amax(-1), since[b, :, h])                     # the running maximum starts at 0
            s = torch.exp(logs - most[:, None]) * (q[b, :, h] @ k[b, :, h].T)
            o[b, :, h] = (s @ v[b, :, h]) / (torch.maximum(s.sum(-1).abs(), torch.exp(-most)) + 1e-6)[:, None]
    return _rms(o, eps).flatten(2) * w(p + "norm") * torch.sigmoid(x @ w(p + "g").T)


def _routed(f, w, p, x):
    def expert(q, y, limit):
        g, u = torch.clamp(y @ w(q + "gate").T, max=limit), torch.clamp(y @ w(q + "up").T, -limit, limit)
        return (g * torch.sigmoid(1.702 * g) * (u + 1)) @ w(q + "down").T
    logits, choice = torch.topk(x @ w(p + "router").T + w(p + "router.b"), f["router"]["top"], dim=-1)
    weight = torch.softmax(logits, -1)
    out = torch.sigmoid(x @ w(p + "shared.sg").T) * expert(p + "shared.", x, f["shared"]["limit"])
    for k in range(f["router"]["experts"]):
        chosen = (choice == k)
        rows = chosen.any(-1)
        out[rows] += (weight * chosen).sum(-1)[rows][:, None] * expert(f"{p}e{k}.", x[rows], f["expert"]["limit"])
    return out


def _exact_design(c, w, ids):
    eps, batasun, rows_of = c["norm"]["eps"], c["architecture"] == "Batasun", {}
    x = w("embed", ids)
    x = _rms(x, eps) * (1 + w("embed.norm")) if batasun else x * c["embedding"]["scale"]
    for i, layer in enumerate(c["layers"]):
        p, m = f"l{i}.mix.", layer["mixer"]
        if layer["type"] == "latent_attention":
            a, rows_of[i] = _latent(m, w, p, x, eps, rows_of.get(m.get("kv_from")), neighbours=not batasun)
            a = a * torch.sigmoid(x @ w(p + "g").T) if batasun else a
        elif layer["type"] == "mamba2":
            a = _mamba2(m, w, p, x, eps)
        elif layer["type"] == "mlstm":
            a = _mlstm(m, w, p, x, eps)
        else:
            B, T, _ = x.shape
            freq, _ = _frequencies(m["rot"])
            q = (_rms(x @ w(p + "q").T, eps) * w(p + "q.norm")).view(B, T, m["heads"], m["dim"])
            k = (_rms(x @ w(p + "k").T, eps) * w(p + "k.norm")).view(B, T, m["kv_heads"], m["dim"])
            v = (x @ w(p + "v").T).view(B, T, m["kv_heads"], m["vdim"])
            a = _attend(_turn(q, freq), _turn(k, freq), v, m["scale"], cap=m["softcap"])
        a = a @ w(p + "o").T
        p, f = f"l{i}.mlp.", layer["mlp"]
        if batasun:
            x = x + _rms(a, eps) * (1 + w(f"l{i}.norm1"))
            x = x + _rms(_routed(f, w, p, x), eps) * (1 + w(f"l{i}.norm2"))
        else:
            x = _rms(c["postln_alpha"] * x + a, eps) * w(f"l{i}.norm1")
            g, u = x @ w(p + "gate").T + w(p + "gate.b"), x @ w(p + "up").T + w(p + "up.b")
            x = _rms(c["postln_alpha"] * x + (g * torch.sigmoid(g) * u) @ w(p + "down").T + w(p + "down.b"), eps) * w(f"l{i}.norm2")
    return _rms(x, eps) * (w("final.norm") + (1 if batasun else 0)), "head"


def exact(case, seed):
    config = MODELS[case["model"]][0]
    _kept.clear()                                   # (room)
    tensors, tokens, lengths, steps = _weights(case["model"]), _tokens(case, seed), _lengths(case), int(case["steps"])

    def w(name, rows=None):
        return (tensors[name] if rows is None else tensors[name][rows]).double()
    # sequences of about one length go together; those that are shorter are filled up behind their end, where nothing looks
    order, groups = sorted(range(len(tokens)), key=lambda i: len(tokens[i])), []
    for i in order:
        if groups and len(groups[-1]) < 8 and len(tokens[i]) <= 2 * len(tokens[groups[-1][0]]) + 64:
            groups[-1].append(i)
        else:
            groups.append([i])
    first, last = [None] * len(tokens), [None] * len(tokens)
    for group in groups:
        T = max(len(tokens[i]) for i in group)
        ids = torch.tensor([tokens[i] + [0] * (T - len(tokens[i])) for i in group], device="cuda")
        x, head = (_exact_design if "layers" in config else _exact_gemma)(config, w, ids)
        for j, i in enumerate(group):
            first[i], last[i] = x[j, lengths[i] - 1], x[j, lengths[i] + steps - 1]
    matrix = w(head)
    out = {"prompt": torch.stack(first) @ matrix.T}
    if steps:
        out["last"] = torch.stack(last) @ matrix.T
    return out
