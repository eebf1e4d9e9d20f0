"""The work whose speed counts: cases of the engine's step function at the sizes its users run it.

A case is a dict of plain values.  Its `kind` says which direction of serving it is:
  decode  a batch of requests in mid-generation takes one token each, or several one after the other (the requests are taken
          back to their lengths afterwards, so that a pass can be repeated);
  prompt  prompts arrive, run in one step from an empty cache to the logits of their last rows (one for the next token,
          several where an answer's tokens are scored), and end;
  mixed   decoding requests take a token each beside a portion of a prompt that arrives: what a scheduler issues;
  score   a text's logits at every position, as perplexity reads them;
  replay  one request from its prompt through a few decoded tokens to its end: for models that keep a state a request,
          which cannot be taken back.
Its `model` names the sizes: "m3" MiniMax-M3's real layer sizes with four layers (the benchmark's configuration has 24 of
them, all alike), "m3_w2048", "bonerax" and "nenotar" the design bench's width of 2,048 ("bonerax" with dense feed-forwards:
attention beside a small delta rule, and a delta rule alone, in turn), "m3_w256" its smallest.
Weights are random (N(0, 0.02), norms and biases spread about their usual values), token ids uniform.
"""

from __future__ import annotations

import math

import numpy as np
import torch

DTYPES = {"bf16": "bfloat16", "f32": "float32"}
PORTION = 2048              # a prompt's context comes into the cache in portions of this many tokens
WARM_STEPS = 3              # decode steps a request in mid-generation has behind it


# ---------------------------------------------------------------------------------------------------------------- cases
def listed():
    return [
        # one chat turn on a small model: nothing but latency and launches
        {"name": "tiny_decode", "kind": "decode", "model": "m3_w256", "dtype": "bf16", "batch": 1, "context": 40, "steps": 1},
        # a single user of the real sizes: a sentence of an answer
        {"name": "decode_1", "kind": "decode", "model": "m3", "dtype": "bf16", "batch": 1, "context": 4096, "steps": 16},
        # the benchmark's default batch, contexts of unequal and odd length about its 4,096 tokens
        {"name": "decode_8", "kind": "decode", "model": "m3", "dtype": "bf16", "batch": 8, "context": 4096, "steps": 2},
        # a full server of short conversations
        {"name": "decode_64", "kind": "decode", "model": "m3", "dtype": "bf16", "batch": 64, "context": 1280, "steps": 1},
        # two long documents being continued
        {"name": "decode_long", "kind": "decode", "model": "m3", "dtype": "bf16", "batch": 2, "context": 20011, "steps": 8},
        # one prompt of the benchmark's length, whose last 16 tokens are an answer to be scored
        {"name": "prompt_2048", "kind": "prompt", "model": "m3", "dtype": "bf16", "prompts": 1, "tokens": 2048, "want": 16},
        # many short prompts at once, of unequal and odd length: their rows pick most of the experts in every layer
        {"name": "prompts_short", "kind": "prompt", "model": "m3", "dtype": "bf16", "prompts": 37, "tokens": 45, "want": 1},
        # a portion of a prompt that arrives while eight requests decode
        {"name": "mixed_512", "kind": "mixed", "model": "m3", "dtype": "bf16", "batch": 8, "context": 1500, "tokens": 512},
        # a text scored in 32 bits: perplexity, and the reference a served model is compared with
        {"name": "score_f32", "kind": "score", "model": "m3_w2048", "dtype": "f32", "tokens": 333},
        # and generation in 32 bits
        {"name": "decode_f32", "kind": "decode", "model": "m3_w2048", "dtype": "f32", "batch": 4, "context": 600, "steps": 1},
        # matrix-state recurrences beside attention: a prompt, then a few tokens
        {"name": "bonerax_replay", "kind": "replay", "model": "bonerax", "dtype": "bf16", "tokens": 1999, "decoded": 6},
        # latent attention and a vector recurrence: a prompt, then a few tokens
        {"name": "nenotar_replay", "kind": "replay", "model": "nenotar", "dtype": "bf16", "tokens": 2048, "decoded": 6},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the same ranges: batches of 1 to 64, contexts of 32 to 24,576 tokens (81,920 in all at most),
    prompts of 16 to 2,048 tokens, alone or many at once (2,048 rows at most), portions of 16 to 1,024."""
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "mixed", "score", "f32", "replay"])
    if kind == "decode":
        batch = _log(rng, 1, 64)
        model = rng.choice(["m3", "m3", "m3_w256"])
        return {"kind": "decode", "model": model, "dtype": "bf16", "batch": batch, "steps": -(-16 // batch),
                "context": _log(rng, 32, min(24576 if model == "m3" else 4096, 81920 // batch))}
    if kind == "prompt":
        prompts = _log(rng, 1, 48)
        return {"kind": "prompt", "model": "m3", "dtype": "bf16", "prompts": prompts, "tokens": _log(rng, 16, 2048 // prompts), "want": -(-16 // prompts)}
    if kind == "mixed":
        return {"kind": "mixed", "model": "m3", "dtype": "bf16", "batch": _log(rng, 1, 32), "context": _log(rng, 32, 4096),
                "tokens": _log(rng, 16, 1024)}
    if kind == "score":
        return {"kind": "score", "model": "m3_w2048", "dtype": "f32", "tokens": _log(rng, 16, 333)}
    if kind == "f32":
        return {"kind": "decode", "model": "m3_w2048", "dtype": "f32", "batch": _log(rng, 1, 8), "context": _log(rng, 32, 1024), "steps": 1}
    return {"kind": "replay", "model": rng.choice(["bonerax", "nenotar"]), "dtype": "bf16", "tokens": _log(rng, 16, 2048),
            "decoded": rng.randint(1, 8)}


# --------------------------------------------------------------------------------------------------------------- models
def _m3(hidden, layers, heads, kv_heads, experts, top, inter, vocab, positions, theta):
    from llmx_amd import MiniMaxM3Config
    return MiniMaxM3Config(vocab_size=vocab, hidden_size=hidden, num_hidden_layers=layers, num_attention_heads=heads, num_key_value_heads=kv_heads,
                           head_dim=128, rotary_dim=64, rope_theta=theta, rms_norm_eps=1e-6, num_local_experts=experts, num_experts_per_tok=top,
                           intermediate_size=inter, routed_scaling_factor=1.0, norm_topk_prob=True, tie_word_embeddings=False,
                           max_position_embeddings=positions)


def _config(case):
    from llmx_amd.tools import design_bench
    model = case["model"]
    if model == "m3":
        return _m3(3072, 4, 48, 8, 256, 8, 1536, 200064, 65536, 5e6)
    if model == "m3_w2048":
        return _m3(2048, 8, 16, 4, 8, 2, 2688, 32768, 8192, 1e6)
    if model == "m3_w256":
        return _m3(256, 2, 2, 1, 8, 2, 256, 1024, 8192, 1e6)
    if model == "bonerax":
        return design_bench.vivulorn_bonerax(*design_bench.VIVULORN_SIZES["w2048"])
    return design_bench.nenotar_config(*design_bench.SIZES["w2048"])


def _vocab(cfg):
    return cfg.vocab_size if hasattr(cfg, "vocab_size") else cfg.vocab


def _lengths(case):
    """Tokens of each request before the pass (decode, mixed) or of each prompt: about the case's figure, unequal where
    there are several."""
    if case["kind"] == "prompt":
        n, about = case["prompts"], case["tokens"]
    else:
        n, about = case.get("batch", 0), case.get("context", 0)
    if n <= 2:
        return [about] * n
    return [max(1, int(round(about * f))) for f in np.random.default_rng([n, about]).uniform(0.6, 1.4, n)]


def _tokens(case, seed):
    """The case's token ids: the requests' texts before the pass, the tokens decoded in it, and the prompt or text of it."""
    rng = np.random.default_rng([seed, 20])
    vocab = _vocab(_config(case))
    ids = lambda n: rng.integers(0, vocab, n).tolist()
    texts = [ids(max(n, WARM_STEPS + 1)) for n in _lengths(case)]
    return {"texts": texts, "next": [ids(case.get("steps", 1)) for _ in texts], "text": ids(case["tokens"]) if case["kind"] in ("mixed", "score", "replay") else [],
            "decoded": ids(case.get("decoded", 0))}


def _last(text, case):
    return list(range(max(0, len(text) - case["want"]), len(text)))


def _engine(case, seed, tokens_out=None, kv_tokens=16, requests=1):
    from llmx_amd import Engine, RandomInit
    return Engine.from_random(_config(case), RandomInit(seed=seed, std=0.02, norm_std=0.05, bias_range=0.02), dtype=DTYPES[case["dtype"]],
                              tensors_out=tokens_out, kv_tokens=kv_tokens, page_tokens=16, max_requests=requests)


# ----------------------------------------------------------------------------------------------------------- the passes
def prepare(case, seed):
    """An engine with its weights; for decode and mixed cases requests in mid-generation: their prompts run, their last
    tokens before the pass decoded one by one."""
    from llmx_amd import StepEntry
    t = _tokens(case, seed)
    requests = len(t["texts"]) + 1
    total = sum(len(x) for x in t["texts"]) + (16 + case.get("steps", 1)) * requests + len(t["text"]) + len(t["decoded"]) + 16
    engine = _engine(case, seed, kv_tokens=total, requests=requests)
    if case["kind"] in ("decode", "mixed"):
        for i, text in enumerate(t["texts"]):
            engine.add_request(i)
            known = text[:-WARM_STEPS]
            for s in range(0, len(known), PORTION):
                engine.step([StepEntry(i, known[s:s + PORTION], [])])
        for j in range(-WARM_STEPS, 0):
            engine.step([StepEntry(i, [text[j]], [0]) for i, text in enumerate(t["texts"])])
    return {"case": case, "engine": engine, "tokens": t}


def run(state):
    from llmx_amd import StepEntry
    case, engine, t = state["case"], state["engine"], state["tokens"]
    kind, texts = case["kind"], t["texts"]
    if kind == "decode":
        out = torch.empty(case["steps"], len(texts), engine.vocab_size, device=engine.device) if case["steps"] > 1 else None
        for j in range(case["steps"]):
            logits = engine.step([StepEntry(i, [tokens[j]], [0]) for i, tokens in enumerate(t["next"])])
            if out is not None:
                out[j] = logits
        for i, text in enumerate(texts):
            engine.truncate(i, len(text))
        return logits if out is None else out
    if kind == "mixed":
        engine.add_request("new")
        logits = engine.step([StepEntry(i, tokens, [0]) for i, tokens in enumerate(t["next"])]
                             + [StepEntry("new", t["text"], [len(t["text"]) - 1])])
        engine.end_request("new")
        for i, text in enumerate(texts):
            engine.truncate(i, len(text))
        return logits
    if kind == "prompt":
        for i in range(len(texts)):
            engine.add_request(i)
        logits = engine.step([StepEntry(i, text, _last(text, case)) for i, text in enumerate(texts)])
        for i in range(len(texts)):
            engine.end_request(i)
        return logits
    engine.add_request("text")
    if kind == "score":
        rows = engine.score("text", t["text"])
    else:
        out = [engine.prefill("text", t["text"], portion=PORTION).clone()]
        for token in t["decoded"]:
            out.append(engine.decode_one("text", token).clone())
        rows = torch.stack(out)
    engine.end_request("text")
    return rows


# ------------------------------------------------------------------------------------------------------- what it needs
def _m3_work(cfg, wb, rows, keys, wants, kv_read, apart):
    """`rows` rows through the layers, `keys` (row, key) pairs, `wants` rows of logits, `kv_read` cached tokens read.  Rows of
    different requests (`apart`) pick experts independently.  Rows of one text grow alike in a model with random weights:
    from the third layer on they pick about 55 of 256 experts, as measured."""
    E, q, kv, X, k = cfg.hidden_size, cfg.num_attention_heads * cfg.head_dim, cfg.num_key_value_heads * cfg.head_dim, cfg.num_local_experts, cfg.num_experts_per_tok
    attention, expert = E * (q + 2 * kv) + q * E, 3 * E * cfg.intermediate_size
    bytes_ = flops = 0.0
    for layer in range(cfg.num_hidden_layers):
        distinct = X * (1.0 - (1.0 - k / X) ** rows)
        if not apart and layer >= 2:
            distinct = min(distinct, max(k, 55 / 256 * X))
        bytes_ += attention * wb + (X * E + X + 2 * E + q + kv) * 4 + distinct * expert * wb + (kv_read + rows) * 2 * kv * wb
        flops += 2.0 * rows * (attention + X * E + k * expert) + 4.0 * q * keys
    head = E * cfg.vocab_size
    return {"bytes": bytes_ + head * wb + E * 4 + rows * E * wb + wants * cfg.vocab_size * 4, "flops": flops + 2.0 * wants * head}


def _design_work(cfg, tokens, decoded):
    """A replay's bytes and operations: every weight a step uses once a step, prompt rows and decoded rows through the layers."""
    E, V, T = cfg.width, cfg.vocab, tokens
    weights = 0.0                  # elements every step reads and multiplies a row by
    mixing = state = cached = 0.0  # multiply-adds x 2 of the prompt's mixing; state bytes; cached bytes a token
    pairs = T * (T + 1) / 2.0
    for i, layer in enumerate(cfg.layers):
        m = layer.mixer
        if layer.type == "mingru":
            w, state = 4 * E * m.width, state + 8 * m.width
            mixing += 4.0 * T * m.width
        elif layer.type == "latent_attention":
            w = E * (m.heads * (m.dim + m.rot_dim) + m.kv_rank + m.rot_dim + m.heads) + m.heads * m.kv_rank * (m.dim + m.vdim) + m.heads * m.vdim * E
            mixing += 2.0 * m.heads * (m.dim + m.rot_dim + m.vdim) * pairs
            cached += 2 * (m.kv_rank + m.rot_dim)
        else:
            w = 0
            parts = [m.right] if layer.type == "parallel" else [m]
            if layer.type == "parallel":
                a = m.left
                w += E * (a.heads * a.dim + a.kv_heads * (a.dim + a.vdim)) + a.heads * a.vdim * E
                mixing += 2.0 * a.heads * (a.dim + a.vdim) * sum(min(t + 1, a.window) for t in range(T))
                cached += 2 * a.kv_heads * (a.dim + a.vdim) * min(T, a.window) / max(T, 1)
            for r in parts:
                ranks = cfg.ranks[i]
                w += E * (2 * r.kv_heads * r.dim + r.heads * r.vdim) + r.heads * r.vdim * E + E * (ranks["decay"] + ranks["gate"] + r.heads)
                w += ranks["decay"] * r.heads * r.dim + ranks["gate"] * r.heads * r.vdim
                mixing += 7.0 * T * r.heads * r.dim * r.vdim
                state += 8 * r.heads * r.dim * r.vdim
        w += 2 * E * layer.ff if hasattr(layer, "ff") else 3 * E * layer.mlp.ff
        side = getattr(cfg, "token_side_dim", None) or 0
        weights += w + 2 * E * side
    read = 2 * (weights + E * V)
    bytes_ = read + decoded * (read + cached * (T + decoded / 2.0)) + (1 + decoded) * (state + 4 * V) + T * (cached + 2 * E)
    flops = 2.0 * (T + decoded) * weights + mixing + 2.0 * (1 + decoded) * E * V
    return {"bytes": bytes_, "flops": flops}


def work(case):
    cfg = _config(case)
    kind = case["kind"]
    if kind == "replay":
        return _design_work(cfg, case["tokens"], case["decoded"])
    wb = 2 if case["dtype"] == "bf16" else 4
    if kind == "decode":
        held = case["batch"] * case["context"]
        return {k: v * case["steps"] for k, v in _m3_work(cfg, wb, case["batch"], held, case["batch"], held, True).items()}
    if kind == "prompt":
        n, T = case["prompts"], case["tokens"]
        return _m3_work(cfg, wb, n * T, n * T * (T + 1) / 2.0, n * min(T, case["want"]), 0, n > 8)
    T = case["tokens"]
    if kind == "mixed":
        held = case["batch"] * case["context"]
        return _m3_work(cfg, wb, case["batch"] + T, held + T * (T + 1) / 2.0, case["batch"] + 1, held, False)
    return _m3_work(cfg, wb, T, T * (T + 1) / 2.0, T, 0, False)


def tolerance(case):
    """About four times the distance from the 64-bit results that was measured over listed and drawn cases."""
    if case["dtype"] == "f32":
        return {"rel": 1.2e-5, "max": 6e-5}      # 3e-6 and 1.5e-5: 32-bit sums through eight layers
    if case["model"] in ("m3", "m3_w256"):
        # 0.004 to 0.01 where every row picks the experts it picks in 64 bits; 0.04 to 0.07 over the rows of a pass of which some
        # have a last pick and a best expert left out within a bf16 rounding of each other that change places (that row: 0.13)
        return {"rel": 0.2}
    return {"rel": 0.03, "max": 0.18}            # 0.004 to 0.008 and 0.02 to 0.045


# --------------------------------------------------------------------------------------------------- the same in 64 bits
def _f(x):
    return x.to(torch.float64)


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(z):
    return z * torch.sigmoid(z)


def _layer_norm(x, w, eps):
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps) * _f(w)


def _attend(q, k, v, scale, first_row, window=None):
    """q [T, H, D] of positions first_row.., k [S, G, D], v [S, G, V], all in 64 bits -> [T, H, V]; causal, a window if given."""
    T, H, _ = q.shape
    S, G, V = v.shape
    out = torch.empty(T, H, V, dtype=q.dtype, device=q.device)
    for at in range(0, T, 1024):
        n = min(1024, T - at)
        hi = first_row + at + n
        lo = 0 if window is None else max(0, first_row + at - window + 1)
        row = torch.arange(first_row + at, hi, device=q.device)[:, None]
        key = torch.arange(lo, hi, device=q.device)[None, :]
        hidden = key > row
        if window is not None:
            hidden |= key <= row - window
        for h in range(H):
            g = h // (H // G)
            s = (q[at:at + n, h] @ k[lo:hi, g].t()) * scale
            s.masked_fill_(hidden, float("-inf"))
            out[at:at + n, h] = torch.softmax(s, -1) @ v[lo:hi, g]
    return out


def _experts(h, ids, weights, gate_up, down):
    """sum_j weights[t, j] expert_ids[t, j](h[t]) for SwiGLU experts, gate rows first."""
    out = torch.zeros_like(h)
    for e in torch.unique(ids).tolist():
        rows, slot = torch.nonzero(ids == e, as_tuple=True)
        z = h[rows] @ _f(gate_up[e]).t()
        F = z.shape[1] // 2
        out.index_add_(0, rows, ((_silu(z[:, :F]) * z[:, F:]) @ _f(down[e]).t()) * weights[rows, slot][:, None])
    return out


def _angles(positions, freq, magnitude=1.0):
    """cos and sin [T, 1, pairs]; the models define an angle as the 32-bit product of position and 32-bit frequency."""
    a = _f(positions.float()[:, None] * torch.from_numpy(freq.astype(np.float32)).to(positions.device)[None, :])[:, None, :]
    return torch.cos(a) * magnitude, torch.sin(a) * magnitude


def _m3_exact(cfg, w, sequences, wanted):
    """Logits of the wanted places (one list a sequence) of whole sequences."""
    eps, D, R = cfg.rms_norm_eps, cfg.head_dim, cfg.rotary_dim
    H, G = cfg.num_attention_heads, cfg.num_key_value_heads
    dev = w["model.norm.weight"].device
    lens = [len(s) for s in sequences]
    starts = np.concatenate([[0], np.cumsum(lens)]).tolist()
    x = _f(w["model.embed_tokens.weight"][torch.tensor(sum(sequences, []), device=dev)])
    pos = torch.cat([torch.arange(n, device=dev) for n in lens])
    rows = torch.tensor([starts[i] + j for i, want in enumerate(wanted) for j in want], device=dev)
    exponent = (2.0 * np.arange(R // 2, dtype=np.float32)) / np.float32(R)
    power = np.power(np.float64(np.float32(cfg.rope_theta)), exponent.astype(np.float64)).astype(np.float32)
    cos, sin = _angles(pos, np.float32(1.0) / power)

    def turn(y, at):
        a, b = y[..., :R // 2], y[..., R // 2:R]
        return torch.cat([a * cos[at] - b * sin[at], b * cos[at] + a * sin[at], y[..., R:]], -1)

    for layer in range(cfg.num_hidden_layers):
        p = f"model.layers.{layer}."
        a = p + "self_attn."
        last = layer == cfg.num_hidden_layers - 1
        h = _rms(x, eps) * _f(w[p + "input_layernorm.weight"])
        k = turn((_rms(h @ _f(w[a + "k_proj.weight"]).t(), eps) * _f(w[a + "k_norm.weight"])).view(-1, G, D), slice(None))
        v = (h @ _f(w[a + "v_proj.weight"]).t()).view(-1, G, D)
        at = rows if last else torch.arange(x.shape[0], device=dev)      # of the last layer only the wanted rows go on
        q = turn((_rms(h[at] @ _f(w[a + "q_proj.weight"]).t(), eps) * _f(w[a + "q_norm.weight"])).view(-1, H, D), at)
        o = torch.empty_like(q)
        done = 0
        for i, want in enumerate(wanted):
            ks, vs = k[starts[i]:starts[i + 1]], v[starts[i]:starts[i + 1]]
            if last:
                for j in ([want] if len(want) == lens[i] else [[j] for j in want]):
                    o[done:done + len(j)] = _attend(q[done:done + len(j)], ks, vs, D ** -0.5, j[0])
                    done += len(j)
            else:
                o[starts[i]:starts[i + 1]] = _attend(q[starts[i]:starts[i + 1]], ks, vs, D ** -0.5, 0)
        x = x[at] + o.reshape(-1, H * D) @ _f(w[a + "o_proj.weight"]).t()
        del q, k, v, o
        h = _rms(x, eps) * _f(w[p + "post_attention_layernorm.weight"])
        s = torch.sigmoid(h @ _f(w[p + "mlp.gate.weight"]).t())
        ids = torch.topk(s + _f(w[p + "mlp.gate.e_score_correction_bias"]), cfg.num_experts_per_tok, dim=1).indices
        chosen = s.gather(1, ids)
        x = x + _experts(h, ids, chosen / chosen.sum(1, keepdim=True), w[p + "mlp.experts.gate_up_proj"], w[p + "mlp.experts.down_proj"])
    return (_rms(x, eps) * _f(w["model.norm.weight"])) @ _f(w["lm_head.weight"]).t()


def _pairs(y, cos, sin):
    """Dims (2i, 2i + 1) of every head turn; those beyond the angles' pairs pass."""
    n = 2 * cos.shape[-1]
    a, b = y[..., 0:n:2], y[..., 1:n:2]
    return torch.cat([torch.stack([a * cos - b * sin, b * cos + a * sin], -1).flatten(-2), y[..., n:]], -1)


def _blended(dims, base, s):
    """Rotary frequencies, slow pairs slowed down by the scaling's factor, and the factor on cos and sin."""
    i = np.arange(dims // 2, dtype=np.float64)
    f = float(base) ** (-2.0 * i / dims)
    if s is None:
        return f, 1.0
    pair = lambda turns: dims * math.log(s.original / (2.0 * math.pi * turns)) / (2.0 * math.log(base))
    lo, hi = max(math.floor(pair(s.fast)), 0), min(math.ceil(pair(s.slow)), dims - 1)
    ramp = np.clip((i - lo) / max(hi - lo, 0.001), 0.0, 1.0)
    return f / s.factor * ramp + f * (1.0 - ramp), 0.1 * math.log(s.factor) + 1.0


def _conv_silu(x, taps):
    n = taps.shape[1]
    padded = torch.cat([torch.zeros(n - 1, x.shape[1], dtype=x.dtype, device=x.device), x])
    return _silu(sum(padded[j:j + x.shape[0]] * _f(taps[:, j]) for j in range(n)))


def _delta(w, p, x, m, eps):
    T, H, G, D, V = x.shape[0], m.heads, m.kv_heads, m.dim, m.vdim
    lin = lambda name, y=x: y @ _f(w[p + name]).t()
    q, k, v = (_conv_silu(lin(n), w[p + n + ".conv"]).view(T, -1, d) for n, d in (("q", D), ("k", D), ("v", V)))
    unit = lambda y: (y / torch.sqrt((y * y).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, 1)
    q, k = unit(q) * D ** -0.5, unit(k)
    beta = torch.sigmoid(lin("b"))
    step = torch.nn.functional.softplus(lin("a2", lin("a1")) + _f(w[p + "dt_bias"])).view(T, H, D)
    decay = torch.exp(-torch.exp(_f(w[p + "A_log"]))[None, :, None] * step)
    S, o = torch.zeros(H, D, V, dtype=x.dtype, device=x.device), torch.empty(T, H, V, dtype=x.dtype, device=x.device)
    for t in range(T):
        S = S * decay[t][:, :, None]
        u = beta[t][:, None] * (v[t] - (S * k[t][:, :, None]).sum(1))
        S = S + k[t][:, :, None] * u[:, None, :]
        o[t] = (S * q[t][:, :, None]).sum(1)
    o = _rms(o, eps) * _f(w[p + "norm"]) * torch.sigmoid(lin("g2", lin("g1"))).view(T, H, V)
    return o.view(T, -1) @ _f(w[p + "o"]).t()


def _bonerax_exact(cfg, w, tokens, wanted):
    eps = cfg.norm_eps
    dev = w["head"].device
    x = _f(w["embed"][torch.tensor(tokens, device=dev)])
    T = x.shape[0]
    pos = torch.arange(T, device=dev)
    for i, layer in enumerate(cfg.layers):
        p, m = f"l{i}.mix.", layer.mixer
        if layer.type == "channel_delta":
            y = _delta(w, p, x, m, eps)
        else:
            a, l = m.left, p + "left."
            lin = lambda n, width: (x @ _f(w[l + n]).t() + _f(w[l + n + ".b"])).view(T, -1, width)
            cos, sin = _angles(pos, *_blended(a.rot_dims, a.rot_base, a.rot_scaling))
            q = _pairs(_rms(lin("q", a.dim), eps) * _f(w[l + "q.norm"]), cos, sin)
            k = _pairs(_rms(lin("k", a.dim), eps) * _f(w[l + "k.norm"]), cos, sin)
            o = _attend(q, k, lin("v", a.vdim), a.scale, 0, a.window).reshape(T, -1)
            y = m.left_scale * (o @ _f(w[l + "o"]).t() + _f(w[l + "o.b"])) + m.right_scale * _delta(w, p + "right.", x, m.right, eps)
        x = x + _layer_norm(y, w[f"l{i}.norm1"], eps)
        lin = lambda n, y=x: y @ _f(w[f"l{i}.mlp.{n}"]).t()
        y = lin("down", _silu(lin("gate")) * lin("up"))
        x = x + _layer_norm(y, w[f"l{i}.norm2"], eps)
    x = _layer_norm(x[wanted], w["final.norm"], eps)
    return cfg.logit_softcap * torch.tanh(x @ _f(w["head"]).t() * cfg.logit_scale / cfg.logit_softcap)


def _latent(w, p, h, m, eps):
    T, H = h.shape[0], m.heads
    lin = lambda name, y=h: y @ _f(w[p + name]).t()
    cos, sin = _angles(torch.arange(T, device=h.device), *_blended(m.rot_dims, m.rot_base, m.rot_scaling))
    q = lin("q").view(T, H, m.dim + m.rot_dim)
    q = torch.cat([q[..., :m.dim], _pairs(q[..., m.dim:], cos, sin)], -1)
    down = lin("dkv")
    c = _rms(down[:, :m.kv_rank], eps) * _f(w[p + "dkv.norm"])
    shared = _pairs(down[:, None, m.kv_rank:], cos, sin).expand(T, H, m.rot_dim)
    k = torch.cat([lin("uk", c).view(T, H, m.dim), shared], -1)
    o = _attend(q, k, lin("uv", c).view(T, H, m.vdim), m.scale, 0) * torch.sigmoid(lin("g"))[:, :, None]
    return o.reshape(T, -1) @ _f(w[p + "o"]).t()


def _mingru(w, p, h, m):
    lin = lambda name, y=h: y @ _f(w[p + name]).t()
    z, u = torch.sigmoid(lin("z") + _f(w[p + "z.b"])), lin("x") + _f(w[p + "x.b"])
    c = z * torch.where(u >= 0, u + 0.5, torch.sigmoid(u))
    S, rows = torch.zeros(m.width, dtype=h.dtype, device=h.device), torch.empty_like(c)
    for t in range(h.shape[0]):
        S = (1.0 - z[t]) * S + c[t]
        rows[t] = S
    return lin("o", rows * _silu(lin("g")))


def _nenotar_exact(cfg, w, tokens, wanted):
    eps, dim = cfg.norm_eps, cfg.token_side_dim
    ids = torch.tensor(tokens, device=w["head"].device)
    x = _f(w["embed"][ids]) * cfg.embedding_scale
    for i, layer in enumerate(cfg.layers):
        p = f"l{i}."
        h = _rms(x, eps) * _f(w[p + "norm1"])
        y = (_mingru(w, p + "mix.", h, layer.mixer) if layer.type == "mingru" else _latent(w, p + "mix.", h, layer.mixer, eps)) * _f(w[p + "ls1"])
        h = _rms(x, eps) * _f(w[p + "norm2"])
        z = h @ _f(w[p + "mlp.up"]).t()
        up, low = torch.nn.functional.softplus(_f(w[p + "mlp.act"]))
        z = torch.where(z > 0, up * z * z, (0.5 + low) * (torch.expm1(z.clamp(max=0.0)) - z)) + 0.5 * z
        x = x + y + (z @ _f(w[p + "mlp.down"]).t()) * _f(w[p + "ls2"])
        g = torch.nn.functional.gelu(x @ _f(w[p + "side.gate"]).t(), approximate="tanh") * _f(w["side.embed"][ids, i * dim:(i + 1) * dim])
        x = x + _rms(g @ _f(w[p + "side.proj"]).t(), eps) * _f(w[p + "side.norm"])
    return (_rms(x[wanted], eps) * _f(w["final.norm"])) @ _f(w["head"]).t()


def exact(case, seed):
    """The pass's logits in 64 bits from the same weights and tokens."""
    cfg, t, w = _config(case), _tokens(case, seed), {}
    _engine(case, seed, tokens_out=w)        # the weights by name; nothing of the engine is kept
    kind = case["kind"]
    if kind == "replay":
        places = [case["tokens"] - 1 + j for j in range(case["decoded"] + 1)]
        forward = _bonerax_exact if case["model"] == "bonerax" else _nenotar_exact
        return forward(cfg, w, t["text"] + t["decoded"], places)
    if kind == "score":
        return _m3_exact(cfg, w, [t["text"]], [list(range(len(t["text"])))])
    if kind == "prompt":
        return _m3_exact(cfg, w, t["texts"], [_last(x, case) for x in t["texts"]])
    sequences = [x + n for x, n in zip(t["texts"], t["next"])]
    if kind == "mixed":
        sequences.append(t["text"])
        return _m3_exact(cfg, w, sequences, [[len(s) - 1] for s in sequences])
    steps = case["steps"]
    rows = _m3_exact(cfg, w, sequences, [list(range(len(s) - steps, len(s))) for s in sequences])
    return rows if steps == 1 else rows.view(len(sequences), steps, -1).transpose(0, 1)
