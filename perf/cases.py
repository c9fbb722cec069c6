"""The work by which this framework's speed is measured: what one GPU worker
does for its users, through the engine.

A case is one engine step (`LlamaEngine.feed`, the step of generation with the
tokens given, so that its results do not hang on a tie between two logits):

* `users` conversations of about `context` tokens get one token each.  They
  are ragged: half to one and a half times `context`, evenly spread;
* `prompts` new prompts of about `length` tokens, as ragged, run from their
  first token to the logits of their last.

Both in one step are a mixed batch, as when somebody asks while others are
answered.  Weights are random, drawn from the seed, with the architectures of
the presets; `layers` of 0 is the whole model, else a stack of that many of its
layers over a vocabulary of 32000, which is how bench.py --layers measures
designs of equal size.

    decode       users 1 to 128, contexts 16 to 12288
    prompts      1 to 16, lengths 8 to 8192, up to 8192 tokens a step
"""
import dataclasses
import math
import random

import torch

from ollamamq_amd.engine import LlamaEngine, cache_for_model
from ollamamq_amd.models import PRESETS, build_model

STACK_VOCAB = 32000
PAGE = 16
BATCH = 128             # most conversations of one step
PORTION = 8192          # tokens of conversation that prepare() feeds at once
MODELS = ("llama3-8b", "llama3.1-8b", "mistral-7b", "qwen2-7b", "llama2-7b",
          "kavedra-1b", "kavedra-8b")


def _case(name, model, layers, users=0, context=0, prompts=0, length=0):
    case = dict(model=model, layers=layers, users=users, context=context,
                prompts=prompts, length=length)
    return dict(case, name=name) if name else case


def listed():
    return [
        # one person chatting with the flagship model
        _case("8b 1 user", "llama3-8b", 0, 1, 300),
        # the headline workload: 32 concurrent users of the flagship model
        _case("8b 32 users", "llama3-8b", 0, 32, 512),
        # a busy node: the largest batches that a worker captures
        _case("busy node 128 users", "llama3-8b", 4, 128, 700),
        # questions about long documents: the cache outweighs the weights
        _case("long context 12 users", "llama3.1-8b", 4, 12, 8192),
        # grouped heads in sevens, biases, and an odd batch above 32
        _case("qwen2 45 users", "qwen2-7b", 4, 45, 600),
        # no grouped heads: four times the keys and values per token
        _case("llama2 20 users", "llama2-7b", 4, 20, 1100),
        # the first line of a chat, nobody else there
        _case("short prompt", "llama3-8b", 4, prompts=1, length=37),
        # several requests admitted together
        _case("ragged prompts", "llama3-8b", 4, prompts=7, length=330),
        # a document handed in whole; the window is shorter than it
        _case("long prompt", "mistral-7b", 4, prompts=1, length=8100),
        # a prompt admitted while others are being answered
        _case("prompt among 24 users", "llama3-8b", 4, 24, 800, 1, 517),
        # recurrent, softmax and latent layers: a small model's decode ...
        _case("kavedra 1b 32 users", "kavedra-1b", 4, 32, 512),
        # ... and a large one's prompts
        _case("kavedra 8b prompts", "kavedra-8b", 4, prompts=2,
              length=2048),
    ]


def _between(rng, lo, hi):
    return round(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    model = rng.choice(MODELS)
    limit = min(12288, PRESETS[model].max_ctx)
    kind = rng.choice(("decode", "decode", "prompts", "mixed"))
    users = context = prompts = length = 0
    if kind != "prompts":
        users = _between(rng, 1, 128 if kind == "decode" else 48)
        context = _between(rng, 16, min(limit // 2 if users > 1
                                        else limit - 8, 90000 // users))
    if kind != "decode":
        prompts = _between(rng, 1, 16) if kind == "prompts" else 1
        length = _between(rng, 8, min(
            limit // 2 if prompts > 1 else limit - 8,
            (7168 if kind == "prompts" else 2048) // prompts))
    return _case(None, model, 4, users, context, prompts, length)


def _ragged(n, mean):
    """n lengths about a mean: half to one and a half times, evenly."""
    if n == 1:
        return [mean]
    return [max(1, round(mean * (0.5 + i / (n - 1)))) for i in range(n)]


def _lengths(case):
    return (_ragged(case["users"], case["context"]),
            _ragged(case["prompts"], case["length"]))


def _config(case):
    cfg = PRESETS[case["model"]]
    n = case["layers"]
    if not n:
        return cfg
    if cfg.family == "llama":
        return dataclasses.replace(cfg, n_layers=n, vocab=STACK_VOCAB)
    return dataclasses.replace(cfg, layers=cfg.layers[:n], vocab=STACK_VOCAB)


def _texts(case, seed, vocab):
    """The tokens of every conversation, the new one last, and of every
    prompt."""
    rng = random.Random(seed)
    held, new = _lengths(case)
    return ([[rng.randrange(vocab) for _ in range(n + 1)] for n in held],
            [[rng.randrange(vocab) for _ in range(n)] for n in new])


def prepare(case, seed):
    """An engine with its model loaded and the conversations in its cache."""
    cfg = _config(case)
    held, new = _lengths(case)
    longest = max(held + new) + 2
    model = build_model(cfg, device="cuda:0", dtype=torch.bfloat16,
                        seed=seed, fast_init=True)
    slots = len(held) + len(new) + 2
    pages = sum(n // PAGE + 2 for n in held + new) + 8
    cache = cache_for_model(cfg, n_pages=pages, max_slots=slots,
                            max_ctx=longest, device="cuda:0",
                            dtype=torch.bfloat16)
    engine = LlamaEngine(model, cache, max_batch=BATCH)
    talks, prompts = _texts(case, seed, cfg.vocab)
    streams = [engine.open_stream() for _ in talks]
    # whole conversations but for their last token, some at a time
    at, parts = 0, []
    for stream, talk in zip(streams, talks):
        text = talk[:-2]
        if text:
            parts.append((stream, text, []))
            at += len(text)
        if parts and at >= PORTION:
            engine.feed(parts)
            at, parts = 0, []
    if parts:
        engine.feed(parts)
    if streams:                     # a decode step, as generation does
        engine.feed([(s, [t[-2]], []) for s, t in zip(streams, talks)])
    return {"engine": engine, "prompts": prompts,
            "talks": [(s, n, t[-1]) for s, n, t in
                      zip(streams, held, talks)]}


def run(state):
    """One step; logits [users + prompts, vocab].  A conversation goes on from
    the same length in every pass."""
    engine = state["engine"]
    parts = []
    for stream, length, token in state["talks"]:
        engine.kv.ensure(stream.slot, length)
        parts.append((stream, [token], [0]))
    fresh = []
    for prompt in state["prompts"]:
        fresh.append(engine.open_stream())
        parts.append((fresh[-1], prompt, [len(prompt) - 1]))
    logits = engine.feed(parts)
    for stream in fresh:
        engine.close_stream(stream)
    return logits


# ------------------------------------------------------------ what it takes

def _seen(n, window):
    """(key, query) pairs of a sequence of n tokens from its first on."""
    w = min(n, window or n)
    return w * (w + 1) // 2 + (n - w) * w


def _mixers(cfg):
    """Per layer: weights, cached values per token, state values, operations
    per (key, query) pair, the window, operations of a recurrence per
    token."""
    if cfg.family == "llama":
        return [(cfg.hidden * (2 * cfg.q_dim + 2 * cfg.kv_dim + 3 * cfg.ffn),
                 2 * cfg.kv_dim, 0, 4 * cfg.q_dim, cfg.sliding_window, 0)
                ] * cfg.n_layers
    found, width = [], cfg.width
    for s in cfg.layers:
        qk, v, ff = s.heads * s.dim, s.heads * s.vdim, 3 * width * s.ff
        if s.type == "lightning":
            found.append((ff + width * (2 * qk + 3 * v), 0, qk * s.vdim, 0,
                          0, 4 * qk * s.vdim))
        elif s.type == "attention":
            kv = s.kv_heads * (s.dim + s.vdim)
            found.append((ff + width * (qk + v + kv), kv, 0, 2 * (qk + v),
                          s.window, 0))
        else:
            row = s.kv_rank + s.rot_dim
            found.append((ff + width * (qk + s.heads * s.rot_dim + row + 2 * v)
                          + s.kv_rank * (qk + v), row, 0,
                          2 * (qk + v + s.heads * s.rot_dim), s.window, 0))
    return found


def work(case):
    """Every weight and every cached value that a step sees read once, new
    cache rows, states and logits written once."""
    cfg = _config(case)
    width = cfg.hidden if cfg.family == "llama" else cfg.width
    held, new = _lengths(case)
    rows, tokens = len(held) + len(new), len(held) + sum(new)
    nbytes = 2 * cfg.vocab * width + 2 * tokens * width + 2 * rows * cfg.vocab
    flops = 2 * rows * cfg.vocab * width
    for weights, cached, state, per_pair, window, per_token in _mixers(cfg):
        reach = [min(n + 1, window or n + 1) for n in held]
        nbytes += 2 * weights + 2 * cached * (sum(reach) + sum(new))
        nbytes += 4 * state * (2 * len(held) + len(new))
        flops += 2 * weights * tokens + per_token * tokens
        flops += per_pair * (sum(reach) + sum(_seen(n, window) for n in new))
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Llama's residual stream is bf16, so the roundings of every layer stay in
    it: 0.009 to 0.015 against 64 bits, and two orders of summing are that far
    from each other.  Kavedra's is fp32: 0.004 to 0.005."""
    if case["model"].startswith("kavedra"):
        return {"rel": 0.02, "max": 0.15}
    return {"rel": 0.03, "max": 0.2}


# ------------------------------------- the same in 64 bits, in plain torch

F64 = torch.float64
ROWS = 16384            # rows of a product at a time


class _Draws:
    """The seeded weights in the order in which a model draws them."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def __call__(self, *shape, mean=0.0, spread=None):
        if spread is None:
            spread = 1.0 / math.sqrt(shape[-1])
        w = torch.empty(shape, device="cuda", dtype=torch.float32)
        w.normal_(mean, spread, generator=self.gen)
        return w.to(torch.bfloat16).to(F64)


def _times(x, w):
    return torch.cat([part @ w.T for part in x.split(ROWS)])


def _rms(x, eps):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt()


def _silu(x):
    return x / (1 + (-x).exp())


def _gated(x, w_gate, w_up, w_down):
    return torch.cat([(_silu(part @ w_gate.T) * (part @ w_up.T)) @ w_down.T
                      for part in x.split(ROWS // 2)])


def _turn(x, angles, magnitude, halves):
    """Rotary positions over the last dimension of x [T, heads, dim]."""
    c, s = (f(angles)[:, None] * magnitude for f in (torch.cos, torch.sin))
    if halves:
        u, v = x.chunk(2, -1)
        return torch.cat([u * c - v * s, v * c + u * s], -1)
    u, v = x[..., 0::2], x[..., 1::2]
    return torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2)


def _attend(q, k, v, scale, window=0, sink=None):
    """Causal softmax attention of one sequence: q [T, H, D], k and v
    [T, G, .]; `sink` is one more term of the denominator."""
    n, heads = q.shape[:2]
    group = heads // k.shape[1]
    at = torch.arange(n, device=q.device)
    out = q.new_empty(n, heads, v.shape[2])
    for lo in range(0, n, 2048):
        hi = min(n, lo + 2048)
        gone = at[None, :hi] > at[lo:hi, None]
        if window:
            gone |= at[None, :hi] <= at[lo:hi, None] - window
        for h in range(heads):
            s = q[lo:hi, h] @ k[:hi, h // group].T * scale
            s.masked_fill_(gone, -math.inf)
            if sink is not None:
                s = torch.cat([s, sink[h].expand(hi - lo, 1)], 1)
            s = s.softmax(-1)[:, :hi]
            out[lo:hi, h] = s @ v[:hi, h // group]
    return out.flatten(1)


def _per_text(lengths, fn, *rows):
    """fn over the rows of one sequence after another."""
    return torch.cat([fn(*part) for part in
                      zip(*(r.split(lengths) for r in rows))])


def _exact_llama(cfg, seed, tokens, lengths):
    get, hid, d = _Draws(seed), cfg.hidden, cfg.head_dim
    by_width = 1.0 / math.sqrt(hid)
    x = get(cfg.vocab, hid)[tokens]
    pair = torch.arange(0, d, 2, dtype=F64, device="cuda")
    turn = cfg.rope_theta ** (-pair / d)
    if cfg.rope_scaling:
        factor, low, high, first = cfg.rope_scaling
        turns = first * turn / (2 * math.pi)
        kept = ((turns - low) / (high - low)).clamp(0, 1)
        turn = turn * (kept + (1 - kept) / factor)

    def attend(rows):
        at = torch.arange(len(rows), dtype=F64, device="cuda")
        angles = torch.outer(at, turn)
        q, k, v = (t.unflatten(1, (-1, d)) for t in rows.split(
            [cfg.q_dim, cfg.kv_dim, cfg.kv_dim], 1))
        return _attend(_turn(q, angles, 1.0, True),
                       _turn(k, angles, 1.0, True), v, d ** -0.5,
                       cfg.sliding_window)

    for _ in range(cfg.n_layers):
        w_in = get(cfg.q_dim + 2 * cfg.kv_dim, hid)
        rows = _times(_rms(x, cfg.norm_eps), w_in)
        if cfg.qkv_bias:
            rows += get(len(w_in), spread=by_width)
        o = _per_text(lengths, attend, rows)
        x = x + _times(o, get(hid, cfg.q_dim, spread=by_width))
        w_gate, w_up = get(2 * cfg.ffn, hid).chunk(2)
        x = x + _gated(_rms(x, cfg.norm_eps), w_gate, w_up,
                       get(hid, cfg.ffn))
    ends = torch.tensor(lengths, device="cuda").cumsum(0) - 1
    return _rms(x[ends], cfg.norm_eps) @ get(cfg.vocab, hid).T


def _pair_turns(spec):
    """Angle per token of every pair of a head, and the factor of its
    rotation: YaRN's where the spec has a scaling."""
    n = spec.dims
    pair = torch.arange(n // 2, dtype=F64, device="cuda")
    turn = spec.base ** (-2 * pair / n)
    if spec.scaling is None:
        return turn, 1.0
    factor, first, fast, slow = spec.scaling

    def at(turns):
        return n * math.log(first / (2 * math.pi * turns)) \
            / (2 * math.log(spec.base))

    lo = max(math.floor(at(fast)), 0)
    hi = min(math.ceil(at(slow)), n - 1)
    ramp = ((pair - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    return turn * (1 - ramp + ramp / factor), 0.1 * math.log(factor) + 1


def _exact_kavedra(cfg, seed, tokens, lengths):
    get, width, eps = _Draws(seed), cfg.width, cfg.eps

    def vec(n, mean=0.0):
        return get(n, mean=mean, spread=0.1)

    def turned(t, spec):
        turn, magnitude = _pair_turns(spec)
        at = torch.arange(len(t), dtype=F64, device="cuda")
        return _turn(t, torch.outer(at, turn), magnitude, spec.halves)

    def lightning(s, h):
        qk, v = s.heads * s.dim, s.heads * s.vdim
        mats = [get(n, width) for n in (qk, qk, v, v)]
        w_norm = vec(v, 1.0)

        def mix(q, k, v):
            q, k, v = (_silu(t).unflatten(1, (s.heads, -1))
                       for t in (q, k, v))
            at = torch.arange(len(q), dtype=F64, device="cuda")
            gap = at[:, None] - at
            return torch.stack([
                ((s.decay[i] ** gap.clamp(min=0)) * (gap >= 0)
                 * (q[:, i] @ k[:, i].T)) @ v[:, i]
                for i in range(s.heads)], 1).flatten(1)

        q, k, v, gate = (_times(h, m) for m in mats)
        o = _per_text(lengths, mix, q, k, v)
        return _rms(o, eps) * w_norm * gate.sigmoid()

    def softmax(s, h):
        sizes = [s.heads * s.dim, s.kv_heads * s.dim, s.kv_heads * s.vdim]
        mats = [get(n, width) for n in sizes]
        bias = [vec(n) for n in sizes]
        sink = vec(s.heads)

        def mix(q, k, v):
            q, k = (turned(t.unflatten(1, (-1, s.dim)), s.rope)
                    for t in (q, k))
            return _attend(q, k, v.unflatten(1, (-1, s.vdim)), s.scale,
                           s.window, sink)

        return _per_text(lengths, mix, *(
            _times(h, m) + b for m, b in zip(mats, bias)))

    def latent(s, h):
        qk, v = s.heads * s.dim, s.heads * s.vdim
        rank, rot = s.kv_rank, s.rot_dim
        mats = [get(n, width) for n in (qk + s.heads * rot, rank + rot, v)]
        w_norm = vec(rank, 1.0)
        w_k, w_v = get(qk, rank), get(v, rank)

        def mix(q, row):
            q = q.unflatten(1, (s.heads, -1))
            q = torch.cat([q[..., :s.dim],
                           turned(q[..., s.dim:], s.rope)], -1)
            c = _rms(row[:, :rank], eps) * w_norm
            shared = turned(row[:, None, rank:], s.rope)
            k = torch.cat([(c @ w_k.T).unflatten(1, (s.heads, -1)),
                           shared.expand(-1, s.heads, -1)], -1)
            return _attend(q, k, (c @ w_v.T).unflatten(1, (s.heads, -1)),
                           s.scale, s.window)

        q, row, gate = (_times(h, m) for m in mats)
        return _per_text(lengths, mix, q, row) * gate.sigmoid()

    mixers = {"lightning": lightning, "attention": softmax,
              "latent_attention": latent}
    x = get(cfg.vocab, width, spread=1.0)[tokens]
    for s in cfg.layers:
        o = mixers[s.type](s, _rms(x, eps) * (1 + vec(width)))
        x = x + _times(o, get(width, s.heads * s.vdim))
        h = _rms(x, eps) * (1 + vec(width))
        mats = [get(s.ff, width), get(s.ff, width), get(width, s.ff)]
        x = x + _gated(h, *mats)
    ends = torch.tensor(lengths, device="cuda").cumsum(0) - 1
    h = _rms(x[ends], eps) * (1 + vec(width)) * cfg.logit_scale
    return h @ get(cfg.vocab, width).T


def exact(case, seed):
    cfg = _config(case)
    talks, prompts = _texts(case, seed, cfg.vocab)
    texts = talks + prompts
    tokens = torch.tensor([t for text in texts for t in text], device="cuda")
    of = _exact_llama if cfg.family == "llama" else _exact_kavedra
    return of(cfg, seed, tokens, [len(t) for t in texts])
