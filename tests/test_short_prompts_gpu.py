"""Steps of few tokens take the fused chain whatever they are made of: the same
logits, keys and values as the general path gives.

Tolerance: both paths round the residual stream and the operands of every
product to bf16, at other places: some 12 roundings a path and layer, each off
by 2^-9 / sqrt(3) of a value's size in the mean, sum to sqrt(2 * 2 * 12) times
that or 2^-7 of the logits' norm; twice that is allowed.  Single values differ
like normal ones: they are nearly alike in the first layer and up to the
allowed 2^-6 off in the mean in the last, and of 300000 normal values the
furthest lies 5 times the mean off: 10 times 2^-7.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _close(a, b):
    size = b.square().mean().sqrt()
    off = (a - b).abs()
    assert off.square().mean().sqrt() <= 2 ** -6 * size
    assert off.max() <= 10 * 2 ** -7 * size


def _run(model, cfg, fused, steps, streams=5, ctx=256, pages=96):
    """Logits of every step, and the keys and values at the end; a step is a
    list of (stream, tokens, wanted places)."""
    from ollamamq_amd.engine import LlamaEngine, PagedKVCache
    model.fused_chain = fused
    kv = PagedKVCache.for_model(cfg, n_pages=pages, max_slots=streams + 1,
                                max_ctx=ctx, device="cuda:0",
                                dtype=torch.bfloat16)
    eng = LlamaEngine(model, kv, max_batch=4)
    eng.use_graphs = False
    streams = [eng.open_stream() for _ in range(streams)]
    out = [eng.feed([(streams[i], list(t), list(w)) for i, t, w in step])
           for step in steps]
    return out, kv.k_pool.float(), kv.v_pool.float()


STEPS = [
    # one portion, its last place wanted; every place; none
    [(0, range(1, 38), [36])],
    [(0, range(9, 41), range(32))],
    [(1, range(64), [])],
    # portions and single tokens, unsorted, places repeated and out of order
    [(2, range(3, 20), [16, 2, 2]), (0, [5], [0]), (3, range(40), [39]),
     (1, [7], [0])],
    # more than 64 tokens, and places
    [(4, range(65), [64, 0])],
    [(4, range(12), [3] * 70)],
    [(i, [i], [0]) for i in range(5)],
    # as many tokens as the chain takes, one too many, and more places
    [(1, range(128), [127])],
    [(2, range(129), [128, 0])],
    [(3, range(20), [11] * 129)],
]


@pytest.mark.parametrize("name", ["tiny", "tiny-qwen", "tiny-swa"])
def test_chain_and_general_path(name):
    from ollamamq_amd.models import LlamaModel, PRESETS
    cfg = PRESETS[name]
    model = LlamaModel(cfg, device="cuda:0", dtype=torch.bfloat16, seed=5)
    assert model.fused_chain
    got, k1, v1 = _run(model, cfg, True, STEPS)
    want, k2, v2 = _run(model, cfg, False, STEPS)
    for a, b, step in zip(got, want, STEPS):
        assert a.shape == b.shape == (sum(len(w) for _, _, w in step),
                                      cfg.vocab)
        if len(b):
            _close(a.float(), b.float())
    # the pools hold zeros where nothing was cached
    _close(k1[k2 != 0], k2[k2 != 0])
    _close(v1[v2 != 0], v2[v2 != 0])
    assert torch.equal(k1 != 0, k2 != 0) and torch.equal(v1 != 0, v2 != 0)


@pytest.mark.parametrize("env, every, over_tiles", [
    ({}, None, {512, 1024}), ({"OLLAMAMQ_WS_KS_512": "1"}, None, {1024}),
    ({"OLLAMAMQ_WS_KS_1024": "2"}, None, {512}), ({}, "1", set())])
def test_parts_asked_for(env, every, over_tiles, monkeypatch):
    """OLLAMAMQ_WS_KS and OLLAMAMQ_WS_KS_<K> reach o and down of a step of any
    size: a product that they name is streamed."""
    from ollamamq_amd.models import LlamaModel, PRESETS
    from ollamamq_amd.ops import hip
    cfg = PRESETS["tiny"]
    model = LlamaModel(cfg, device="cuda:0", dtype=torch.bfloat16, seed=5)
    assert (cfg.q_dim, cfg.ffn) == (512, 1024)
    step = [[(0, range(64), [63])]]
    want = _run(model, cfg, False, step)[0][0]
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    monkeypatch.setattr(hip, "_WS_KS", every)
    seen, product = set(), hip.tile_residual
    monkeypatch.setattr(hip, "tile_residual",
                        lambda x, w, M, N, K, *a: seen.add(K)
                        or product(x, w, M, N, K, *a))
    _close(_run(model, cfg, True, step)[0][0].float(), want.float())
    assert seen == over_tiles


@pytest.mark.parametrize("heads, rounds", [(48, 1), (56, 2), (64, 2)])
def test_second_round_of_streams(heads, rounds, monkeypatch):
    """Rotated products go over tiles where their streams' blocks of 32
    columns are more than the CUs."""
    import dataclasses
    from ollamamq_amd.models import LlamaModel, PRESETS
    from ollamamq_amd.ops import hip
    cfg = dataclasses.replace(PRESETS["tiny"], n_heads=heads, n_kv_heads=8)
    blocks = (cfg.q_dim + 2 * cfg.kv_dim) // 32
    assert -(-blocks // hip._cus(0)) == rounds
    model = LlamaModel(cfg, device="cuda:0", dtype=torch.bfloat16, seed=5)
    seen, product = [], hip.tile_qkv_rope
    monkeypatch.setattr(hip, "tile_qkv_rope",
                        lambda *a: seen.append(a) or product(*a))
    for n in (49, 128):
        step = [[(0, range(n), [n - 1])]]
        got, k1, v1 = _run(model, cfg, True, step)
        want, k2, v2 = _run(model, cfg, False, step)
        _close(got[0].float(), want[0].float())
        for a, b in ((k1, k2), (v1, v2)):
            _close(a[b != 0], b[b != 0])    # the pools hold zeros elsewhere
    assert len(seen) == (2 * cfg.n_layers if rounds > 1 else 0)


@pytest.mark.parametrize("streams", [True, False])
def test_library_products_asked_for(streams, monkeypatch):
    """OLLAMAMQ_NO_WSTREAM reaches prompts of more rows than the chain's."""
    from ollamamq_amd.models import LlamaModel, PRESETS
    from ollamamq_amd.ops import hip
    cfg = PRESETS["tiny"]
    model = LlamaModel(cfg, device="cuda:0", dtype=torch.bfloat16, seed=5)
    monkeypatch.setattr(hip, "USE_WSTREAM", streams)
    seen, product = [], hip.tile_gu
    monkeypatch.setattr(hip, "tile_gu",
                        lambda *a: seen.append(a) or product(*a))
    _run(model, cfg, True, [[(0, range(129), [128])]])
    assert len(seen) == (cfg.n_layers if streams else 0)


@pytest.mark.parametrize("H", [64, 512, 4096])
def test_rows(H):
    from ollamamq_amd.ops import hip
    hip.require()
    x = torch.randn(64, H, device="cuda").bfloat16()
    xf, sq = hip.fragify_sumsq(x)
    for idx in ([0], [63, 0, 31, 32], list(range(64)), [5] * 40, []):
        rows = torch.tensor(idx, dtype=torch.long, device="cuda")
        got, n = hip.frag_rows(xf, rows, H)
        d = got.view(-1, H // 64, 4, 2, 32, 8).permute(0, 4, 1, 2, 3, 5)
        assert torch.equal(d.reshape(-1, H)[:len(idx)], x[rows])
        assert torch.equal(n, sq[rows])
