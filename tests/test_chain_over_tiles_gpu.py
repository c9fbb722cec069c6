"""The fused chain where its products go over tiles, in a model as wide as the
7 and 8 billion ones: parts of K and their sums of squares from product to
product, rotated products of steps of 49 to 128 rows, and single tokens beside
prompts of more than 128, against the general path.  Tolerance: see
test_short_prompts_gpu.py.
"""
import dataclasses

import pytest
import torch

from test_short_prompts_gpu import _close, _run

pytestmark = pytest.mark.gpu


def _text(n, first=0):
    return [(first + 7 * i) % 512 for i in range(n)]


STEPS = [
    # rows of the smallest tiles, of more, and of more than the streams take
    [(0, _text(49), [48])],
    [(1, _text(64, 3), [63, 0])],
    [(2, _text(65, 5), [64])],
    [(3, _text(128, 9), [127, 31, 32])],
    [(4, _text(130, 11), [129])],
    # single tokens and a long prompt: their attention in parts draws tickets
    # in every layer, gate-up takes several rounds of tiles
    [(0, [5], [0]), (3, [6], [0]), (2, _text(550, 2), [549, 0]),
     (1, [7], [0]), (4, [8], [0])],
    # as many as fill the step by themselves, and two prompts
    [(i, [i], [0]) for i in range(60)] + [(60, _text(200), [199]),
                                          (61, _text(37), [36])],
    # decode of 62: longest contexts 615
    [(i, [i + 1], [0]) for i in range(62)],
    [(2, _text(131, 4), [130]), (0, _text(300, 1), [299]), (3, [9], [0])],
]
ROWS = [49, 64, 65, 128, 130, 554, 297, 62, 432]


@pytest.mark.parametrize("kv_heads, bias, window", [
    (32, False, 0), (8, True, 0), (32, False, 100)])
def test_against_general_path(kv_heads, bias, window, monkeypatch):
    from ollamamq_amd.models import LlamaModel, PRESETS
    from ollamamq_amd.ops import hip
    cfg = dataclasses.replace(
        PRESETS["llama2-7b"], name="wide", n_layers=2, n_kv_heads=kv_heads,
        ffn=6144, vocab=512, qkv_bias=bias, sliding_window=window,
        max_ctx=1024)
    model = LlamaModel(cfg, device="cuda:0", dtype=torch.bfloat16, seed=5,
                       fast_init=True)
    seen, product = [], hip._tile_gemm

    def spy(epi, y, x, packed, M, *a, **k):
        seen.append((epi, M))
        product(epi, y, x, packed, M, *a, **k)
    monkeypatch.setattr(hip, "_tile_gemm", spy)
    size = dict(streams=62, ctx=1024, pages=260)
    got, k1, v1 = _run(model, cfg, True, STEPS, **size)
    took, many = set(seen), len(seen)
    assert {M for epi, M in took
            if epi in (hip.TILE_RESIDUAL, hip.TILE_PARTS)} == set(ROWS)
    assert {M for epi, M in took if epi == hip.TILE_PARTS} >= {
        49, 64, 65, 128, 130, 554}
    assert {M for epi, M in took if epi == hip.TILE_ROPE} == {
        M for M in ROWS if M > 128 or kv_heads == 32}
    assert {M for epi, M in took if epi == hip.TILE_GATED} == {
        M for M in ROWS if M > 128}
    want, k2, v2 = _run(model, cfg, False, STEPS, **size)
    assert len(seen) == many
    for a, b, step in zip(got, want, STEPS):
        assert a.shape == b.shape == (sum(len(w) for _, _, w in step),
                                      cfg.vocab)
        _close(a.float(), b.float())
    # the pools hold zeros where nothing was cached
    for a, b in ((k1, k2), (v1, v2)):
        _close(a[b != 0], b[b != 0])
        assert torch.equal(a != 0, b != 0)


@pytest.mark.parametrize("hidden, heads, kv_heads, taken", [
    (4096, 32, 8, {97, 128}),                   # two parts
    (3584, 28, 4, {49, 64, 65, 96, 97, 128})])  # three
def test_qkv_in_parts(hidden, heads, kv_heads, taken, monkeypatch):
    """Which steps take them, and that their queries, keys and values are the
    general path's: over tiles of 64 and of 128 rows, prompts and decode."""
    from ollamamq_amd.models import LlamaModel, PRESETS
    from ollamamq_amd.ops import hip
    cfg = dataclasses.replace(
        PRESETS["qwen2-7b"], name="wide", hidden=hidden, n_heads=heads,
        n_kv_heads=kv_heads, n_layers=2, ffn=2048, vocab=512, max_ctx=256)
    model = LlamaModel(cfg, device="cuda:0", dtype=torch.bfloat16, seed=5,
                       fast_init=True)
    rows, product = [], hip.tile_qkv_parts

    def spy(x, packed, M, *a):
        rows.append(M)
        return product(x, packed, M, *a)
    monkeypatch.setattr(hip, "tile_qkv_parts", spy)
    steps = [[(i, _text(n, i), [n - 1])]
             for i, n in enumerate((48, 49, 64, 65, 96, 97, 128))]
    steps += [[(i, [i], [0]) for i in range(n)] for n in (49, 97)]
    size = dict(streams=97, ctx=256, pages=400)
    got, k1, v1 = _run(model, cfg, True, steps, **size)
    assert set(rows) == taken
    took = len(rows)
    assert took == 2 * (len(taken) + len(taken & {49, 97}))
    want, k2, v2 = _run(model, cfg, False, steps, **size)
    assert len(rows) == took
    for a, b in zip(got, want):
        _close(a.float(), b.float())
    for a, b in ((k1, k2), (v1, v2)):
        _close(a[b != 0], b[b != 0])
        assert torch.equal(a != 0, b != 0)
