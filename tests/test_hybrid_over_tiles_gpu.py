"""Products over tiles whose rows are normed already, and a Kavedra model's
prompts of more tokens than the weight streams take over them: against float64
and against the general path.

Tolerance of the latter: that of test_hybrid_short_prompts_gpu.py, for roundings
of six layer runs instead of four: sqrt(6 / 4) times as much."""
import dataclasses

import pytest
import torch

from ollamamq_amd.models import KavedraConfig, build_model
from ollamamq_amd.models.hybrid import RopeSpec
from ollamamq_amd.models.kavedra import KavedraLayerSpec
from ollamamq_amd.ops import hip
from ollamamq_amd.ops.interface import FragRows
from test_hybrid_short_prompts_gpu import _run
from test_tile_gemm_gpu import frag, near, rand, unfrag


@pytest.mark.gpu
@pytest.mark.parametrize("tile", hip.TILES, ids=str)
@pytest.mark.parametrize("M, N, K", [
    (1, 64, 768), (33, 448, 768), (129, 576, 768), (577, 64, 1024),
    (2817, 6144, 768)])
def test_product(tile, M, N, K):
    """Rows and columns around the edges of tiles, the last in several rounds
    of blocks."""
    hip.require()
    torch.manual_seed(M + N)
    x, w = rand(M, K), rand(N, K, scale=K ** -0.5)
    xf, y = FragRows(frag(x), M, K), x.double() @ w.double().T
    pk = hip.pack_weight(w)
    near(hip.tile_linear(xf, pk, N, plan=(*tile, 1)), y)
    for ks in (1, 3):
        parts = hip.tile_linear(xf, pk, N, f32=True, plan=(*tile, ks)).parts
        assert parts.shape == (ks, M, N)
        # fp32 sums of sqrt(K) times the result, K / 32 of them, each off by
        # 2^-24 of it: 2^-14 of values about 1, twice that is allowed
        torch.testing.assert_close(parts.double().sum(0), y, rtol=2 ** -13,
                                   atol=2 ** -13)
    for glu in ("silu", "gelu_tanh"):
        act = hip.tile_act(xf, hip.pack_weight_gu(w), N, glu, (*tile, 1))
        assert (act.rows, act.cols) == (M, N // 2)
        g, u = y.chunk(2, 1)
        g = (torch.nn.functional.silu(g) if glu == "silu" else
             torch.nn.functional.gelu(g, approximate="tanh"))
        near(unfrag(act.buf, M, N // 2), g * u)


@pytest.mark.parametrize("dev", [
    "cpu", pytest.param("cuda:0", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("M", [1, 64, 65, 128, 129])
def test_own_plan(M, dev, monkeypatch):
    """Without a plan a product takes tiles that there are for its results,
    also of as few rows as others have smaller ones for."""
    hip.require()
    torch.manual_seed(M)
    N, K = 576, 8192
    x = torch.randn(M, K).bfloat16()
    w = torch.randn(N, K).mul_(K ** -0.5).bfloat16()
    plans, product = [], hip._tile_rows
    if dev == "cpu":
        monkeypatch.setattr(hip, "_cus", lambda index: 256)

    def spy(epi, y, x, packed, N, plan, *a, **k):
        plans.append(plan)
        if dev != "cpu":
            product(epi, y, x, packed, N, plan, *a, **k)
    monkeypatch.setattr(hip, "_tile_rows", spy)
    xf = FragRows(frag(x.to(dev)), M, K)
    pk = hip.pack_weight(w.to(dev)) if dev != "cpu" else w.flatten()
    got = [hip.tile_linear(xf, pk, N, most=8), hip.tile_linear(xf, pk, N),
           hip.tile_linear(xf, pk, N, 8, True)]
    assert len(plans) == 3 and all(p[:2] in hip.TILES for p in plans)
    if dev != "cpu":
        y = x.double() @ w.double().T
        for out in got:
            if not isinstance(out, torch.Tensor):
                out = out.parts.sum(0)
            near(out.cpu(), y)


def test_refused():
    lib = hip._lib if hip.available() else None
    if lib is None:
        pytest.skip("the extension is not built")
    some = 1 << 20                      # nothing reads it

    def call(y=some, part=some, M=129, N=64, K=256, epi=hip.TILE_ROWS, hm=4,
             hn=4, ks=1, gm=8):
        return lib.tile_rows_bf16(y, part, some, some, M, N, K, epi, hm, hn,
                                  ks, gm, 0, 256, None)
    for bad in (dict(M=0), dict(N=48), dict(N=0), dict(K=128), dict(ks=2),
                dict(ks=0), dict(gm=0), dict(hm=2, hn=2), dict(hm=5, hn=5),
                dict(y=None), dict(y=None, epi=hip.TILE_GATED),
                dict(part=None, epi=hip.TILE_ROW_PARTS),
                dict(epi=hip.TILE_ROW_PARTS, ks=2),
                *(dict(epi=e) for e in (-1, 0, 2, 3, 6))):
        assert call(**bad) < 0, bad


def _config(vdim=32):
    rope = RopeSpec(16, 1e4)
    kinds = {
        "s": KavedraLayerSpec("lightning", 4, 24, vdim,
                              decay=(0.5, 0.9, 0.99, 0.999), ff=200),
        "a": KavedraLayerSpec("attention", 4, 32, vdim, kv_heads=2, scale=0.2,
                              rope=rope, ff=200),
        "l": KavedraLayerSpec("latent_attention", 4, 16, vdim, kv_rank=48,
                              rot_dim=16, scale=0.17, window=50, ff=200,
                              rope=rope)}
    return KavedraConfig(name="many", width=256, vocab=320,
                         layers=[kinds[c] for c in "slsa"], logit_scale=0.5,
                         loop=(1, 3, 2), max_ctx=512)


def _close(a, b, alike=True):
    size = b.square().mean().sqrt() * 1.5 ** 0.5
    off = (a - b).abs()
    assert off.square().mean().sqrt() <= 2 ** -6.2 * size
    assert not alike or off.max() <= 8 * 2 ** -7.2 * size


STEPS = [
    # one row more than the streams take
    [(0, range(129), [128])],
    # the first eight rows of 64 blocks that lie apart, and blocks beyond
    [(1, range(200), [199, 0, 63, 64])],
    [(2, range(3, 303), [299]), (3, range(9), [8]), (0, [5], [0])],
    # single tokens of many, and all places of a prompt
    [(i, [i + 2], [0]) for i in range(90)] + [(91, range(77), range(77))],
    # more places than the streams take
    [(4, range(150), [3] * 130)],
    # decode of more than the streams take is the general path
    [(i, [i + 2], [0]) for i in range(129)],
]


@pytest.mark.gpu
def test_prompts_against_general_path(monkeypatch):
    cfg = _config()
    model = build_model(cfg, device="cuda:0", dtype=torch.bfloat16, seed=3)
    assert model.frag_decode and model.whole_heads
    rows, product = [], hip._tile_rows

    def spy(epi, y, x, *a, **k):
        rows.append((epi, x.rows))
        product(epi, y, x, *a, **k)
    monkeypatch.setattr(hip, "_tile_rows", spy)
    got = _run(model, cfg, True, STEPS)
    many = {129, 200, 310, 167, 150}
    for epis in ((hip.TILE_ROWS, hip.TILE_ROW_PARTS), (hip.TILE_GATED,),
                 (hip.TILE_ROW_PARTS,)):
        assert {n for epi, n in rows if epi in epis} == many
    took = len(rows)
    want = _run(model, cfg, False, STEPS)
    assert len(rows) == took
    for a, b, step in zip(got[0], want[0], STEPS):
        assert a.shape == b.shape == (sum(len(w) for _, _, w in step),
                                      cfg.vocab)
        _close(a.float(), b.float())
    for i, (mine, theirs) in enumerate(zip(got[1:], want[1:])):
        for a, b in zip(mine, theirs):
            if a is not None:
                a, b = a[:400].float(), b[:400].float()
                there = b.any(-1)
                assert torch.equal(a.any(-1), there)
                _close(a[there], b[there], alike=i < 3)


@pytest.mark.gpu
@pytest.mark.parametrize("change", [dict(vdim=20), dict(width=192), "switch"],
                         ids=str)
def test_what_stays_general(change, monkeypatch):
    """Heads that are not whole vectors, products that are not whole tiles,
    and the switch that asks for the library."""
    cfg = _config(20 if change == dict(vdim=20) else 32)
    if change == dict(width=192):
        cfg = dataclasses.replace(cfg, width=192)
    elif change == "switch":
        monkeypatch.setattr(hip, "USE_WSTREAM", False)
    model = build_model(cfg, device="cuda:0", dtype=torch.bfloat16, seed=3)
    monkeypatch.setattr(hip, "_tile_rows", None)
    got = _run(model, cfg, True, STEPS[:1])
    want = _run(model, cfg, False, STEPS[:1])
    for a, b in zip(got[0], want[0]):
        # but for the logits' product: see test_hybrid_short_prompts_gpu.py
        torch.testing.assert_close(a, b, rtol=2 ** -7, atol=1e-4)


@pytest.mark.gpu
def test_heads_that_are_not_whole_vectors_stay_general(monkeypatch):
    """All of whose products would go over tiles: 32 heads of 20 are 640."""
    rope, wide = RopeSpec(16, 1e4), dict(ff=200)
    decay = tuple(0.5 + 0.015 * i for i in range(32))
    kinds = {
        "s": KavedraLayerSpec("lightning", 32, 24, 20, decay=decay, **wide),
        "a": KavedraLayerSpec("attention", 32, 32, 20, kv_heads=16, scale=0.2,
                              rope=rope, **wide),
        "l": KavedraLayerSpec("latent_attention", 32, 16, 20, kv_rank=48,
                              rot_dim=16, scale=0.17, window=50, rope=rope,
                              **wide)}
    cfg = KavedraConfig(name="many", width=256, vocab=320,
                        layers=[kinds[c] for c in "slsa"], logit_scale=0.5,
                        loop=(1, 3, 2), max_ctx=512)
    model = build_model(cfg, device="cuda:0", dtype=torch.bfloat16, seed=3)
    assert model.frag_decode and model.tiles_take(129)
    assert not model.whole_heads
    monkeypatch.setattr(hip, "_tile_rows", None)
    got = _run(model, cfg, True, STEPS[:1])
    want = _run(model, cfg, False, STEPS[:1])
    for a, b in zip(got[0], want[0]):
        # but for the logits' product: see test_hybrid_short_prompts_gpu.py
        torch.testing.assert_close(a, b, rtol=2 ** -7, atol=1e-4)
