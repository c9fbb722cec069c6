"""Products of many rows over tiles (tile_gemm.hip) against float64."""
import math
import time
from types import SimpleNamespace

import pytest
import torch

from ollamamq_amd.ops import hip

SMALL = hip.TILE_LEAST
PLANS = [(*t, ks) for t in (*hip.TILES, SMALL) for ks in (1, 3)]


def test_plans_are_possible():
    """What is chosen is a tile that the kernel has and parts that K has."""
    for M in (1, 49, 64, 65, 129, 130, 300, 541, 2317, 8192):
        for N, K in ((64, 128), (448, 384), (4096, 14336), (37888, 3584)):
            for epi in (hip.TILE_RESIDUAL, hip.TILE_GATED, hip.TILE_ROPE):
                hm, hn, ks = hip.tile_plan(M, N, K, epi)
                unit = 256 if hm + hn <= 8 else 128
                assert (hm, hn) in (*hip.TILES, SMALL) and K % unit == 0
                assert (hm, hn) != SMALL or epi != hip.TILE_GATED
                assert 1 <= ks <= K // unit
                assert epi == hip.TILE_RESIDUAL or ks == 1
                assert epi != hip.TILE_ROPE or hn % 2 == 0


def estimate(M, N, K, epi, cus):
    """{(rows, columns, parts): us} of every plan that is weighed."""
    took = {}
    for hm, hn in hip.TILES:
        unit = 256 if hm + hn <= 8 else 128
        if K % unit or (epi == hip.TILE_ROPE and hn % 2):
            continue
        tiles, area = -(-M // (32 * hm)) * -(-N // (32 * hn)), hm * hn
        for ks in range(1, 9 if epi == hip.TILE_RESIDUAL else 2):
            if ks > 1 and (tiles * ks > 2.5 * cus or K // unit < 2 * ks):
                break
            slabs = -(-K // unit // ks) * unit / 32
            slab = max(area * 0.00715, hm * 0.0239 + hn * 0.0223)
            busiest = -(-tiles * ks // cus) * (slabs * slab + 2.6
                                               + area * 0.202)
            power = tiles * ks * area / cus * (slabs * 0.0079 + 0.202)
            t = (busiest ** 8 + power ** 8 + (N * K * 4e-7) ** 8) ** 0.125
            took[hm, hn, ks] = t + (3.0 + ks * M * N * 1.5e-6) * (ks > 1)
    return took


def test_plans_take_least():
    """The choice is the one that the estimate likes best; for a new number of
    rows it takes no more host time than a launch."""
    for cus in (32, 256, 304):
        for N, K in ((64, 128), (384, 1536), (4096, 14336), (6144, 4096),
                     (37888, 3584), (5120, 13824)):
            for M in (65, 129, 541, 1000, 2317, 8100):
                for epi in range(3):
                    took = estimate(M, N, K, epi, cus)
                    plan = hip.tile_plan(M, N, K, epi, cus)
                    assert took[plan] <= min(took.values()) * (1 + 1e-9)
    for cus, N, K, parts in ((256, 4096, 4096, 2), (256, 4096, 14336, 4),
                             (256, 64, 65536, 8), (64, 4096, 14336, 1),
                             (256, 512, 512, 1)):
        assert hip.tile_plan(64, N, K, hip.TILE_RESIDUAL, cus) == (
            *SMALL, parts)
        assert hip.tile_plan(64, N, K, hip.TILE_ROPE, cus) == (*SMALL, 1)
    times = []                          # 1.6 us; in Python 68
    for M in range(1000, 1301):
        t0 = time.perf_counter()
        hip.tile_plan(M, 4096, 14336, hip.TILE_RESIDUAL)
        times.append(time.perf_counter() - t0)
    assert sorted(times)[150] < 20e-6


def test_plans_refused():
    for bad in ((0, 64, 128), (129, 0, 128), (129, 64, 64), (129, 64, 192)):
        with pytest.raises(ValueError):
            hip.tile_plan(*bad, hip.TILE_GATED)


@pytest.mark.parametrize("cus", [32, 64, 256])
def test_plans_are_the_devices(cus, monkeypatch):
    """Tiles and parts are chosen for as many CUs as the device has, which is
    what the grid is sized for: a partition of a card has fewer."""
    seen = []
    monkeypatch.setattr(hip, "_cus", lambda index: cus)
    monkeypatch.setattr(
        hip, "_tile_gemm", lambda epi, y, x, packed, M, N, K, plan, **k:
        seen.append(plan))
    M, N, K = 300, 384, 1536
    x, w, y = torch.empty(320 * K), torch.empty(N * K), torch.empty(320 * N)
    cache = SimpleNamespace(page_size=16, k_pool=torch.empty(1, 1),
                            v_pool=torch.empty(1, 1),
                            page_table=torch.empty(1, 1).int())
    hip.tile_residual(x, w, M, N, K, y)
    hip.tile_gu(x, w, M, N, K, None, 1, 0.0, 0.0)
    hip.tile_qkv_rope(x, w, M, N, K, None, cache, 0, torch.empty(M).int(),
                      torch.empty(M).int(), None, None, 1, 1, None, 1, 0.0,
                      0.0)
    assert seen == [hip.tile_plan(M, N, K, epi, cus) for epi in
                    (hip.TILE_RESIDUAL, hip.TILE_GATED, hip.TILE_ROPE)]


def frag(x):
    rows = -(-x.shape[0] // 32) * 32
    f = x.new_full((rows, x.shape[1]), math.nan)   # what no row may see
    f[:len(x)] = x
    return f.view(rows // 32, 32, -1, 8).transpose(1, 2).flatten()


def unfrag(f, rows, cols):
    return f.view(-1, cols // 8, 32, 8).transpose(1, 2).reshape(-1, cols)[:rows]


def rand(*shape, scale=1.0):
    return (torch.randn(*shape, device="cuda") * scale).bfloat16()


def off(a, b):
    return ((a.double() - b).norm() / b.norm()).item()


# One rounding to bf16, half a step of 2^-7 at most of every value, of fp32 sums: K / 32 steps
# of up to K terms, together sqrt(K) times the result, each rounded to 2^-24 of
# it, are 2^-14 for K = 1024; twice that for the product of two such sums.
ROUNDED = 2 ** -8 + 2 ** -13


def near(got, want):
    """Every value, so that no store is missing or astray: that rounding, half
    a step of 2^-8 at most, and 2^-12 of values about 1 for what the sums are
    off by, 2^-24 of some sqrt(K) of them."""
    torch.testing.assert_close(got.double(), want, rtol=2 ** -8,
                               atol=2 ** -12)
    assert off(got, want) < ROUNDED


@pytest.mark.gpu
@pytest.mark.parametrize("plan", PLANS, ids=str)
@pytest.mark.parametrize("M, N, K", [
    (1, 64, 768), (32, 64, 768), (33, 448, 768), (129, 576, 768),
    (577, 64, 1024), (2500, 3072, 768), (2817, 6144, 768)])
def test_product(plan, M, N, K):
    """Rows and columns around the edges of tiles; the last in several rounds
    of blocks with every tile (288 of the largest)."""
    hip.require()
    torch.manual_seed(M + N)
    x, w, eps = rand(M, K), rand(N, K, scale=K ** -0.5), 1e-5
    xf, y = frag(x), x.double() @ w.double().T
    res = rand(M, N)
    rf = frag(res)
    sq, nt = hip.tile_residual(xf, hip.pack_weight(w), M, N, K, rf, plan=plan)
    near(unfrag(rf, M, N), y + res.double())
    # fp32 sums of squares of at most 2^13 values before their rounding
    assert sq.shape == (M, nt)
    squares = (y + res.double()).square().sum(1)
    assert off(sq.sum(1), squares) < 2 ** -18
    torch.testing.assert_close(sq.double().sum(1), squares, rtol=2 ** -16,
                               atol=0)
    if plan[2] > 1 or plan[:2] == SMALL:
        return
    for nt in (1, 3, 40):
        sq = (torch.rand(M, nt, device="cuda") + 0.5) * (K / nt)
        scale = (sq.double().sum(1) / K + eps).rsqrt()[:, None]
        for glu in ("silu", "gelu_tanh"):
            act = hip.tile_gu(xf, hip.pack_weight_gu(w), M, N, K, sq, nt,
                              1.0 / K, eps, glu, plan=plan)
            g, u = (y * scale).chunk(2, 1)
            g = (torch.nn.functional.silu(g) if glu == "silu" else
                 torch.nn.functional.gelu(g, approximate="tanh"))
            near(unfrag(act, M, N // 2), g * u)


@pytest.mark.gpu
@pytest.mark.parametrize("glu", ["silu", "gelu_tanh"])
def test_activation_is_the_chains(glu):
    """Sums of whole numbers are exact in any order, so what is left is the
    epilogue: bit for bit that of the weight stream.  A reciprocal off by a
    unit of fp32 turns one value of 2^16 to another bf16."""
    hip.require()
    torch.manual_seed(7)
    M, N, K = 128, 28672, 256
    x = torch.randint(-2, 3, (M, K), device="cuda").bfloat16()
    w = torch.randint(-1, 2, (N, K), device="cuda").bfloat16()
    # scales about 1/8, another for every row
    sq = (torch.rand(M, device="cuda") + 0.5) * 64 * K
    args = (frag(x), hip.pack_weight_gu(w))
    norm = dict(rstd=sq, rstd_nt=1, inv_h=1.0 / K, eps=1e-5, glu=glu)
    want = hip.linear_gu(*args, N, K=K, yfrag=1, M_frag=M, **norm)
    for plan in ((8, 8, 1), (9, 7, 1)):
        got = hip.tile_gu(*args, M, N, K, plan=plan, **norm)
        assert torch.equal(unfrag(got, M, N // 2), unfrag(want, M, N // 2))


@pytest.mark.gpu
@pytest.mark.parametrize("plan", [p for p in (*hip.TILES, SMALL)
                                  if p[1] % 2 == 0],
                         ids=str)
@pytest.mark.parametrize("M, nl, nkl, page, bias", [
    (1, 1, 1, 16, False), (131, 4, 2, 16, True), (300, 7, 1, 48, True),
    (2500, 32, 4, 64, False), (3400, 32, 4, 64, True)])
def test_rotated(plan, M, nl, nkl, page, bias):
    hip.require()
    torch.manual_seed(M)
    K, slots, eps = 256, 3, 1e-5
    N, per = (nl + 2 * nkl) * 128, -(-(M // slots + 9) // page)
    n_pages = slots * per + 1
    w = rand(N, K, scale=K ** -0.5)
    b = rand(N) if bias else None
    x = rand(M, K)
    # a buffer of its own for each, so that a stray write shows
    cache = SimpleNamespace(
        n_kv_heads=nkl, page_size=page,
        k_pool=torch.zeros(2, n_pages, nkl, page, 128, device="cuda",
                           dtype=torch.bfloat16),
        page_table=torch.randperm(n_pages, device="cuda")[:slots * per]
        .view(slots, per).int().contiguous())
    cache.v_pool = torch.zeros_like(cache.k_pool)
    pos = torch.arange(M, device="cuda").int() // slots + 5
    slot = torch.arange(M, device="cuda").int() % slots
    angle = torch.rand(per * page, 64, device="cuda") * 6
    cos, sin = angle.cos(), angle.sin()
    sq = (torch.rand(M, 9, device="cuda") + 0.5) * (K / 9)
    order = torch.tensor(hip.qkv_rope_order(nl, nkl), device="cuda")
    q = hip.tile_qkv_rope(
        frag(x), hip.pack_weight_qkv_rope(w, nl, nkl), M, N, K,
        b[order].contiguous() if bias else None, cache, 1, pos, slot, cos,
        sin, nl, nkl, sq, 9, 1.0 / K, eps, plan=(*plan, 1))
    y = x.double() @ w.double().T
    y *= (sq.double().sum(1) / K + eps).rsqrt()[:, None]
    if bias:
        y += b.double()
    wq, wk, wv = (t.unflatten(1, (-1, 128)) for t in
                  y.split([nl * 128, nkl * 128, nkl * 128], 1))

    def turn(t):
        c, s = (f[pos.long()].double()[:, None] for f in (cos, sin))
        lo, hi = t.chunk(2, -1)
        return torch.cat([lo * c - hi * s, hi * c + lo * s], -1)

    at = cache.page_table[slot.long(), pos.long() // page].long()
    place = pos.long() % page
    near(q[:, :nl * 128].unflatten(1, (-1, 128)), turn(wq))
    near(cache.k_pool[1][at, :, place], turn(wk))
    near(cache.v_pool[1][at, :, place], wv)
    for pool in (cache.k_pool, cache.v_pool):
        assert not pool[0].any()
        pool[1][at, :, place] = 0
        assert not pool[1].any()


def test_refused():
    lib = hip._lib if hip.available() else None
    if lib is None:
        pytest.skip("the extension is not built")
    none = [None] * 8

    def call(M=129, N=64, K=256, epi=0, hm=4, hn=4, ks=1):
        return lib.tile_gemm_bf16(*none, 1, 0.0, 0.0, M, N, K, epi, hm, hn,
                                  ks, 8, 8, 0, 256, *none[:7], 1, 1, 16, 1,
                                  None)
    for bad in (dict(M=0), dict(N=48), dict(K=128), dict(K=192, hm=9, hn=7),
                dict(ks=2), dict(epi=3, ks=2), dict(hm=5, hn=5), dict(epi=2)):
        assert call(**bad) < 0


def test_refused_scratch():
    """Scratch, sums and pieces that a product cannot do without, and
    epilogues that there are none of."""
    lib = hip._lib if hip.available() else None
    if lib is None:
        pytest.skip("the extension is not built")
    some = 1 << 20                      # nothing reads it

    def call(epi, part=some, rstd=some, rstd_nt=1, pieces=16):
        return lib.tile_gemm_bf16(
            some, part, some, some, None, some, some, rstd, rstd_nt, 0.0, 0.0,
            129, 384, 256, epi, 4, 4, 1, 8, pieces, 0, 256, *[some] * 7, 1, 1,
            16, 1, None)
    if not torch.cuda.is_available():   # nothing but the device is missing
        for epi in range(4):
            assert call(epi) > 0
    for bad in (dict(epi=3, pieces=0), dict(epi=3, pieces=-1),
                dict(epi=3, part=None), dict(epi=1, part=None, rstd_nt=3),
                dict(epi=2, part=None, rstd_nt=3), dict(epi=1, rstd_nt=0),
                dict(epi=2, rstd=None), dict(epi=-1), dict(epi=4)):
        assert call(**bad) < 0, bad
