"""Gated and rotated products over tiles in two launches: the same rows as in one.

Inputs are whole numbers, so sums are exact in any order and one launch and two
have to agree bit for bit."""
import pytest
import torch

from ollamamq_amd.ops import hip
from ollamamq_amd.ops.interface import FragRows

TWO = [[(0, 256, (8, 8, 1)), (256, 45, (4, 4, 1))],
       [(0, 32 * 9, (9, 7, 1)), (32 * 9, 13, (10, 4, 1))],
       [(0, 96, (4, 2, 1)), (96, 205, (8, 6, 1))]]
M, K = 301, 256


@pytest.mark.parametrize("cus", [32, 256, 304])
def test_plans_cover_the_rows(cus):
    """What is chosen has every row once, tiles that there are, and in the first
    launch whole tiles and rounds that are nearly full."""
    hip.require()
    two = 0
    for N, K in ((28672, 4096), (37888, 3584), (16384, 2048), (12288, 4096),
                 (384, 384)):
        for epi in (hip.TILE_GATED, hip.TILE_ROPE):
            for M in (1, 64, 128, 129, 541, 1399, 2310, 4161, 5903, 8100):
                plans = hip.tile_plans(M, N, K, epi, cus)
                at = 0
                for first, rows, (hm, hn, ks) in plans:
                    assert first == at and rows > 0 and ks == 1
                    assert (hm, hn) in (*hip.TILES, hip.TILE_LEAST)
                    assert K % (256 if hm + hn <= 8 else 128) == 0
                    assert epi != hip.TILE_ROPE or hn % 2 == 0
                    at += rows
                assert at == M and len(plans) <= 2
                if len(plans) == 1:
                    assert plans[0][2] == hip.tile_plan(M, N, K, epi, cus)
                    continue
                two += 1
                hm, hn, _ = plans[0][2]
                tiles = plans[0][1] // (32 * hm) * -(-N // (32 * hn))
                assert plans[0][1] % (32 * hm) == 0
                assert tiles >= 0.92 * cus * -(-tiles // cus)
    assert two
    for bad in ((129, 0, 128, 1, 256), (129, 64, 192, 1, 256),
                (129, 64, 128, 0, 256), (0, 64, 128, 1, 256),
                (129, 64, 128, 1, 0)):
        assert hip._lib.tile_gemm_split(*bad) == 0


@pytest.mark.parametrize("N, K, epi, M, plans", [
    # us in one launch and in two
    (28672, 4096, 1, 1600, [(9, 7), (7, 7)]),              # 296 283
    (28672, 4096, 1, 2310, [(9, 7), (7, 7)]),              # 449 412
    (28672, 4096, 1, 3000, [(9, 7), (8, 6)]),              # 539 522
    (37888, 3584, 1, 2310, [(9, 7), (7, 7)]),              # 510 488
    (22016, 4096, 1, 1600, [(7, 7), (8, 6)]),              # 247 232
    (22016, 4096, 1, 4500, [(7, 7), (8, 6)]),              # 633 610
    (6144, 4096, 2, 6451, [(8, 8), (8, 6)]),               # 9 % less in two
    # last rounds that are nearly full, or a launch's price
    (28672, 4096, 1, 541, [(9, 7)]), (28672, 4096, 1, 2048, [(8, 6)]),
    (28672, 4096, 1, 4500, [(9, 7)]), (28672, 4096, 1, 8100, [(8, 8)]),
    (37888, 3584, 1, 1600, [(9, 7)]), (37888, 3584, 1, 8100, [(8, 8)]),
    (22016, 4096, 1, 2310, [(6, 6)]), (6144, 4096, 2, 2310, [(8, 8)]),
    (12288, 4096, 2, 1600, [(10, 4)]), (12288, 4096, 2, 8100, [(8, 8)]),
])
def test_which_go_in_two(N, K, epi, M, plans):
    hip.require()
    assert (hip.TILE_GATED, hip.TILE_ROPE) == (1, 2)
    assert [p[2][:2] for p in hip.tile_plans(M, N, K, epi, 256)] == plans


def frag(x):
    rows = -(-x.shape[0] // 32) * 32
    f = x.new_zeros((rows, x.shape[1]))
    f[:len(x)] = x
    return f.view(rows // 32, 32, -1, 8).transpose(1, 2).flatten()


def whole(*shape):
    return torch.randint(-2, 3, shape, device="cuda").bfloat16()


@pytest.mark.gpu
@pytest.mark.parametrize("two", TWO)
@pytest.mark.parametrize("nt", [0, 1, 9])
def test_gated(two, nt, monkeypatch):
    hip.require()
    torch.manual_seed(nt)
    N = 448
    x, w = frag(whole(M, K)), hip.pack_weight_gu(whole(N, K))
    got = []
    for plans in ([(0, M, (8, 8, 1))], two):
        monkeypatch.setattr(hip, "tile_plans", lambda *a: plans)
        torch.manual_seed(1)
        if nt:
            sq = (torch.rand(M, nt, device="cuda") + 0.5) * K
            act = hip.tile_gu(x, w, M, N, K, sq, nt, 1.0 / K, 1e-5)
        else:                                   # normed already
            act = hip.tile_act(FragRows(x, M, K), w, N).buf
        rows = act.view(-1, N // 2 // 8, 32, 8).transpose(1, 2) \
            .reshape(-1, N // 2)[:M]
        got.append(rows.clone())
    assert got[0].abs().max() > 1 and torch.equal(*got)


@pytest.mark.gpu
@pytest.mark.parametrize("two", [TWO[0], TWO[2]])
def test_rotated(two, monkeypatch):
    from ollamamq_amd.engine import PagedKVCache
    hip.require()
    nl, nkl, nt = 3, 2, 5
    N = (nl + 2 * nkl) * 128
    x, w = frag(whole(M, K)), hip.pack_weight_qkv_rope(whole(N, K), nl, nkl)
    bias = whole(N)
    sq = (torch.rand(M, nt, device="cuda") + 0.5) * K
    ang = torch.rand(M + 3, 64, device="cuda") * 6
    pos = torch.arange(3, M + 3, device="cuda", dtype=torch.int32)
    got = []
    for plans in ([(0, M, (8, 8, 1))], two):
        monkeypatch.setattr(hip, "tile_plans", lambda *a: plans)
        cache = PagedKVCache(1, nkl, 128, n_pages=32, max_slots=1,
                             max_ctx=M + 3, device="cuda",
                             dtype=torch.bfloat16)
        slot = cache.alloc_slot()
        cache.ensure(slot, M + 3)
        q = hip.tile_qkv_rope(x, w, M, N, K, bias, cache, 0, pos,
                              torch.full_like(pos, slot), ang.cos(),
                              ang.sin(), nl, nkl, sq, nt, 1.0 / K, 1e-5)
        got.append([q[:, :nl * 128].clone(), cache.k_pool, cache.v_pool])
    for a, b in zip(*got):
        assert a.abs().max() > 1 and torch.equal(a, b)
