"""Sums of squares of rows that a product over tiles takes in parts.  Parts
that are whole numbers add up exactly in any order, so the result is bit for
bit that with one sum per row, whichever way they come: 16 bytes or 4 at a
time into a stage's place, past its end, or by another launch."""
from types import SimpleNamespace

import pytest
import torch

from ollamamq_amd.ops import hip


def parts_of(sq, nt, shift):
    """[M, nt] whole numbers whose sums are sq, `shift` floats into a buffer
    with NaN before and behind."""
    M = sq.shape[0]
    parts = torch.randint(0, 512, (M, nt), device="cuda").float()
    parts[:, 0] += sq - parts.sum(1)
    buf = torch.full((M * nt + 16,), float("nan"), device="cuda")
    out = buf[shift:shift + M * nt].view(M, nt)
    return out.copy_(parts)


# 28 and 32 of most tiles fill the last stage or pass its end, 60 and more do
# not fit beside some of them; 2500 rows take more than one round of blocks
@pytest.mark.gpu
@pytest.mark.parametrize("nt, shift", [
    (2, 0), (3, 0), (4, 0), (4, 1), (22, 0), (28, 0), (32, 0), (53, 0),
    (60, 0), (96, 2), (257, 0)])
@pytest.mark.parametrize("M", [1, 33, 257, 607, 2500])
def test_parts_of_rows(M, nt, shift):
    hip.require()
    torch.manual_seed(nt)
    N, K, nl, nkl, page = 1024, 256, 6, 1, 16
    x = torch.randn((M + 31) // 32 * 32 * K, device="cuda").bfloat16()
    w = torch.randn(N * K, device="cuda").mul_(K ** -0.5).bfloat16()
    sq = torch.randint(1 << 18, 1 << 20, (M,), device="cuda").float()
    parts = parts_of(sq, nt, shift)
    n_pages = -(-M // page)
    pos = torch.randperm(M, device="cuda").int()
    slot = torch.zeros_like(pos)
    cos, sin = torch.rand(2, n_pages * page, 64, device="cuda")
    table = torch.randperm(n_pages, device="cuda").int().view(1, -1)

    def outputs(plan, rstd, n):
        if plan[1] % 2 == 0:
            cache = SimpleNamespace(
                n_kv_heads=nkl, page_size=page, page_table=table,
                k_pool=torch.zeros(1, n_pages, nkl, page, 128, device="cuda",
                                   dtype=torch.bfloat16))
            cache.v_pool = torch.zeros_like(cache.k_pool)
            q = hip.tile_qkv_rope(x, w, M, N, K, None, cache, 0, pos, slot,
                                  cos, sin, nl, nkl, rstd, n, 1.0 / K, 1e-5,
                                  plan=plan)
            yield from (q[:, :nl * 128], cache.k_pool, cache.v_pool)
        if plan[:2] != hip.TILE_LEAST:
            act = hip.tile_gu(x, w, M, N, K, rstd, n, 1.0 / K, 1e-5,
                              plan=plan)
            yield act.view(-1, N // 16, 32, 8).transpose(1, 2) \
                .reshape(-1, N // 2)[:M]

    for tile in (*hip.TILES, hip.TILE_LEAST):
        plan = (*tile, 1)
        want = outputs(plan, sq, 1)
        for got, one in zip(outputs(plan, parts, nt), want):
            assert one.any() and torch.equal(got, one), plan


def eight_side_by_side(parts):
    """fp32 sums of rows as eight lanes add them up, and then the lanes."""
    parts = parts.cpu()
    lanes = torch.zeros(parts.shape[0], 8)
    for e in range(parts.shape[1]):
        lanes[:, e % 8] += parts[:, e]
    while lanes.shape[1] > 1:
        lanes = lanes[:, ::2] + lanes[:, 1::2]
    return lanes[:, 0].contiguous().cuda()


# 2^25 has no room for what is added to it before it is taken away again, so a
# sum in another order is another sum: only every eighth part may be together.
# Sums of 33 rows are added up by the product itself, of 20000, more than one
# round of blocks of every tile, by a kernel of their own.
@pytest.mark.gpu
@pytest.mark.parametrize("nt", [2, 9, 12, 16, 19, 22, 32, 53])
@pytest.mark.parametrize("M", [33, 20000])
def test_order_of_sums(M, nt):
    hip.require()
    torch.manual_seed(nt)
    N, K = 1024, 256
    x = torch.randn((M + 31) // 32 * 32 * K, device="cuda").bfloat16()
    w = torch.randn(N * K, device="cuda").mul_(K ** -0.5).bfloat16()
    parts = torch.rand(M, nt, device="cuda") * 100
    if nt > 8:
        parts[:, 0], parts[:, 8] = 2 ** 25, -2 ** 25
    for tile in hip.TILES:
        one, got = (hip.tile_gu(x, w, M, N, K, rstd, n, 1.0 / K, 1e-5,
                                plan=(*tile, 1)).view(-1, N // 16, 32, 8)
                    .transpose(1, 2).reshape(-1, N // 2)[:M]
                    for rstd, n in ((eight_side_by_side(parts), 1),
                                    (parts, nt)))
        assert one.any() and torch.equal(got, one), tile
