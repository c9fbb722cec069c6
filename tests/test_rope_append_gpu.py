"""Rotary positions with the append to the paged pool: rows on 16 bytes, read
by vectors, and rows that are not, read one element at a time.

Tolerance: two fp32 products and their sum, rounded to bf16 once: 2^-8 of the
value (2^-9 doubled, as the sum's own error can cross a tie) and 1e-6 where the
terms cancel.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu
D = 128


def _turned(x, cos, sin):
    lo, hi = x.double().chunk(2, -1)
    c, s = cos.double()[:, None], sin.double()[:, None]
    return torch.cat((lo * c - hi * s, hi * c + lo * s), -1)


@pytest.mark.parametrize("T,Hq,KVH,page", [
    (1, 32, 8, 16), (1, 1, 1, 16), (5, 28, 4, 5), (37, 8, 8, 16),
    (130, 5, 1, 32)])
@pytest.mark.parametrize("first,row", [(0, 0), (1, 0), (8, 8), (0, 2), (2, 3)])
def test_rows(T, Hq, KVH, page, first, row):
    from ollamamq_amd.engine import PagedKVCache
    from ollamamq_amd.ops import hip
    hip.require()
    g = torch.Generator(device="cuda").manual_seed(2)
    W = (Hq + 2 * KVH) * D
    cache = PagedKVCache(2, KVH, D, page_size=page, n_pages=64, max_slots=2,
                         max_ctx=256, device="cuda", dtype=torch.bfloat16)
    cache.alloc_slot()
    slot = cache.alloc_slot()
    cache.ensure(slot, T + 3)
    buf = torch.randn(first + T * (W + row), generator=g,
                      device="cuda").bfloat16()
    kept = buf.clone()
    qkv = buf[first:].view(T, W + row)[:, :W]
    q, k, v = (p.unflatten(1, (-1, D)) for p in qkv.split(
        [Hq * D, KVH * D, KVH * D], 1))
    pos = torch.arange(3, T + 3, dtype=torch.int32, device="cuda")
    ang = torch.rand(T + 3, D // 2, generator=g, device="cuda") * 6.28
    cos, sin = ang.cos(), ang.sin()
    want_q = _turned(q, cos[3:], sin[3:])
    want_k, want_v = _turned(k, cos[3:], sin[3:]), v.clone()
    hip.rope_append(cache, 1, q, k, v, pos,
                    torch.full_like(pos, slot), cos, sin)
    close = dict(rtol=2 ** -8, atol=1e-6)
    torch.testing.assert_close(q.double(), want_q, **close)
    torch.testing.assert_close(k.double(), want_k, **close)
    pages = cache.page_table[slot].long()
    for pool, want in ((cache.k_pool, k), (cache.v_pool, want_v)):
        rows = pool[1][pages].transpose(1, 2).flatten(0, 1)
        assert torch.equal(rows[3:T + 3], want)
        assert not rows[:3].any() and not pool[0].any()
    # nothing beside the rows has changed
    qkv.copy_(kept[first:].view(T, W + row)[:, :W])
    assert torch.equal(buf, kept)
