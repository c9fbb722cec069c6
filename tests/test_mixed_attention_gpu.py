"""Single tokens and portions of prompts in one launch: as each kind alone,
which other tests compare with float64.

A single token's sum is the same numbers in the same order, unless its context
goes in other parts: then fp32 sums in another order, and a rounding to bf16
(relative 2^-9) on either side.  A prompt's row shares its wave with the same
rows in blocks of any size, so it is the same bits.
"""
import pytest
import torch

from ollamamq_amd.engine import PagedKVCache
from ollamamq_amd.ops.interface import AttnMeta

pytestmark = pytest.mark.gpu
D = 128


def _meta(slots, q_lens, kv_lens, nd, window):
    i32 = dict(dtype=torch.int32, device="cuda")
    cu = [0]
    for n in q_lens:
        cu.append(cu[-1] + n)
    return AttnMeta(
        mode="mixed" if nd < len(slots) else "decode",
        slot_ids=torch.tensor(slots, **i32),
        seq_lens=torch.tensor(kv_lens, **i32), cu_q=torch.tensor(cu, **i32),
        logits_idx=None, max_q=max(q_lens), max_kv=max(kv_lens),
        n_decode=nd, window=window)


@pytest.mark.parametrize("Hq,KVH,page", [
    (32, 8, 16), (28, 4, 16), (8, 8, 32), (5, 1, 16), (8, 2, 5), (4, 4, 8)])
@pytest.mark.parametrize("window", [0, 70])
@pytest.mark.parametrize("singles,prompts", [
    ([300], [(37, 37)]),
    ([1, 16, 33, 500, 1100], [(2, 90), (130, 130), (65, 400)]),
    ([20] * 60, [(300, 300)]),
    ([1900, 5], [(2, 2)]),
    # prompts of 512 blocks and more go by themselves
    ([40, 900], [(2048, 2048), (2047, 2048)])])
def test_as_each_alone(Hq, KVH, page, window, singles, prompts):
    from ollamamq_amd.ops import hip
    hip.require()
    torch.manual_seed(6)
    q_lens = [1] * len(singles) + [n for n, _ in prompts]
    kv_lens = singles + [kv for _, kv in prompts]
    cache = PagedKVCache(2, KVH, D, page_size=page,
                         n_pages=sum(n // page + 1 for n in kv_lens),
                         max_slots=len(kv_lens), max_ctx=2064, device="cuda",
                         dtype=torch.bfloat16)
    slots = [cache.alloc_slot() for _ in kv_lens]
    for s, n in zip(slots, kv_lens):
        cache.ensure(s, n)
    cache.k_pool.normal_()
    cache.v_pool.normal_()
    T, nd = sum(q_lens), len(singles)
    qkv = torch.randn(T, (Hq + 2 * KVH) * D, device="cuda").bfloat16()
    q = qkv[:, :Hq * D].view(T, Hq, D)
    sem = torch.zeros(len(kv_lens) * KVH, dtype=torch.int32, device="cuda")
    alone = hip.attention_decode(
        q[:nd], cache, 1, _meta(slots[:nd], q_lens[:nd], kv_lens[:nd], nd,
                                window))
    rest = hip.attention_mixed(q[nd:], cache, 1, _meta(
        slots[nd:], q_lens[nd:], kv_lens[nd:], 0, window))
    for _ in range(3):
        got = hip.attention_mixed(q, cache, 1, _meta(
            slots, q_lens, kv_lens, nd, window), sem=sem)
        assert not sem.any()
        close = dict(rtol=0, atol=0) if hip._decode_split(
            nd * KVH, max(kv_lens)) == hip._decode_split(
            nd * KVH, max(singles)) else dict(rtol=2 ** -8, atol=1e-5)
        torch.testing.assert_close(got[:nd], alone, **close)
        assert torch.equal(got[nd:], rest)
    frag = hip.attention_mixed(q, cache, 1, _meta(
        slots, q_lens, kv_lens, nd, window), True, sem)
    if Hq * D % 64 == 0:
        frag = frag.view(-1, Hq * D // 64, 4, 2, 32, 8) \
            .permute(0, 4, 1, 2, 3, 5).reshape(-1, Hq, D)
        assert torch.equal(frag[:T], got)
    # rows that do not lie on 16 bytes
    odd = torch.empty(T * Hq * D + 1, dtype=q.dtype, device="cuda")[1:]
    odd = odd.view(T, Hq, D).copy_(q)
    again = hip.attention_mixed(odd, cache, 1, _meta(
        slots, q_lens, kv_lens, nd, window))
    assert torch.equal(again, got)


@pytest.mark.parametrize("S,KVH", [(48, 4), (25, 8), (40, 8), (61, 8)])
@pytest.mark.parametrize("window", [0, 1600])
def test_long_parts_of_many_users(S, KVH, window):
    """Between 192 and 511 pairs contexts of 96 steps and more go in parts of
    at least 48, against float64; tickets are zero again."""
    from ollamamq_amd.ops import hip
    hip.require()
    assert hip._decode_split(S * KVH, 4000) == (1 if S == 61 else 4)
    torch.manual_seed(7)
    G = 2
    lens = [(1, 1535, 1536, 1537, 3071, 3072, 3300, 40)[i % 8]
            for i in range(S)]
    cache = PagedKVCache(1, KVH, D, page_size=16,
                         n_pages=sum(n // 16 + 1 for n in lens), max_slots=S,
                         max_ctx=4000, device="cuda", dtype=torch.bfloat16)
    slots = [cache.alloc_slot() for _ in lens]
    for s, n in zip(slots, lens):
        cache.ensure(s, n)
    cache.k_pool.normal_()
    cache.v_pool.normal_()
    q = torch.randn(S, G * KVH, D, device="cuda").bfloat16()
    sem = torch.zeros(S * KVH, dtype=torch.int32, device="cuda")
    meta = _meta(slots, [1] * S, lens, S, window)
    first = None
    for _ in range(3):
        got = hip.attention_decode(q, cache, 0, meta, sem=sem)
        assert not sem.any()
        assert first is None or torch.equal(first, got)
        first = got
    for i, n in enumerate(lens):
        pages = cache.page_table[slots[i], :-(-n // 16)].long()
        k, v = (p[0][pages].transpose(1, 2).flatten(0, 1)[:n].double()
                for p in (cache.k_pool, cache.v_pool))
        lo = max(0, n - window) if window else 0
        s = torch.einsum("hgd,nhd->hgn", q[i].double().view(KVH, G, D),
                         k[lo:]) / D ** 0.5
        want = torch.einsum("hgn,nhd->hgd", s.softmax(-1), v[lo:])
        # one rounding to bf16, and fp32 sums
        torch.testing.assert_close(got[i].double(), want.flatten(0, 1),
                                   rtol=2 ** -8, atol=1e-5)


@pytest.mark.parametrize("singles,KVH", [(12, 8), (3, 32), (33, 4)])
@pytest.mark.parametrize("window", [0, 1600])
def test_even_shares_beside_a_prompt(singles, KVH, window):
    """Single tokens of 65 to 191 pairs beside a prompt: parts by the lengths of
    all single tokens, against float64; tickets are zero again."""
    from ollamamq_amd.ops import hip
    hip.require()
    torch.manual_seed(8)
    G, page = 2, 16
    lens = [300 + i * 2700 // (singles - 1) for i in range(singles)]
    q_lens, kv_lens = [1] * singles + [70], lens + [200]
    assert 64 < singles * KVH < 192
    assert hip._decode_split(singles * KVH, max(kv_lens)) > 1
    cache = PagedKVCache(1, KVH, D, page_size=page,
                         n_pages=sum(n // page + 1 for n in kv_lens),
                         max_slots=len(kv_lens), max_ctx=3072, device="cuda",
                         dtype=torch.bfloat16)
    slots = [cache.alloc_slot() for _ in kv_lens]
    for s, n in zip(slots, kv_lens):
        cache.ensure(s, n)
    cache.k_pool.normal_()
    cache.v_pool.normal_()
    q = torch.randn(sum(q_lens), G * KVH, D, device="cuda").bfloat16()
    sem = torch.zeros(len(kv_lens) * KVH, dtype=torch.int32, device="cuda")
    first = None
    for _ in range(2):
        got = hip.attention_mixed(q, cache, 0, _meta(
            slots, q_lens, kv_lens, singles, window), sem=sem)
        assert not sem.any()
        assert first is None or torch.equal(first, got)
        first = got
    for i, n in enumerate(lens):
        pages = cache.page_table[slots[i], :-(-n // page)].long()
        k, v = (p[0][pages].transpose(1, 2).flatten(0, 1)[:n].double()
                for p in (cache.k_pool, cache.v_pool))
        lo = max(0, n - window) if window else 0
        s = torch.einsum("hgd,nhd->hgn", q[i].double().view(KVH, G, D),
                         k[lo:]) / D ** 0.5
        want = torch.einsum("hgn,nhd->hgd", s.softmax(-1), v[lo:])
        # one rounding to bf16, and fp32 sums
        torch.testing.assert_close(got[i].double(), want.flatten(0, 1),
                                   rtol=2 ** -8, atol=1e-5)
