"""The attention kernels of the Llama path at the edges of their tiles, against
float64.

Tolerance: the result is rounded once to bf16 (relative 2^-9, doubled for ties
and for sums of fp32 products), decode keeps weights in fp32; the absolute part
covers results that cancel: 128 to 4000 products of size one with errors of
2^-24 each.
"""
import pytest
import torch

from ollamamq_amd.engine.kvcache import PagedKVCache
from ollamamq_amd.ops.interface import AttnMeta

pytestmark = pytest.mark.gpu
D = 128


def _hip():
    from ollamamq_amd.ops import hip
    hip.require()
    return hip


def _cache(lens, heads, page, seed):
    cache = PagedKVCache(2, heads, D, page_size=page,
                         n_pages=sum(-(-n // page) for n in lens) + 2,
                         max_slots=len(lens) + 1, max_ctx=max(lens) + page,
                         device="cuda", dtype=torch.bfloat16)
    g = torch.Generator(device="cuda").manual_seed(seed)
    for pool in (cache.k_pool, cache.v_pool):
        pool.normal_(generator=g)
    slots = [cache.alloc_slot() for _ in lens]
    cache.alloc_slot()
    for at in range(0, max(lens), 3 * page):        # pages interleave
        for slot, n in zip(slots, lens):
            if at < n:
                cache.ensure(slot, min(n, at + 3 * page))
    return cache, slots


def _meta(slots, lens, q_lens, window, mode):
    def i32(v):
        return torch.tensor(v, dtype=torch.int32, device="cuda")
    cu = [0]
    for n in q_lens:
        cu.append(cu[-1] + n)
    return AttnMeta(mode=mode, slot_ids=i32(slots), seq_lens=i32(lens),
                    cu_q=i32(cu), logits_idx=None, max_q=max(q_lens),
                    max_kv=max(lens), window=window)


def _exact(q, cache, layer, slots, lens, q_lens, window):
    """q [T, Hq, D]; float64."""
    out, at = [], 0
    for slot, n, m in zip(slots, lens, q_lens):
        pages = cache.page_table[slot, :-(-n // cache.page_size)].long()
        k, v = (pool[layer][pages].transpose(1, 2).flatten(0, 1)[:n].double()
                for pool in (cache.k_pool, cache.v_pool))
        group = q.shape[1] // k.shape[1]
        k, v = (t.repeat_interleave(group, 1).transpose(0, 1).contiguous()
                for t in (k, v))
        pos = torch.arange(n - m, n, device="cuda")[:, None]
        key = torch.arange(n, device="cuda")[None]
        gone = key > pos
        if window:
            gone |= key <= pos - window
        x = q[at:at + m].double().transpose(0, 1).contiguous()
        s = (x @ k.transpose(1, 2).contiguous()) / D ** 0.5
        s = s.masked_fill(gone, float("-inf")).softmax(-1)
        out.append((s @ v).transpose(0, 1))
        at += m
    return torch.cat(out)


def _defrag(buf, rows, cols):
    x = buf.view(-1, cols // 64, 4, 2, 32, 8).permute(0, 4, 1, 2, 3, 5)
    return x.reshape(-1, cols)[:rows]


STEPS = [1, 15, 16, 17, 31, 32, 33, 64, 255, 256, 257, 511, 700]


@pytest.mark.parametrize("heads,kv_heads", [(1, 1), (6, 3), (3, 1), (8, 2),
                                            (5, 1), (6, 1), (14, 2), (16, 2)])
@pytest.mark.parametrize("page,window", [(16, 0), (64, 0), (16, 33),
                                         (24, 0), (8, 100)])
def test_decode(heads, kv_heads, page, window):
    hip = _hip()
    cache, slots = _cache(STEPS, kv_heads, page, 7)
    q = torch.randn(len(STEPS), heads, D, device="cuda").bfloat16()
    meta = _meta(slots, STEPS, [1] * len(STEPS), window, "decode")
    want = _exact(q, cache, 1, slots, STEPS, meta.q_lens or [1] * len(STEPS),
                  window)
    got = hip.attention_decode(q, cache, 1, meta)
    torch.testing.assert_close(got.double(), want, rtol=2 ** -8, atol=1e-5)
    frag = hip.attention_decode(q, cache, 1, meta, fragout=True)
    assert torch.equal(_defrag(frag, len(STEPS), heads * D),
                       got.flatten(1))


@pytest.mark.parametrize("page,window", [(16, 0), (64, 0), (5, 0), (24, 0),
                                         (33, 0), (16, 8225), (24, 8225)])
def test_decode_long_walks(page, window, monkeypatch):
    """More steps a wave than it looks up pages for at once, and as many."""
    hip = _hip()
    lens = [8160, 8192, 8193, 8225, 16385, 16640]
    cache, slots = _cache(lens, 2, page, 9)
    monkeypatch.setenv("OLLAMAMQ_DECODE_SPLIT", "1")
    q = torch.randn(len(lens), 8, D, device="cuda").bfloat16()
    ones = [1] * len(lens)
    want = _exact(q, cache, 1, slots, lens, ones, window)
    got = hip.attention_decode(q, cache, 1,
                               _meta(slots, lens, ones, window, "decode"))
    torch.testing.assert_close(got.double(), want, rtol=2 ** -8, atol=1e-5)


@pytest.mark.parametrize("S,heads,window", [
    (2, 2, 0), (64, 1, 0), (65, 1, 0), (129, 1, 0), (90, 2, 700), (30, 4, 0)])
def test_decode_even_shares(S, heads, window):
    """Parts by the lengths of all sequences, more than a wave has lanes too;
    tickets are zero again."""
    hip = _hip()
    lens = [(3000, 31, 1, 256, 257, 600, 1500, 33)[i * 3 % 8]
            for i in range(S)]
    cache, slots = _cache(lens, heads, 16, 11)
    assert hip._decode_split(S * heads, max(lens)) > 1
    q = torch.randn(S, 4 * heads, D, device="cuda").bfloat16()
    ones = [1] * S
    want = _exact(q, cache, 1, slots, lens, ones, window)
    sem = torch.zeros(S * heads, dtype=torch.int32, device="cuda")
    for _ in range(2):
        got = hip.attention_decode(
            q, cache, 1, _meta(slots, lens, ones, window, "decode"), sem=sem)
        torch.testing.assert_close(got.double(), want, rtol=2 ** -8,
                                   atol=1e-5)
        assert not sem.any()


@pytest.mark.parametrize("page", [16, 32, 64, 256, 8, 24])
@pytest.mark.parametrize("window", [0, 20])
def test_decode_reads_no_row_past_the_end(page, window):
    """What lies behind a context, in its last page and in others, is not a
    number; contexts end in every part of a step."""
    hip = _hip()
    lens = [1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 250, 257, 300]
    cache, slots = _cache(lens, 2, page, 13)
    for pool in (cache.k_pool, cache.v_pool):
        held = pool[1].clone()
        pool.fill_(float("nan"))
        for slot, n in zip(slots, lens):
            for at in range(0, n, page):
                p, m = cache.page_table[slot, at // page].long(), n - at
                pool[1, p, :, :m] = held[p, :, :m]
    q = torch.randn(len(lens), 8, D, device="cuda").bfloat16()
    ones = [1] * len(lens)
    want = _exact(q, cache, 1, slots, lens, ones, window)
    got = hip.attention_decode(q, cache, 1,
                               _meta(slots, lens, ones, window, "decode"))
    torch.testing.assert_close(got.double(), want, rtol=2 ** -8, atol=1e-5)


@pytest.mark.parametrize("split", [1, 2, 3, 32])
def test_decode_parts(split, monkeypatch):
    """Any number of parts, some of them without keys, and queries that lie
    anywhere in their projection."""
    hip = _hip()
    lens = [1, 200, 257, 3000, 8100]
    cache, slots = _cache(lens, 2, 16, 8)
    monkeypatch.setenv("OLLAMAMQ_DECODE_SPLIT", str(split))
    whole = torch.randn(len(lens), 11 * D + 3, device="cuda").bfloat16()
    for first, stride in ((0, 11 * D + 3), (1, 11 * D + 3), (8, 11 * D)):
        q = whole.flatten()[first:].as_strided((len(lens), 8, D),
                                               (stride, D, 1))
        meta = _meta(slots, lens, [1] * len(lens), 0, "decode")
        want = _exact(q, cache, 0, slots, lens, [1] * len(lens), 0)
        sem = torch.zeros(2 * len(lens), dtype=torch.int32, device="cuda")
        for tickets in (None, sem, sem, sem):       # given and shared
            got = hip.attention_decode(q, cache, 0, meta, sem=tickets)
            torch.testing.assert_close(got.double(), want, rtol=2 ** -8,
                                       atol=1e-5)
            assert not sem.any()


# queries, cached tokens before them
PORTIONS = [(1, 0), (2, 63), (31, 0), (32, 1), (33, 31), (64, 0), (65, 64),
            (127, 130), (200, 57), (300, 0)]


@pytest.mark.parametrize("heads,kv_heads", [(1, 1), (4, 2), (3, 1), (8, 2),
                                            (5, 1), (6, 1), (14, 2), (8, 1)])
@pytest.mark.parametrize("page,window", [(16, 0), (128, 0), (16, 1),
                                         (16, 40), (24, 0), (8, 129)])
def test_portions(heads, kv_heads, page, window):
    """Weights are rounded to bf16 before they meet the values: relative 2^-9
    of a sum of weighted values of size one, doubled for the result's own."""
    hip = _hip()
    q_lens = [m for m, _ in PORTIONS]
    lens = [m + n for m, n in PORTIONS]
    cache, slots = _cache(lens, kv_heads, page, 9)
    q = torch.randn(sum(q_lens), heads, D, device="cuda").bfloat16()
    meta = _meta(slots, lens, q_lens, window, "prefill")
    got = hip.attention_prefill(q, cache, 1, meta)
    want = _exact(q, cache, 1, slots, lens, q_lens, window)
    torch.testing.assert_close(got.double(), want, rtol=2 ** -8,
                               atol=2 ** -7)
    assert ((got - want).norm() / want.norm()).item() < 2 ** -8


@pytest.mark.parametrize("singles", [1, 5])
def test_single_tokens_before_portions(singles):
    hip = _hip()
    lens = [90 + 40 * i for i in range(singles)] + [70, 400]
    q_lens = [1] * singles + [70, 33]
    cache, slots = _cache(lens, 2, 16, 10)
    whole = torch.randn(sum(q_lens), 12 * D, device="cuda").bfloat16()
    q = whole[:, :8 * D].view(-1, 8, D)
    meta = _meta(slots, lens, q_lens, 0, "mixed")
    meta.n_decode = singles
    got = hip.attention_mixed(q, cache, 0, meta)
    want = _exact(q, cache, 0, slots, lens, q_lens, 0)
    torch.testing.assert_close(got.double(), want, rtol=2 ** -8,
                               atol=2 ** -7)
