"""Growing several sequences at once leaves what growing them one by one
does, also when the pages run out on the way."""
import pytest
import torch

from ollamamq_amd.engine.kvcache import SequenceCache


def _cache(pages=20):
    c = SequenceCache(4, pages, 3, 40, torch.device("cpu"))
    return c, [c.alloc_slot() for _ in range(3)]


@pytest.mark.parametrize("lens", [(1, 1, 1), (4, 5, 9), (13, 1, 20),
                                  (3, 0, 17)])
def test_together(lens):
    one, slots = _cache()
    both, same = _cache()
    assert slots == same
    for n in (lens, [x + 3 for x in lens[:2]]):
        for slot, k in zip(slots, n):
            one.ensure(slot, k)
        both.ensure_all(list(zip(slots, n)))
        assert torch.equal(one.page_table, both.page_table)
        assert one.seq_lens == both.seq_lens
        assert one._free_pages == both._free_pages


@pytest.mark.parametrize("last,message", [(40, "out of pages"),
                                          (41, "exceeds max_ctx")])
def test_the_first_are_kept(last, message):
    c, (a, b, d) = _cache(9)
    with pytest.raises(RuntimeError, match=message):
        c.ensure_all([(a, 6), (b, last), (d, 4)])
    assert c.page_table[a, :2].tolist() == c._slot_pages[a]
    assert c.seq_lens == [6 if s == a else 0 for s in range(3)]
    assert c.free_page_count() == 7
    c.ensure(d, 28)
    assert c.page_table[d, :7].tolist() == c._slot_pages[d]


@pytest.mark.parametrize("slot", [-1, 3, 4])
def test_slots_that_there_are_none_of(slot):
    """Refused before anything is taken: a closed stream has the slot -1, and
    the last slot's pages are not its own."""
    c, (a, b, d) = _cache()
    c.ensure_all([(a, 6), (d, 4)])
    table, lens, free = c.page_table.clone(), list(c.seq_lens), \
        list(c._free_pages)
    for grow in (c.ensure_all, lambda w: c.grow(w, [], [])):
        with pytest.raises(IndexError):
            grow([(slot, 20)])
        assert torch.equal(c.page_table, table)
        assert c.seq_lens == lens and c._free_pages == free
