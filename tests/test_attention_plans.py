"""Tiles of prompt attention, built on the host: every grouping of heads and
every first sequence has its own on one batch."""
import pytest
import torch

from ollamamq_amd.engine import PagedKVCache
from ollamamq_amd.ops import hip
from ollamamq_amd.ops.interface import AttnMeta


def _meta(q_lens, kv_lens, singles):
    cu = [0]
    for n in q_lens:
        cu.append(cu[-1] + n)
    i32 = dict(dtype=torch.int32)
    return AttnMeta(
        mode="mixed", slot_ids=torch.arange(len(q_lens), **i32),
        seq_lens=torch.tensor(kv_lens, **i32), cu_q=torch.tensor(cu, **i32),
        logits_idx=None, max_q=max(q_lens), max_kv=max(kv_lens),
        n_decode=singles)


def test_groupings_and_first_sequences_share_a_batch(monkeypatch):
    monkeypatch.setattr(hip, "upload", lambda values, dev: torch.tensor(
        values, dtype=torch.int32, device=dev))
    q_lens, kv_lens, singles = [1, 1, 70, 33, 300], [9, 40, 70, 80, 301], 2
    meta = _meta(q_lens, kv_lens, singles)
    starts = meta.cu_q.tolist()
    for first, G, KVH in [(0, 8, 1), (singles, 8, 1), (0, 1, 8), (0, 4, 2),
                          (singles, 1, 200), (0, 8, 1)]:
        tiles, waves = hip._prefill_plan(meta, first, G, KVH, "cpu")
        rows = set()
        for slot, tok, pos, row, n in tiles.tolist():
            assert tok == starts[slot] and 0 < n <= 32 * waves
            assert pos == kv_lens[slot] - q_lens[slot]
            rows.update((slot, r) for r in range(row, row + n))
        # each row of each portion, and none past its last token
        assert rows == {(s, r) for s in range(first, len(q_lens))
                        for r in range(q_lens[s] * G)}
        assert sum(n for *_, n in tiles.tolist()) == len(rows)
        again, _ = hip._prefill_plan(meta, first, G, KVH, "cpu")
        assert again is tiles


@pytest.mark.parametrize("singles, KVH, prompt, cus", [
    (12, 8, 40, 248), (12, 8, 200, 224),    # blocks of 256 rows of four heads
    (5, 32, 100, 192), (12, 8, 2047, 0),    # as many as there are CUs
    (8, 8, 40, 0), (24, 8, 40, 0)])         # no shares
def test_single_tokens_share_what_prompts_leave(singles, KVH, prompt, cus,
                                                monkeypatch):
    hip.require()
    seen = []

    class Spy:
        def mixed_attn_bf16(self, *args):
            seen.append(args)
            return 0
    monkeypatch.setattr(hip, "_lib", Spy())
    monkeypatch.setattr(hip, "_cus", lambda index: 256)
    monkeypatch.setattr(hip, "_stream", lambda: None)
    monkeypatch.setattr(hip, "upload", lambda values, dev: torch.tensor(
        values, dtype=torch.int32, device=dev))
    lens = [300 + 50 * i for i in range(singles)] + [prompt]
    meta = _meta([1] * singles + [prompt], lens, singles)
    cache = PagedKVCache(1, KVH, 128, page_size=16, n_pages=4, max_slots=64,
                         max_ctx=4096, device="cpu", dtype=torch.bfloat16)
    q = torch.zeros(singles + prompt, 4 * KVH, 128, dtype=torch.bfloat16)
    hip.attention_mixed(q, cache, 0, meta)
    n_items, S, split, least, got = seen[0][8], *seen[0][11:15]
    assert S == singles and least == (48 if singles * KVH >= 192 else 8)
    assert got == cus
    assert got in (0, 256 - n_items * KVH)
