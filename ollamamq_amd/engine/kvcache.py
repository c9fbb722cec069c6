"""Sequence memory sized for 288 GB HBM3E per MI355X: paged caches for
attention and per-slot state for recurrent layers.

SequenceCache owns what every model needs: sequence slots, the page pool's
free list and the int32 page table per slot.  Its subclasses add storage:

* PagedKVCache, layout [L, n_pages, KVH, page_size, D]: one (page, kv-head)
  is a contiguous page_size*D*2B run (4 KiB at page=16, D=128), the unit the
  decode-attention kernel streams with wide vector loads;
* HybridCache: one store per layer run of a model that mixes mechanisms --
  a paged pool with one latent row per token, paged keys and values of any
  width, and fp32 state per slot.

The reference has no KV concept (its context handling is only plumbing the
`num_ctx` option to Ollama, reference src/control.rs:804-806); the paged pool
is this framework's realization of "model loaded with context N" -- "load"
allocates weights + this pool in HBM, "unload" frees them.
"""
from __future__ import annotations

from dataclasses import dataclass
from typing import List, Optional, Tuple

import torch


class SequenceCache:
    """Slots and pages.  `scratch` adds one slot row and one page that no
    sequence ever gets: work that must not touch live state (graph warmups,
    batch padding) runs there."""

    scratch_slot: Optional[int] = None

    def __init__(self, page_size: int, n_pages: int, max_slots: int,
                 max_ctx: int, dev: torch.device, scratch: bool = False):
        self.page_size = page_size
        self.max_ctx = max_ctx
        max_pages = (max_ctx + page_size - 1) // page_size
        self.page_table = torch.zeros(
            (max_slots + scratch, max_pages), device=dev, dtype=torch.int32
        )
        if scratch:
            self.scratch_slot = max_slots
            self.page_table[max_slots].fill_(n_pages)
        self._free_pages: List[int] = list(range(n_pages - 1, -1, -1))
        self._free_slots: List[int] = list(range(max_slots - 1, -1, -1))
        self._slot_pages: List[List[int]] = [[] for _ in range(max_slots)]
        # host-side truth
        self.seq_lens = [0] * (max_slots + scratch)
        self.max_slots = max_slots
        self.n_pages = n_pages

    def free_page_count(self) -> int:
        return len(self._free_pages)

    def alloc_slot(self) -> int:
        if not self._free_slots:
            raise RuntimeError("KV cache: no free sequence slots")
        slot = self._free_slots.pop()
        self.seq_lens[slot] = 0
        return slot

    def free_slot(self, slot: int) -> None:
        self._free_pages.extend(self._slot_pages[slot])
        self._slot_pages[slot] = []
        self.seq_lens[slot] = 0
        self._free_slots.append(slot)

    def ensure(self, slot: int, new_len: int) -> None:
        """Grow slot's page list to cover new_len tokens."""
        self.ensure_all([(slot, new_len)])

    def ensure_all(self, wanted: List[Tuple[int, int]]) -> None:
        """Grow page lists to cover new_len tokens each, (slot, new_len)
        pairs.  New entries of the page table go to the device together, and
        nothing waits for what it still has to do."""
        places: List[int] = []
        values: List[int] = []
        try:
            self.grow(wanted, places, values)
        finally:
            table = self.page_table.view(-1)
            if len(places) == 1:
                table[places[0]] = values[0]
            elif places:
                both = torch.tensor([places, values], dtype=torch.int64)
                if table.is_cuda:
                    both = both.pin_memory()
                both = both.to(table.device, non_blocking=True)
                table.index_copy_(0, both[0], both[1].int())

    def grow(self, wanted: List[Tuple[int, int]], places: List[int],
             values: List[int]) -> None:
        """ensure_all without the device: adds the page table's new entries
        and where they go in the flat table.  What was grown before an error
        stays, and its entries are there.  Whether a slot is one of the
        cache's is asked here: on the device an entry outside the table is
        left out without a word."""
        width, size = self.page_table.shape[1], self.page_size
        for slot, new_len in wanted:
            if not 0 <= slot < self.max_slots:
                raise IndexError(f"KV cache: no sequence slot {slot}")
            if new_len > self.max_ctx:
                raise RuntimeError(
                    f"sequence exceeds max_ctx {self.max_ctx}")
            pages = self._slot_pages[slot]
            had = len(pages)
            if new_len > had * size:
                need = (new_len + size - 1) // size
                if need - had > len(self._free_pages):
                    raise RuntimeError("KV cache: out of pages")
                while len(pages) < need:
                    pages.append(self._free_pages.pop())
                places.extend(range(slot * width + had, slot * width + need))
                values.extend(pages[had:])
            self.seq_lens[slot] = new_len

    def can_fit(self, extra_tokens: int) -> bool:
        return len(self._free_pages) * self.page_size >= extra_tokens


class PagedKVCache(SequenceCache):
    def __init__(
        self,
        n_layers: int,
        n_kv_heads: int,
        head_dim: int,
        page_size: int = 16,
        n_pages: int = 1024,
        max_slots: int = 64,
        max_ctx: int = 8192,
        device: str = "cpu",
        dtype: torch.dtype = torch.float32,
    ):
        dev = torch.device(device)
        super().__init__(page_size, n_pages, max_slots, max_ctx, dev)
        self.head_dim = head_dim
        self.n_kv_heads = n_kv_heads
        shape = (n_layers, n_pages, n_kv_heads, page_size, head_dim)
        self.k_pool = torch.zeros(shape, device=dev, dtype=dtype)
        self.v_pool = torch.zeros(shape, device=dev, dtype=dtype)

    @classmethod
    def for_model(cls, cfg, tp_size=1, **kw):
        n_kv = max(1, cfg.n_kv_heads // tp_size)
        return cls(cfg.n_layers, n_kv, cfg.head_dim, **kw)


@dataclass(frozen=True)
class RunStore:
    """What one layer run keeps for a sequence: `latent` values per token in
    the paged pool (0: nothing), keys and values per token, `kv` = (heads,
    key width, value width), and named fp32 tensors of fixed shape."""
    latent: int = 0
    kv: Optional[Tuple[int, int, int]] = None
    state: Tuple[Tuple[str, Tuple[int, ...]], ...] = ()


class HybridCache(SequenceCache):
    """Storage for a model whose config lists a RunStore per layer run.

    Slots are reused without clearing: a layer takes its state as zero
    wherever a token's position is 0.
    """

    def __init__(
        self,
        stores: List[RunStore],
        page_size: int = 16,
        n_pages: int = 1024,
        max_slots: int = 64,
        max_ctx: int = 8192,
        device: str = "cpu",
        dtype: torch.dtype = torch.float32,
    ):
        dev = torch.device(device)
        super().__init__(page_size, n_pages, max_slots, max_ctx, dev,
                         scratch=True)
        self.latent_pool = [
            torch.zeros((n_pages + 1, page_size, s.latent), device=dev,
                        dtype=dtype) if s.latent else None for s in stores]
        # keys and values [pages, heads, page_size, width]; rows are filled
        # up with zeros to whole 8-element vectors
        self.key_pool, self.value_pool = (
            [torch.zeros((n_pages + 1, s.kv[0], page_size,
                          -(-s.kv[i] // 8) * 8), device=dev, dtype=dtype)
             if s.kv else None for s in stores] for i in (1, 2))
        self.state = [
            {name: torch.zeros((max_slots + 1, *shape), device=dev,
                               dtype=torch.float32)
             for name, shape in s.state} for s in stores]

    @classmethod
    def for_model(cls, cfg, tp_size=1, **kw):
        if tp_size != 1:
            raise ValueError(f"{cfg.name}: no tensor parallelism")
        return cls(cfg.run_stores(), **kw)


def cache_for_model(cfg, tp_size=1, **kw) -> SequenceCache:
    """The cache a model's config asks for."""
    cls = HybridCache if hasattr(cfg, "run_stores") else PagedKVCache
    return cls.for_model(cfg, tp_size=tp_size, **kw)
