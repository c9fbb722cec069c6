"""A step's batch, its new pages and its plans go to the device together: the
same tensors as one by one, also when something fails on the way."""
from array import array

import numpy as np
import pytest
import torch

from ollamamq_amd.engine import LlamaEngine, cache_for_model
from ollamamq_amd.models import PRESETS, build_model
from ollamamq_amd.ops import hip, interface as ops
from ollamamq_amd.ops.interface import AttnMeta, Stage

WHERE = ["cpu", pytest.param("cuda:0", marks=pytest.mark.gpu)]
PARTS = [[], [5], array("i", range(16)), list(range(17)),
         [(1, 2, 3), (4, 5, 6)], [-1, 2 ** 31 - 1]]


@pytest.mark.parametrize("dev", WHERE)
def test_stage(dev):
    stage = Stage()
    later = [stage.add(p) for p in PARTS]
    sent = stage.send(torch.device(dev))
    for at, part in zip(later, PARTS):
        t = sent[at.index]
        assert t.dtype == torch.int32 and t.is_contiguous()
        assert t.data_ptr() % 64 == 0 or not len(part)
        assert t.tolist() == [list(p) if isinstance(p, tuple) else p
                              for p in part]


@pytest.mark.parametrize("dev", WHERE)
def test_entries(dev):
    table = torch.zeros(3, 400, dtype=torch.int32, device=dev)
    at = torch.randperm(1200, device=dev)[:700].int()
    ops.set_entries(table, at, at + 7)
    want = torch.zeros_like(table).view(-1)
    want[at.long()] = at + 7
    assert torch.equal(table.view(-1), want)
    if table.is_cuda:                   # entries that there are none of
        bad = torch.tensor([-1, 1200, 2 ** 31 - 1], dtype=torch.int32,
                           device=dev)
        ops.set_entries(table, bad, bad)
        assert torch.equal(table.view(-1), want)


@pytest.mark.parametrize("dev", WHERE)
@pytest.mark.parametrize("name", ["tiny", "kavedra-tiny"])
def test_plans_are_those_made_one_by_one(dev, name, monkeypatch):
    """A mixed batch: whatever the forward plans was sent before it."""
    cfg = PRESETS[name]
    dtype = torch.float32 if dev == "cpu" else torch.bfloat16
    model = build_model(cfg, device=dev, dtype=dtype, seed=1)
    kv = cache_for_model(cfg, n_pages=64, max_slots=6, max_ctx=256,
                         device=dev, dtype=dtype)
    eng = LlamaEngine(model, kv, max_batch=4)
    a, b, c = (eng.open_stream() for _ in range(3))
    eng.feed([(a, list(range(9)), [8])])
    seen = []
    forward = model.forward

    def spy(tokens, positions, cache, slots, meta, **k):
        plans = {n: v for n, v in vars(meta).items() if n[0] == "_"}
        lazy = AttnMeta(**{f: getattr(meta, f) for f in
                           AttnMeta.__dataclass_fields__})
        assert meta.stage is None
        model.plan(cache, lazy)
        seen.append((plans, {n: v for n, v in vars(lazy).items()
                             if n[0] == "_"}))
        return forward(tokens, positions, cache, slots, meta, **k)
    monkeypatch.setattr(model, "forward", spy)
    eng.feed([(a, [3], [0]), (b, list(range(70)), [69]),
              (c, list(range(33)), [32])])

    def same(x, y):
        if isinstance(x, torch.Tensor):
            return torch.equal(x, y)
        if isinstance(x, (tuple, list)):
            return len(x) == len(y) and all(map(same, x, y))
        return x == y
    for plans, lazy in seen:
        assert plans.keys() == lazy.keys()
        assert bool(plans) == (dev != "cpu")
        assert all(same(plans[n], lazy[n]) for n in plans)


@pytest.mark.parametrize("fails", ["pages", "plan"])
def test_pages_are_in_the_table_after_an_error(fails, monkeypatch):
    cfg = PRESETS["tiny"]
    model = build_model(cfg, device="cpu", dtype=torch.float32, seed=1)
    kv = cache_for_model(cfg, n_pages=9, max_slots=4, max_ctx=256,
                         device="cpu", dtype=torch.float32)
    eng = LlamaEngine(model, kv, max_batch=4)
    a, b = eng.open_stream(), eng.open_stream()
    long_ = 200 if fails == "pages" else 40

    def broken(*_):
        raise ValueError("no plan")
    if fails == "plan":
        monkeypatch.setattr(model, "plan", broken)
    with pytest.raises(RuntimeError if fails == "pages" else ValueError):
        eng.feed([(a, list(range(20)), [0]), (b, list(range(long_)), [0])])
    for s in (a, b):
        pages = kv._slot_pages[s.slot]
        assert len(pages) == (2 if s is a else 0 if fails == "pages" else 3)
        assert kv.page_table[s.slot, :len(pages)].tolist() == pages


@pytest.mark.parametrize("dev", WHERE)
def test_tokens_are_what_a_tensor_takes(dev):
    """Numbers of any type, of which the whole part counts; RuntimeError where
    they are too large."""
    cfg = PRESETS["tiny"]
    dtype = torch.float32 if dev == "cpu" else torch.bfloat16
    model = build_model(cfg, device=dev, dtype=dtype, seed=1)
    kv = cache_for_model(cfg, n_pages=9, max_slots=4, max_ctx=64, device=dev,
                         dtype=dtype)
    eng = LlamaEngine(model, kv, max_batch=4)
    want = None
    for text in ([3, 1, 4], [3.0, 1.5, 4.0], list(np.array([3., 1., 4.])),
                 [3, torch.tensor(1), True + 3]):
        s = eng.open_stream()
        got = eng.feed([(s, text, [0, 2])])
        eng.close_stream(s)
        want = got if want is None else want
        assert torch.equal(got, want)
    for bad in ([2 ** 31], [1.0, 2.0 ** 40]):
        s = eng.open_stream()
        with pytest.raises(RuntimeError):
            eng._forward([s], bad, [0], [len(bad)], "prefill")
        eng.close_stream(s)
