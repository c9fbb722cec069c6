"""The switches that ask for another attention reach prompts of any length,
also those whose steps the fused chain would take."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _feed(model, cfg, steps):
    from ollamamq_amd.engine import LlamaEngine, PagedKVCache
    kv = PagedKVCache.for_model(cfg, n_pages=96, max_slots=6, max_ctx=256,
                                device="cuda:0", dtype=torch.bfloat16)
    eng = LlamaEngine(model, kv, max_batch=4)
    eng.use_graphs = False
    streams = [eng.open_stream() for _ in range(3)]
    return [eng.feed([(streams[i], list(t), list(w)) for i, t, w in step])
            for step in steps]


PROMPTS = [[(0, range(1, 41), [39])], [(1, range(140), [139, 3])]]
MIXED = [[(0, [7], [0]), (2, range(30), [29])]]


@pytest.mark.parametrize("name", ["tiny", "tiny-swa"])
def test_reference(name, monkeypatch):
    from ollamamq_amd.models import LlamaModel, PRESETS
    from ollamamq_amd.ops import interface
    cfg = PRESETS[name]
    model = LlamaModel(cfg, device="cuda:0", dtype=torch.bfloat16, seed=5)
    assert model.fused_chain
    monkeypatch.setenv("OLLAMAMQ_FORCE_REF", "1")

    def no(*a, **kw):
        raise AssertionError("a kernel where the reference is asked for")

    for f in ("attention_frag", "linear_fused", "fragify_sumsq"):
        monkeypatch.setattr(interface, f, no)
    got = _feed(model, cfg, PROMPTS + MIXED)
    model.fused_chain = False
    for a, b in zip(got, _feed(model, cfg, PROMPTS + MIXED)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("name", ["tiny", "tiny-swa"])
def test_valu_attention(name, monkeypatch):
    from ollamamq_amd.models import LlamaModel, PRESETS
    from ollamamq_amd.ops import hip
    cfg = PRESETS[name]
    model = LlamaModel(cfg, device="cuda:0", dtype=torch.bfloat16, seed=5)
    want = _feed(model, cfg, PROMPTS + MIXED)
    calls = []
    inner = hip._attention
    monkeypatch.setattr(hip, "_attention", lambda q, *a: (
        calls.append(len(q)), inner(q, *a))[1])
    monkeypatch.setenv("OLLAMAMQ_VALU_PREFILL", "1")
    got = _feed(model, cfg, PROMPTS + MIXED)
    # it predates windows, and single tokens beside prompts have no other
    # attention
    assert calls == ([] if cfg.sliding_window else
                     [40] * cfg.n_layers + [140] * cfg.n_layers)
    for a, b in zip(got, want):
        # roundings to bf16 at other places: two orders of summing differ by
        # up to 2^-6 of the logits' norm
        off = (a - b).float().square().mean().sqrt()
        assert off <= 2 ** -6 * b.float().square().mean().sqrt()

