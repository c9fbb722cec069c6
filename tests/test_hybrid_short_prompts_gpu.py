"""A Kavedra model's steps of few tokens keep their activations in fragment
layout whatever they are made of: the same logits and state as the general
path.

Tolerance: both paths round the operands of every product to bf16; the general
one also rounds most products' results, some 8 roundings a layer run and path,
each off by 2^-9 / sqrt(3) of a value's size in the mean: sqrt(4 * 2 * 8) of
them are 2^-7.2 of the logits' norm; twice that is allowed.  Single values
differ like normal ones: of 30000 the furthest lies 4.5 times the mean off, 8
are allowed.
"""
import pytest
import torch

from ollamamq_amd.engine import LlamaEngine, cache_for_model
from ollamamq_amd.models import KavedraConfig, build_model
from ollamamq_amd.models.hybrid import RopeSpec
from ollamamq_amd.models.kavedra import KavedraLayerSpec

pytestmark = pytest.mark.gpu


def _config(vdim=32):
    rope = RopeSpec(16, 1e4)
    kinds = {
        "s": KavedraLayerSpec("lightning", 4, 24, vdim,
                              decay=(0.5, 0.9, 0.99, 0.999), ff=200),
        "a": KavedraLayerSpec("attention", 4, 32, vdim, kv_heads=2, scale=0.2,
                              rope=rope, ff=200),
        "l": KavedraLayerSpec("latent_attention", 4, 24, vdim, kv_rank=40,
                              rot_dim=16, scale=0.17, window=50, ff=200,
                              rope=rope)}
    return KavedraConfig(name="few", width=192, vocab=320,
                         layers=[kinds[c] for c in "slsa"], logit_scale=0.5,
                         max_ctx=512)


def _close(a, b, alike=True):
    size = b.square().mean().sqrt()
    off = (a - b).abs()
    assert off.square().mean().sqrt() <= 2 ** -6.2 * size
    assert not alike or off.max() <= 8 * 2 ** -7.2 * size


def _run(model, cfg, frag, steps):
    was, model.frag_decode = model.frag_decode, frag
    kv = cache_for_model(cfg, n_pages=400, max_slots=130, max_ctx=512,
                         device="cuda:0", dtype=torch.bfloat16)
    eng = LlamaEngine(model, kv, max_batch=4)
    eng.use_graphs = False
    streams = [eng.open_stream() for _ in range(130)]
    out = [eng.feed([(streams[i], list(t), list(w)) for i, t, w in step])
           for step in steps]
    model.frag_decode = was
    state = [s["lightning"] for s in kv.state if s]
    return out, kv.key_pool, kv.value_pool, kv.latent_pool, state


STEPS = [
    # one portion; all places wanted; 17 of them attend in latent space
    [(0, range(77), [76])],
    [(0, range(9, 137), range(128))],
    [(0, range(17), [0, 16])],
    # portions of every length and single tokens, unsorted
    [(1, range(3, 43), [39, 2, 2]), (0, [5], [0]), (2, range(2), [1]),
     (3, range(9), [8]), (4, [7], [0]), (5, range(20, 66), [45])],
    [(1, range(5), [4]), (6, range(123), [122])],
    # one token too many, and more places than fit
    [(7, range(129), [128])],
    [(8, range(12), [3] * 130)],
    # single tokens of many
    [(i, [i + 2], [0]) for i in range(65)],
    [(i, [i + 2], [0]) for i in range(128)],
    [(i, [i + 2], [0]) for i in range(129)],
]


@pytest.mark.parametrize("vdim", [32, 48])
def test_few_tokens(vdim):
    cfg = _config(vdim)
    model = build_model(cfg, device="cuda:0", dtype=torch.bfloat16, seed=3)
    assert model.frag_decode and model.whole_heads
    got = _run(model, cfg, True, STEPS)
    want = _run(model, cfg, False, STEPS)
    for a, b, step in zip(got[0], want[0], STEPS):
        assert a.shape == b.shape == (sum(len(w) for _, _, w in step),
                                      cfg.vocab)
        _close(a.float(), b.float())
    for i, (mine, theirs) in enumerate(zip(got[1:], want[1:])):
        for a, b in zip(mine, theirs):
            if a is not None:
                a, b = a[:400].float(), b[:400].float()
                # rows that were never written are zero, and not of the mean
                there = b.any(-1)
                assert torch.equal(a.any(-1), there)
                # a state's size goes with its head's memory
                _close(a[there], b[there], alike=i < 3)


def test_heads_of_odd_width():
    """Heads that are not whole vectors take the general path for prompts, as
    before."""
    cfg = _config(20)
    cfg = KavedraConfig(**{**cfg.__dict__, "layers": [
        KavedraLayerSpec(**{**s.__dict__, "heads": 16, "decay": (
            [0.9] * 16 if s.type == "lightning" else s.decay)})
        for s in cfg.layers]})
    model = build_model(cfg, device="cuda:0", dtype=torch.bfloat16, seed=3)
    assert model.frag_decode and not model.whole_heads
    got = _run(model, cfg, True, STEPS[:2])
    want = _run(model, cfg, False, STEPS[:2])
    # the same but for the logits' product, whose fp32 sums round to the same
    # bf16 number or a neighbour, at most 2^-7 away
    for a, b in zip(got[0], want[0]):
        torch.testing.assert_close(a, b, rtol=2 ** -7, atol=1e-4)
