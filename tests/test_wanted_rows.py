"""Logits are those of the rows that a step's layout names; a row that the
step does not have is an error, or NaN where only the device knows it."""
import pytest
import torch

from ollamamq_amd.ops.interface import AttnMeta

BAD = [[5], [0, 5], [-6], [0, -1, 99], [2 ** 40]]


def _meta(mode, dev, lens, q_lens, idx, **kw):
    i32 = dict(dtype=torch.int32, device=dev)
    cu = [0]
    for n in q_lens:
        cu.append(cu[-1] + n)
    return AttnMeta(
        mode=mode, slot_ids=torch.arange(len(lens), **i32),
        seq_lens=torch.tensor(lens, **i32), cu_q=torch.tensor(cu, **i32),
        logits_idx=torch.tensor(idx, dtype=torch.long, device=dev),
        max_q=max(q_lens), max_kv=max(lens), **kw)


@pytest.mark.parametrize("host", [False, True])
def test_check(host):
    def check(idx, mode="prefill", n=5):
        _meta(mode, "cpu", [5], [5], idx,
              rows=idx if host else None).check_rows(n)

    for idx in ([0], [-5, 4], [4, 4, -1, 0], []):
        check(idx)
    for idx in BAD:
        with pytest.raises(IndexError):
            check(idx)
        if host:
            with pytest.raises(IndexError):
                check(idx, "decode")
        else:
            check(idx, "decode")       # the kernels' to tell


@pytest.mark.gpu
@pytest.mark.parametrize("H", [64, 512])
def test_kernels(H):
    from ollamamq_amd.ops import hip
    hip.require()
    x, y = torch.randn(2, 5, H, device="cuda").bfloat16()
    xf, _ = hip.fragify_sumsq(x)
    idx = torch.tensor([0, 5, 4, -6, -5, -1, 2 ** 40, -2 ** 40, 3],
                       device="cuda")
    bad = (idx < -5) | (idx >= 5)
    for _, sq in (hip.frag_rows(xf, idx, H, 5),
                  hip.fragify_sumsq(x, rows=idx, add=y)):
        assert torch.equal(sq.isnan(), bad)


def _model(name="tiny"):
    from ollamamq_amd.models import LlamaModel, PRESETS
    model = LlamaModel(PRESETS[name], device="cuda:0", dtype=torch.bfloat16,
                       seed=5)
    assert model.fused_chain
    return model


def _cache(model, slots):
    from ollamamq_amd.engine import PagedKVCache
    kv = PagedKVCache.for_model(model.cfg, n_pages=slots * 10 + 8,
                                max_slots=slots, max_ctx=160, device="cuda:0",
                                dtype=torch.bfloat16)
    for _ in range(slots):
        kv.alloc_slot()
    return kv


@pytest.mark.gpu
@pytest.mark.parametrize("T", [5, 140])
@pytest.mark.parametrize("host", [False, True])
def test_refused(T, host):
    model = _model()
    kv = _cache(model, 1)
    kv.ensure(0, T)
    i32 = dict(dtype=torch.int32, device="cuda:0")
    for idx in ([T], [0, -T - 1]):
        with pytest.raises(IndexError):
            model.forward(torch.arange(T, **i32), torch.arange(T, **i32), kv,
                          torch.zeros(T, **i32),
                          _meta("prefill", "cuda:0", [T], [T], idx,
                                rows=idx if host else None))


@pytest.mark.gpu
@pytest.mark.parametrize("S", [3, 64, 70, 128])
def test_decode_rows(S):
    """Of a decode step too: some of them, repeated and in another order."""
    model = _model()
    kv = _cache(model, S)
    g = torch.Generator().manual_seed(2)
    i32 = dict(dtype=torch.int32, device="cuda:0")
    tok = torch.randint(0, model.cfg.vocab, (S,), generator=g).to(**i32)
    for s in range(S):
        kv.ensure(s, 1)
    slots = torch.arange(S, **i32)

    def go(idx, **kw):
        return model.forward(tok, torch.zeros(S, **i32), kv, slots, _meta(
            "decode", "cuda:0", [1] * S, [1] * S, idx, **kw))

    whole = go(list(range(S)), rows=list(range(S)))
    assert whole.shape[0] == S
    for idx in ([S - 1], list(range(S))[::-1], [2, 0, -1, 2],
                list(range(S))):
        got = go(idx)
        assert got.shape[0] == len(idx)
        # the rows' sums of squares are taken before or after their rounding
        # to bf16: 2^-9 of a value, far less of a row's root mean square, and
        # one more rounding of a logit
        torch.testing.assert_close(got.float(), whole[idx].float(),
                                   rtol=2 ** -7, atol=2 ** -8)
    assert go([S, 0]).isnan().any(1).tolist() == [True, False]
