"""Weight-streaming products for 65 to 128 rows, and those of many columns for
33 rows and more, against float64; steps of so many tokens against the general
path.

Tolerance of the products: fp32 sums of K products of about 1/sqrt(K), then one
rounding to bf16 (relative 2^-9; doubled, as the sum's own error can cross a
tie); the scale of a norm is the hardware's reciprocal root, 1e-6 more.
"""
import pytest
import torch

from test_short_prompts_gpu import _close, _run
from test_wstream_edges_gpu import CLOSE, _case, _defrag, _frag, _hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [65, 95, 96, 97, 127, 128])
@pytest.mark.parametrize("N,K", [(32, 64), (192, 576), (64, 4160)])
def test_rows(M, N, K):
    hip = _hip()
    x, w, want = _case(M, N, K)
    pk, xf = hip.pack_weight(w), _frag(x)
    got = hip.linear_packed(xf, pk, None, N, ks=1, K=K, xlds=2, M_frag=M)
    torch.testing.assert_close(got.double(), want, **CLOSE)
    rows = -(-M // 32) * 32
    norms = torch.rand(rows, 37, device="cuda") / 12 + 0.01
    scale = (norms.double().sum(1) / K + 1e-5).rsqrt()[:M, None]
    bias = torch.randn(N, device="cuda").bfloat16()
    got = hip.linear_packed(xf, pk, bias, N, K=K, xlds=2, M_frag=M,
                            rstd=norms, rstd_nt=37, inv_h=1 / K, eps=1e-5)
    torch.testing.assert_close(got.double(), want * scale + bias.double(),
                               rtol=2 ** -8, atol=2e-3)
    base = torch.randn(M, N, device="cuda").bfloat16()
    total = want + base.double()
    sem = torch.zeros(N // 32, dtype=torch.int32, device="cuda")
    for ks in (1, 2, 8):
        if ks * 8 > K // 64:
            continue
        for _ in range(3):
            res = _frag(base)
            sq = torch.zeros(rows, N // 32, device="cuda")
            y = hip.linear_packed(xf, pk, None, N, ks=ks, res=res, y=res,
                                  sq_out=sq, yfrag=1, K=K, xlds=2, M_frag=M,
                                  sem=sem)
            torch.testing.assert_close(_defrag(y, M, N).double(), total,
                                       **CLOSE)
            torch.testing.assert_close(
                sq[:M].double(), total.square().unflatten(1, (-1, 32)).sum(2),
                rtol=1e-4, atol=1e-3)
            assert not sem.any()
    plain = hip.linear_packed(xf, pk, None, N, ks=3, K=K, xlds=2, M_frag=M)
    torch.testing.assert_close(plain.double(), want, **CLOSE)


# 511 to 1031 tiles: the last block has fewer than the others; one step of K,
# fewer than the groups of waves, and odd numbers of steps
@pytest.mark.parametrize("M", [33, 64, 65, 96, 97, 128])
@pytest.mark.parametrize("tiles,K", [(513, 64), (511, 64), (512, 128),
                                     (517, 192), (1031, 576), (525, 4160)])
def test_many_columns(M, tiles, K):
    hip = _hip()
    N = tiles * 32
    x, w, want = _case(M, N, K)
    xf, rows = _frag(x), -(-M // 32) * 32
    pk = hip.pack_weight(w)
    got = hip.linear_packed(xf, pk, None, N, K=K, xlds=2, M_frag=M)
    torch.testing.assert_close(got.double(), want, **CLOSE)
    norms = torch.rand(rows, 37, device="cuda") / 12 + 0.01
    scale = (norms.double().sum(1) / K + 1e-5).rsqrt()[:M, None]
    got = hip.linear_packed(xf, pk, None, N, K=K, xlds=2, M_frag=M,
                            rstd=norms, rstd_nt=37, inv_h=1 / K, eps=1e-5,
                            yfrag=1 - tiles % 2)
    if tiles % 2 == 0:
        got = _defrag(got, M, N)
    torch.testing.assert_close(got.double(), want * scale, rtol=2 ** -8,
                               atol=2e-3)
    gate, up = want.chunk(2, 1)
    pk = hip.pack_weight_gu(w)
    for glu, act in (("silu", torch.nn.functional.silu),
                     ("gelu_tanh", lambda v: torch.nn.functional.gelu(
                         v, approximate="tanh"))):
        got = hip.linear_gu(xf, pk, N, K=K, M_frag=M, glu=glu)
        torch.testing.assert_close(got.double(), act(gate) * up, **CLOSE)
    if N // 2 % 64 == 0:
        got = hip.linear_gu(xf, pk, N, K=K, M_frag=M, yfrag=1)
        torch.testing.assert_close(
            _defrag(got, M, N // 2).double(),
            torch.nn.functional.silu(gate) * up, **CLOSE)


@pytest.mark.parametrize("M", [33, 64, 65, 96, 128])
@pytest.mark.parametrize("tiles,K", [(129, 7232), (128, 14336), (112, 18944)])
def test_few_columns_in_parts(M, tiles, K):
    """Parts that add themselves up: the residual sum in place, sums of
    squares, a bias, and tickets that are zero again."""
    hip = _hip()
    N = tiles * 32
    x, w, want = _case(M, N, K)
    pk, xf, rows = hip.pack_weight(w), _frag(x), -(-M // 32) * 32
    if tiles % 2 == 0:
        base = torch.randn(M, N, device="cuda").bfloat16()
        bias = torch.randn(N, device="cuda").bfloat16()
        total = want + base.double() + bias.double()
        sem = torch.zeros(tiles, dtype=torch.int32, device="cuda")
        for ks in (None, 2, 4, 8):
            first = None
            for _ in range(3):
                res = _frag(base)
                sq = torch.zeros(rows, tiles, device="cuda")
                y = hip.linear_packed(xf, pk, bias, N, ks=ks, res=res, y=res,
                                      sq_out=sq, yfrag=1, K=K, xlds=2,
                                      M_frag=M, sem=sem)
                got = _defrag(y, M, N).double()
                torch.testing.assert_close(got, total, **CLOSE)
                torch.testing.assert_close(
                    sq[:M].double(),
                    total.square().unflatten(1, (-1, 32)).sum(2),
                    rtol=1e-4, atol=1e-3)
                assert not sem.any()
                # whoever comes last adds up in the same order
                assert first is None or torch.equal(first, got)
                first = got
    for ks in (None, 1, 3, 4, 8):
        got = hip.linear_packed(xf, pk, None, N, ks=ks, K=K, xlds=2, M_frag=M)
        torch.testing.assert_close(got.double(), want, **CLOSE)


def test_more_rows_are_refused():
    hip = _hip()
    x, w, _ = _case(129, 64, 64)
    with pytest.raises(RuntimeError):
        hip.linear_packed(_frag(x), hip.pack_weight(w), None, 64, ks=1, K=64,
                          xlds=2, M_frag=129)


STEPS = [
    [(0, range(65), [64, 0])],
    [(1, range(100), range(97))],
    [(2, range(1, 129), [127])],
    [(0, [5], [0]), (3, range(120), [119, 3]), (1, [7], [0])],
    # one token too many for the chain, and more places than it takes
    [(4, range(129), [128])],
    [(4, range(12), [3] * 130)],
]


@pytest.mark.parametrize("name", ["tiny", "tiny-qwen", "tiny-swa"])
def test_chain_and_general_path(name):
    from ollamamq_amd.models import LlamaModel, PRESETS
    cfg = PRESETS[name]
    model = LlamaModel(cfg, device="cuda:0", dtype=torch.bfloat16, seed=5)
    assert model.fused_chain
    got, k1, v1 = _run(model, cfg, True, STEPS)
    want, k2, v2 = _run(model, cfg, False, STEPS)
    for a, b in zip(got, want):
        assert a.shape == b.shape
        _close(a.float(), b.float())
    # the pools hold zeros where nothing was cached
    _close(k1[k2 != 0], k2[k2 != 0])
    _close(v1[v2 != 0], v2[v2 != 0])
    assert torch.equal(k1 != 0, k2 != 0) and torch.equal(v1 != 0, v2 != 0)


@pytest.mark.parametrize("T", [1, 5, 128, 129])
def test_no_logits_wanted(T):
    """A portion none of whose logits are wanted is refused on either path."""
    from ollamamq_amd.engine import PagedKVCache
    from ollamamq_amd.models import LlamaModel, PRESETS
    from ollamamq_amd.ops.interface import AttnMeta
    cfg = PRESETS["tiny"]
    model = LlamaModel(cfg, device="cuda:0", dtype=torch.bfloat16, seed=5)
    kv = PagedKVCache.for_model(cfg, n_pages=16, max_slots=1, max_ctx=256,
                                device="cuda:0", dtype=torch.bfloat16)
    slot = kv.alloc_slot()
    kv.ensure(slot, T)
    i32 = dict(dtype=torch.int32, device="cuda:0")
    meta = AttnMeta(
        mode="prefill", slot_ids=torch.tensor([slot], **i32),
        seq_lens=torch.tensor([T], **i32), cu_q=torch.tensor([0, T], **i32),
        logits_idx=torch.empty(0, dtype=torch.long, device="cuda:0"),
        max_q=T, max_kv=T)
    with pytest.raises(RuntimeError, match="launch failed"):
        model.forward(torch.arange(T, **i32), torch.arange(T, **i32), kv,
                      torch.full((T,), slot, **i32), meta)


@pytest.mark.parametrize("T,H", [(1, 64), (200, 512), (130, 4096)])
def test_rows_of_a_sum(T, H):
    """Rows by their indexes, from the end where these are negative."""
    hip = _hip()
    x, y = torch.randn(2, T, H, device="cuda").bfloat16()
    for idx in ([0], [-1, 0, T - 1, -T], [T - 1] * 40, list(range(T))):
        rows = torch.tensor(idx, device="cuda")
        want = x[rows] + y[rows]
        for form in (rows, rows.int(), rows.repeat_interleave(2)[::2]):
            xf, sq = hip.fragify_sumsq(x, rows=form, add=y)
            assert torch.equal(_defrag(xf, len(idx), H), want)
            torch.testing.assert_close(
                sq.double(), want.double().square().sum(1), rtol=1e-5,
                atol=0)
        if T <= 128:
            got, _ = hip.frag_rows(_frag(x), rows, H, T)
            assert torch.equal(_defrag(got, len(idx), H), x[rows])
