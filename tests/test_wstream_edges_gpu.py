"""Weight-streaming products over activations in fragment layout at the edges
of their tiles, against float64.

Tolerance: fp32 sums of K products of about 1/sqrt(K), then one rounding to
bf16 (relative 2^-9; doubled, as the sum's own error can cross a tie).
"""
import pytest
import torch

pytestmark = pytest.mark.gpu
CLOSE = dict(rtol=2 ** -8, atol=1e-4)


def _hip():
    from ollamamq_amd.ops import hip
    hip.require()
    return hip


def _frag(x):
    """x in fragment layout; rows that do not exist are NaN."""
    rows = -(-x.shape[0] // 32) * 32
    full = torch.full((rows, x.shape[1]), float("nan"), dtype=x.dtype,
                      device=x.device)
    full[:x.shape[0]] = x
    return full.view(rows // 32, 32, -1, 4, 2, 8).permute(0, 2, 3, 4, 1, 5) \
        .contiguous().flatten()


def _defrag(buf, rows, cols):
    x = buf.view(-1, cols // 64, 4, 2, 32, 8).permute(0, 4, 1, 2, 3, 5)
    return x.reshape(-1, cols)[:rows]


def _case(M, N, K, seed=3):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = (torch.randn(N, K, generator=g, device="cuda") / K ** 0.5).bfloat16()
    return x, w, x.double() @ w.double().T


@pytest.mark.parametrize("M", [1, 2, 15, 16, 17, 31, 32, 33, 48, 63, 64])
@pytest.mark.parametrize("N,K", [(32, 64), (64, 448), (96, 576), (64, 1088),
                                 (128, 4096), (64, 4160)])
def test_whole(M, N, K):
    hip = _hip()
    x, w, want = _case(M, N, K)
    pk = hip.pack_weight(w)
    got = hip.linear_packed(_frag(x), pk, None, N, ks=1, K=K, xlds=2,
                            M_frag=M)
    torch.testing.assert_close(got.double(), want, **CLOSE)
    rows = -(-M // 32) * 32
    norms = torch.rand(rows, 3, device="cuda") + 0.1     # three partials
    bias = torch.randn(N, device="cuda").bfloat16()
    got = hip.linear_packed(_frag(x), pk, bias, N, K=K, xlds=2, M_frag=M,
                            rstd=norms, rstd_nt=3, inv_h=1 / K, eps=1e-5)
    scale = (norms.double().sum(1) / K + 1e-5).rsqrt()[:M, None]
    # the scale is the hardware's reciprocal root: relative 1e-6 more
    torch.testing.assert_close(got.double(), want * scale + bias.double(),
                               rtol=2 ** -8, atol=2e-3)


@pytest.mark.parametrize("M", [1, 17, 32, 33, 64])
@pytest.mark.parametrize("ks", [2, 3, 4, 8, 9, 16])
@pytest.mark.parametrize("N,K", [(64, 512), (192, 1088), (128, 4160)])
def test_parts_add_themselves_up(M, ks, N, K):
    """The residual sum in place, sums of squares, and tickets that are zero
    again, over several products that share them.  More parts than blocks of
    64 columns leave some empty."""
    hip = _hip()
    x, w, want = _case(M, N, K)
    pk, xf = hip.pack_weight(w), _frag(x)
    sem = torch.zeros(N // 32, dtype=torch.int32, device="cuda")
    base = torch.randn(M, N, device="cuda").bfloat16()
    rows = -(-M // 32) * 32
    first = None
    for _ in range(4):
        res = _frag(base)
        sq = torch.zeros(rows, N // 32, device="cuda")
        y = hip.linear_packed(xf, pk, None, N, ks=ks, res=res, y=res,
                              sq_out=sq, yfrag=1, K=K, xlds=2, M_frag=M,
                              sem=sem)
        total = want + base.double()
        got = _defrag(y, M, N).double()
        torch.testing.assert_close(got, total, **CLOSE)
        torch.testing.assert_close(
            sq[:M].double(), total.square().unflatten(1, (-1, 32)).sum(2),
            rtol=1e-4, atol=1e-3)
        assert not sem.any()
        # whoever comes last adds up in the same order
        assert first is None or torch.equal(first, got)
        first = got
    plain = hip.linear_packed(xf, pk, None, N, ks=ks, K=K, xlds=2, M_frag=M)
    torch.testing.assert_close(plain.double(), want, **CLOSE)


@pytest.mark.parametrize("M", [1, 17, 32])
@pytest.mark.parametrize("xlds,depth", [(0, 1), (0, 2), (1, 1)])
@pytest.mark.parametrize("ks,N,K", [(2, 64, 512), (3, 192, 1088),
                                    (8, 128, 4160), (None, 4096, 14336)])
def test_parts_of_plain_rows(M, xlds, depth, ks, N, K):
    """The residual sum and sums of squares of a split product over rows that
    lie in memory one after another, strided ones too."""
    hip = _hip()
    x, w, want = _case(M, N, K)
    x = torch.cat([x, x], 1)[:, :K]
    pk = hip.pack_weight(w)
    assert (ks or hip._wstream_ksplit(N, K)) > 1
    base = torch.randn(M, N, device="cuda").bfloat16()
    bias = torch.randn(N, device="cuda").bfloat16()
    total = want + base.double() + bias.double()
    sem = torch.zeros(N // 32, dtype=torch.int32, device="cuda")
    for tickets in (None, sem):
        res = base.clone()
        sq = torch.zeros(32, N // 32, device="cuda")
        y = hip.linear_packed(x, pk, bias, N, ks=ks, depth=depth, xlds=xlds,
                              res=res, y=res, sq_out=sq, sem=tickets)
        assert y is res and not sem.any()
        torch.testing.assert_close(y.double(), total, **CLOSE)
        torch.testing.assert_close(
            sq[:M].double(), total.square().unflatten(1, (-1, 32)).sum(2),
            rtol=1e-4, atol=1e-3)
    # one of the two alone
    y = hip.linear_packed(x, pk, None, N, ks=ks, depth=depth, xlds=xlds,
                          res=base)
    torch.testing.assert_close(y.double(), want + base.double(), **CLOSE)
    if N % 64 == 0:                      # whole blocks of the layout
        y = hip.linear_packed(x, pk, bias, N, ks=ks, depth=depth, xlds=xlds,
                              yfrag=1)
        torch.testing.assert_close(_defrag(y, M, N).double(),
                                   want + bias.double(), **CLOSE)
    sq = torch.zeros(32, N // 32, device="cuda")
    hip.linear_packed(x, pk, None, N, ks=ks, depth=depth, xlds=xlds,
                      sq_out=sq)
    torch.testing.assert_close(
        sq[:M].double(), want.square().unflatten(1, (-1, 32)).sum(2),
        rtol=1e-4, atol=1e-3)


def test_parts_without_tickets_are_refused_what_needs_sums():
    """Nothing runs: fragment layout, a residual, norms or their sums, asked
    of parts that nobody adds up."""
    hip = _hip()
    x, w, _ = _case(8, 64, 512)
    pk, y = hip.pack_weight(w), torch.zeros(32 * 64, device="cuda").bfloat16()
    part = torch.empty(2 * 32 * 64, device="cuda")
    one = torch.zeros(64, device="cuda")

    def go(xlds, norm=None, res=None, sq=None, yfrag=0):
        return hip._lib.wstream_gemm_bf16(
            *map(hip._p, (y, part, x, pk, None)), 8, 64, 512, 512, 2, 1, xlds,
            hip._p(norm), 1, 1.0, 1.0, hip._p(res), hip._p(sq), yfrag, None,
            hip._stream())

    for xlds in (0, 1):
        for kw in (dict(norm=one), dict(res=y), dict(sq=one), dict(yfrag=1)):
            assert go(xlds, **kw) != 0
    assert not y.any()


def test_more_plain_rows_are_refused():
    """A block has 64 rows of them, with rope 32; none are left out."""
    hip = _hip()
    x, w, want = _case(65, 64, 512)
    pk, gu = hip.pack_weight(w), hip.pack_weight_gu(w)
    got = hip.linear_packed(x[:64], pk, None, 64)
    torch.testing.assert_close(got.double(), want[:64], **CLOSE)
    hip.linear_gu(x[:64], gu, 64)
    for go in (lambda: hip.linear_packed(x, pk, None, 64),
               lambda: hip.linear_packed(x, pk, None, 64, ks=2),
               lambda: hip.linear_gu(x, gu, 64)):
        with pytest.raises(RuntimeError):
            go()
    none = [hip._p(None)]
    assert hip._lib.wstream_qkv_rope_bf16(
        *none * 4, 33, 384, 512, 512, *none, 1, 1.0, 1.0, *none * 7, 1, 1, 16,
        1, 0, hip._stream()) != 0


@pytest.mark.parametrize("M", [1, 16, 32, 33, 64])
@pytest.mark.parametrize("F,K", [(16, 64), (48, 576), (160, 4160)])
def test_gate_up(M, F, K):
    hip = _hip()
    x, w, want = _case(M, 2 * F, K)
    gate, up = want.chunk(2, 1)
    want = torch.nn.functional.silu(gate) * up
    got = hip.linear_gu(_frag(x), hip.pack_weight_gu(w), 2 * F, K=K,
                        M_frag=M)
    torch.testing.assert_close(got.double(), want, **CLOSE)
