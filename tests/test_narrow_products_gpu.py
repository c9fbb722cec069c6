"""Products of up to 64 rows in blocks of 16 columns, or of 64 in parts of K:
residual and sums of squares, rotation and append.

Tolerance: sums of up to K products of bf16 values in fp32, whose error is below
K 2^-24 of the sum of magnitudes, then one rounding to bf16 (2^-9 of the value,
doubled as the sum's error can cross a tie).  A row's sum of squares is taken of
the values before that rounding: K 2^-22 of it at most, as values' errors count
twice.
"""
import pytest
import torch

from ollamamq_amd.ops import hip

pytestmark = pytest.mark.gpu


def _rows(flat, M, W):
    """Rows of an activation in fragment layout."""
    t = flat.view(-1, W // 16, 2, 32, 8)             # 32 rows, 16 and 8 of W
    return t.permute(0, 3, 1, 2, 4).reshape(-1, W)[:M]


def _residual(ks, x, w, r):
    """x w^T + r and its sums of squares a row, in blocks of 16 columns or in ks
    parts of 64; what is beside them stays as it is."""
    (M, K), N = x.shape, len(w)
    xf, rf = (hip.fragify_sumsq(t)[0] for t in (x, r))
    packed, n = hip.pack_weight(w), M * N // (64 if ks else 16)
    sq = torch.full((n + 64,), 7.0, device="cuda")
    if ks:
        rows = -(-M // 32) * 32
        part = torch.full((ks * rows * N + 64,), 7.0, device="cuda")
        sem = torch.zeros(N // 64 + 1, dtype=torch.int32, device="cuda")
        hip._check(hip._lib.wstream_duo_bf16(
            hip._p(rf), hip._p(part), hip._p(xf), hip._p(packed), M, N, K, ks,
            hip._p(rf), hip._p(sq), hip._p(sem), hip._stream()), "duo")
        assert not sem.any() and (part[ks * rows * N:] == 7).all()
    else:
        hip._check(hip._lib.wstream_narrow_bf16(
            hip._p(rf), hip._p(xf), hip._p(packed), M, N, K, hip._p(rf),
            hip._p(sq), hip._stream()), "narrow")
    assert (sq[n:] == 7).all()
    return _rows(rf, M, N), sq[:n].view(M, -1).double().sum(1)


# waves without a step, with one, with whole rounds of those under way and with
# more; halves of a wave's rows
@pytest.mark.parametrize("ks,N,K", [
    (0, 32, 64), (0, 96, 512), (0, 64, 64 * 37), (0, 2048, 2048),
    (0, 32, 64 * 71), (1, 64, 64), (1, 128, 64 * 61), (2, 64, 1024),
    (3, 192, 64 * 71), (4, 256, 64 * 225), (5, 64, 64 * 83), (9, 128, 64 * 80)])
@pytest.mark.parametrize("M", [1, 7, 16, 17, 32, 33, 48, 49, 64])
def test_residual(M, ks, N, K):
    hip.require()
    g = torch.Generator(device="cuda").manual_seed(M * N + K)

    def rand(*shape):
        return torch.randn(shape, generator=g, device="cuda").bfloat16()

    x, w, r = rand(M, K), rand(N, K), rand(M, N)
    got, sums = _residual(ks, x, w, r)
    want = x.double() @ w.double().T + r.double()
    size = x.double().abs() @ w.double().abs().T + r.double().abs()
    err = (got.double() - want).abs()
    assert (err <= 2 ** -8 * want.abs() + K * 2 ** -24 * size).all()
    torch.testing.assert_close(sums, want.square().sum(1), rtol=K * 2 ** -22,
                               atol=0)


@pytest.mark.parametrize("N,K", [(4096, 4096), (3584, 3584), (4096, 14336),
                                 (2048, 2816), (5120, 4096)])
@pytest.mark.parametrize("M", [16, 32, 48, 64])
def test_rounds_no_more_than_streams(M, N, K):
    """Sums whose exact value is zero: what is left is what fp32 rounded, and it
    is no more than in the streamed product's parts (5 % for the sample, of
    32768 sums and more: its rms is off by 0.4 %)."""
    hip.require()
    g = torch.Generator(device="cuda").manual_seed(K + M)
    at = torch.randperm(K, generator=g, device="cuda")
    x, w = (torch.randn(n, K // 2, generator=g, device="cuda").bfloat16()
            for n in (M, N))
    x, w = (torch.cat(p, 1)[:, at].contiguous()
            for p in ((x, x), (w, -w)))
    xf, packed = hip.fragify_sumsq(x)[0], hip.pack_weight(w)
    off = []
    for narrow in (False, True):
        y = torch.zeros(-(-M // 32) * 32 * N, device="cuda").bfloat16()
        sq = torch.empty(64 * N // 16, device="cuda")
        if narrow:
            hip._check(hip._lib.wstream_narrow_bf16(
                hip._p(y), hip._p(xf), hip._p(packed), M, N, K, hip._p(y),
                hip._p(sq), hip._stream()), "narrow")
        else:
            hip.linear_packed(
                xf, packed, None, N, res=y, sq_out=sq, y=y, yfrag=1, K=K,
                xlds=2, M_frag=M,
                sem=torch.zeros(N // 32, dtype=torch.int32, device="cuda"))
        off.append(_rows(y, M, N).double().square().mean().sqrt())
    assert 0 < off[1] <= 1.05 * off[0]


def test_refused():
    hip.require()
    t = torch.zeros(64 * 64, device="cuda", dtype=torch.bfloat16)
    p = hip._p(t)
    for M, N, K, res in ((0, 32, 64, p), (65, 32, 64, p), (1, 16, 64, p),
                         (1, 48, 64, p), (1, 32, 32, p), (1, 32, 64, None)):
        assert hip._lib.wstream_narrow_bf16(p, p, p, M, N, K, res, p,
                                            hip._stream())
    for M, N, K, ks, part, res, sem in (
            (0, 64, 64, 1, p, p, p), (65, 64, 64, 1, p, p, p),
            (1, 32, 64, 1, p, p, p), (1, 96, 64, 1, p, p, p),
            (1, 64, 96, 1, p, p, p), (1, 64, 64, 0, p, p, p),
            (1, 64, 1024, 2, None, p, p), (1, 64, 1024, 2, p, None, p),
            (1, 64, 1024, 2, p, p, None)):
        assert hip._lib.wstream_duo_bf16(p, part, p, p, M, N, K, ks, res, p,
                                         sem, hip._stream())


# more than 256 tiles of 32 columns: up to 16 rows in blocks of 16, above in
# blocks of 32.  A row's results do not hang on the rows beside it.
@pytest.mark.parametrize("nl,nkl,bias", [(66, 1, True), (22, 22, False)])
@pytest.mark.parametrize("M", [1, 9, 16])
def test_rotated(M, nl, nkl, bias):
    from ollamamq_amd.engine import PagedKVCache
    hip.require()
    g = torch.Generator(device="cuda").manual_seed(M)
    N, K, T = (nl + 2 * nkl) * 128, 64 * 29, 17
    assert hip._lib.wstream_rope_narrow(M, N, K)

    def rand(*shape):
        return torch.randn(shape, generator=g, device="cuda").bfloat16()

    x, w = rand(T, K), rand(N, K)
    b = rand(N) if bias else None                    # in the order of the pack
    packed = hip.pack_weight_qkv_rope(w, nl, nkl)
    ang = torch.rand(64, 64, generator=g, device="cuda") * 6.28
    cos, sin = ang.cos(), ang.sin()
    got = []
    for m in (T, M):
        cache = PagedKVCache(1, nkl, 128, n_pages=64, max_slots=T, max_ctx=64,
                             device="cuda", dtype=torch.bfloat16)
        slots = [cache.alloc_slot() for _ in range(m)]
        for i, s in enumerate(slots):
            cache.ensure(s, 2 * i + 1)
        xf, sq = hip.fragify_sumsq(x[:m])
        q = hip.linear_qkv_rope(
            xf, packed, N, b, cache, 0,
            torch.arange(m, device="cuda", dtype=torch.int32) * 2,
            torch.tensor(slots, device="cuda", dtype=torch.int32), cos, sin,
            nl, nkl, sq, 1, 1.0 / K, 1e-5, K=K, M_real=m)
        pools = [torch.stack([
            pool[0, cache.page_table[s, 2 * i // 16].long(), :, 2 * i % 16]
            for i, s in enumerate(slots[:M])])
            for pool in (cache.k_pool, cache.v_pool)]
        got.append([q[:M, :nl * 128], *pools])
    for a, c in zip(*got):
        assert a.abs().max() > 0.1
        # both round sums of the same terms, of size sqrt(K) in fp32
        torch.testing.assert_close(a.float(), c.float(), rtol=2 ** -7,
                                   atol=K * 2 ** -20)


def _halves(head, angle):
    """A head's rotation in 64 bits."""
    lo, hi = head.chunk(2, -1)
    return torch.cat([lo * angle.cos() - hi * angle.sin(),
                      hi * angle.cos() + lo * angle.sin()], -1)


# Sums of squares come in any number: none (rows are taken as they are), and ones
# that 32 lanes a row read in eights, in twos and singly.
@pytest.mark.parametrize("nt", [None, 1, 31, 33, 256, 257, 300])
@pytest.mark.parametrize("M,K", [(1, 64 * 29), (16, 64 * 29), (5, 64 * 75),
                                 (17, 64 * 29), (16, 64 * 9)])
def test_rotated_norms(M, K, nt):
    from ollamamq_amd.engine import PagedKVCache
    hip.require()
    nl, nkl, page = 60, 3, 16
    N, eps = (nl + 2 * nkl) * 128, 0.0 if nt is None else 1e-5
    assert hip._lib.wstream_rope_narrow(M, N, K) == (M < 17 and K > 64 * 9)
    g = torch.Generator(device="cuda").manual_seed(M + (nt or 0))

    def rand(*shape):
        return torch.randn(shape, generator=g, device="cuda").bfloat16()

    x, w, b = rand(M, K), rand(N, K), rand(N)
    sq = None if nt is None else \
        torch.rand(M, nt, generator=g, device="cuda") * 2 * K / nt
    scale = 1.0 if nt is None else \
        (sq.double().sum(1, keepdim=True) / K + eps).rsqrt()
    angle = torch.rand(64, 64, generator=g, device="cuda") * 6.28
    pos = torch.arange(M, device="cuda", dtype=torch.int32) * 3
    cache = PagedKVCache(1, nkl, 128, page_size=page, n_pages=80, max_slots=M,
                         max_ctx=64, device="cuda", dtype=torch.bfloat16)
    slots = [cache.alloc_slot() for _ in range(M)]
    for i, s in enumerate(slots):
        cache.ensure(s, 3 * i + 1)
    order = torch.tensor(hip.qkv_rope_order(nl, nkl), device="cuda")
    got = hip.linear_qkv_rope(
        hip.fragify_sumsq(x)[0], hip.pack_weight_qkv_rope(w, nl, nkl), N,
        b[order], cache, 0, pos,
        torch.tensor(slots, device="cuda", dtype=torch.int32), angle.cos(),
        angle.sin(), nl, nkl, sq, nt or 0, 0.0 if nt is None else 1.0 / K,
        eps, K=K, M_real=M)
    at = [(cache.page_table[s, 3 * i // page].long(), 3 * i % page)
          for i, s in enumerate(slots)]
    got = torch.cat([got[:, :nl * 128].unflatten(1, (nl, 128)), *(
        torch.stack([pool[0, p, :, o] for p, o in at])
        for pool in (cache.k_pool, cache.v_pool))], 1)
    want = (x.double() @ w.double().T * scale + b.double()) \
        .unflatten(1, (-1, 128))
    size = (x.double().abs() @ w.double().abs().T * scale + b.double().abs()) \
        .unflatten(1, (-1, 128))
    turned = nl + nkl                        # values are not
    want[:, :turned] = _halves(want[:, :turned],
                               angle.double()[pos.long()][:, None])
    size[:, :turned] = size[:, :turned] + size[:, :turned].roll(64, -1)
    # as above, and the scale: nt sums and a reciprocal root; sines and cosines
    # are rounded to 24 bits
    err = (got.double() - want).abs()
    assert (err <= 2 ** -8 * want.abs()
            + (K + (nt or 0) + 8) * 2 ** -24 * size).all()
