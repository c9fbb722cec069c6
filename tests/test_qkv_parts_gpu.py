"""Rotated products in parts of K.  Whole numbers add up exactly in any order
and cosines and sines of 0, 1 and -1 rotate them exactly, so queries, keys and
values are bit for bit those of the product that takes K whole."""
from types import SimpleNamespace

import pytest
import torch

from ollamamq_amd.ops import hip
from test_tile_row_sums_gpu import eight_side_by_side


def test_rule():
    """Parts for 49 to 128 rows only, of whole slabs, and of no more blocks
    than CUs; None is the stream."""
    for cus in (32, 64, 256):
        for N, K in ((6144, 4096), (4608, 3584), (512, 1024), (512, 2048),
                     (3072, 2112), (16384, 4096), (128, 65536)):
            for M in range(1, 200):
                plan = hip.rope_parts(M, N, K, cus)
                if plan is None:
                    continue
                hm, hn, ks = plan
                assert 48 < M <= 32 * hm and hn == 2 and K % 256 == 0
                assert 2 <= ks <= K // 1024 and -(-N // 64) * ks <= cus
    assert hip.rope_parts(128, 6144, 4096) == (4, 2, 2)
    assert hip.rope_parts(64, 4608, 3584) == (2, 2, 3)
    assert hip.rope_parts(96, 6144, 4096) is None


@pytest.mark.parametrize("M, N, K, parts", [
    # streams and parts, us
    (97, 6144, 2048, None),             # 15.4, 16.5
    (128, 5120, 2048, None),            # 15.3, 15.9
    (97, 8192, 2816, None),             # 20.0, 20.6
    (49, 5120, 4096, None),             # 15.7, 16.2
    (56, 4608, 3072, None),             # 13.1, 13.4
    (97, 2560, 2048, (4, 2, 2)),        # 14.2, 14.0
    (97, 6144, 2560, (4, 2, 2)),        # 18.6, 17.4
    (97, 6144, 3328, (4, 2, 2)),        # 21.4, 21.0
    (57, 5120, 4096, (2, 2, 3)), (49, 5120, 3584, (2, 2, 3)),
    (49, 5120, 5120, (2, 2, 3)), (49, 2560, 3072, (2, 2, 3))])
def test_no_slower_than_the_stream(M, N, K, parts):
    assert hip.rope_parts(M, N, K) == parts


# the fold loads up to four parts at once; strips of 32 columns by the eight, a
# rest, and fewer than its waves
@pytest.mark.gpu
@pytest.mark.parametrize("ks", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("M, nl, nkl, page, nt, bias", [
    (1, 1, 1, 16, 1, False), (49, 7, 1, 48, 3, True), (64, 4, 2, 16, 16, False),
    (65, 28, 4, 16, 5, True), (128, 32, 8, 64, 32, True),
    (300, 2, 1, 16, 16, True)])
def test_bits(M, nl, nkl, page, nt, bias, ks):
    hip.require()
    torch.manual_seed(M + ks)
    K, slots, rows = 8 * 256, 3, -(-M // 32) * 32
    N, per = (nl + 2 * nkl) * 128, -(-(M // slots + 9) // page)

    def whole(lo, hi, *shape):
        return torch.randint(lo, hi, shape, device="cuda").bfloat16()

    x, w = whole(-2, 3, rows * K), whole(-1, 2, N * K)
    b = whole(-9, 10, N) if bias else None
    n_pages = slots * per + 1
    table = torch.randperm(n_pages, device="cuda")[:slots * per] \
        .view(slots, per).int().contiguous()
    pos = torch.arange(M, device="cuda").int() // slots + 5
    slot = torch.arange(M, device="cuda").int() % slots
    cos, sin = torch.randint(-1, 2, (2, per * page, 64), device="cuda").float()
    sq = torch.randint(1, 4096, (M, nt), device="cuda").float()

    def outputs(product, plan):
        cache = SimpleNamespace(
            n_kv_heads=nkl, page_size=page, page_table=table,
            k_pool=torch.zeros(2, n_pages, nkl, page, 128, device="cuda",
                               dtype=torch.bfloat16))
        cache.v_pool = torch.zeros_like(cache.k_pool)
        q = product(x, w, M, N, K, b, cache, 1, pos, slot, cos, sin, nl, nkl,
                    sq, nt, 1.0 / K, 1e-5, plan=plan)
        return q[:, :nl * 128], cache.k_pool, cache.v_pool

    want = outputs(hip.tile_qkv_rope, (4, 2, 1))
    assert all(t.any() for t in want)
    for tile in ((4, 2), *([(2, 2)] if M <= 64 else [])):
        for got, one in zip(outputs(hip.tile_qkv_parts, (*tile, ks)), want):
            assert torch.equal(got, one)


@pytest.mark.gpu
@pytest.mark.parametrize("nt", [2, 4, 7, 9, 16, 19, 32])
def test_order_of_row_sums(nt):
    """Eight sums side by side, however many a row comes in: 2^25 has no room
    for what is added to it before it is taken away again."""
    hip.require()
    torch.manual_seed(nt)
    M, K, nl, nkl, page = 65, 512, 4, 1, 16
    N = (nl + 2 * nkl) * 128
    x = torch.randn(96 * K, device="cuda").bfloat16()
    w = torch.randn(N * K, device="cuda").mul_(K ** -0.5).bfloat16()
    parts = torch.rand(M, nt, device="cuda") * 100
    if nt > 8:
        parts[:, 0], parts[:, 8] = 2 ** 25, -2 ** 25
    pos = torch.arange(M, device="cuda").int()
    slot = torch.zeros_like(pos)
    table = torch.arange(5, device="cuda").int().view(1, 5)
    cos, sin = torch.rand(2, 80, 64, device="cuda")

    def outputs(sq, n):
        cache = SimpleNamespace(
            n_kv_heads=nkl, page_size=page, page_table=table,
            k_pool=torch.zeros(1, 5, nkl, page, 128, device="cuda",
                               dtype=torch.bfloat16))
        cache.v_pool = torch.zeros_like(cache.k_pool)
        q = hip.tile_qkv_parts(x, w, M, N, K, None, cache, 0, pos, slot, cos,
                               sin, nl, nkl, sq, n, 1.0 / K, 1e-5, (4, 2, 2))
        return q[:, :nl * 128], cache.k_pool, cache.v_pool

    for got, one in zip(outputs(parts, nt),
                        outputs(eight_side_by_side(parts), 1)):
        assert one.any() and torch.equal(got, one)


def test_refused():
    if not hip.available():
        pytest.skip("the extension is not built")
    some = 1 << 20                      # nothing reads it

    def call(part=some, rstd=some, nt=1, M=65, N=384, K=512, hm=4, hn=2, ks=2):
        return hip._lib.tile_rope_parts_bf16(
            some, part, some, some, None, rstd, nt, 0.0, 0.0, M, N, K, hm, hn,
            ks, 8, 256, *[some] * 7, 1, 1, 16, 1, None)
    if not torch.cuda.is_available():   # nothing but the device is missing
        assert call() > 0
    for bad in (dict(part=None), dict(rstd=None), dict(nt=0), dict(M=0),
                dict(N=512), dict(K=320), dict(ks=0), dict(ks=3),
                dict(hm=5, hn=5)):
        assert call(**bad) < 0, bad
