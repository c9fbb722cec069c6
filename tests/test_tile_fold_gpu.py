"""Products over tiles in parts of K.  Whole numbers add up exactly in any order
and in any number of parts, so every value is the one rounding to bf16 of the
exact sum."""
import pytest
import torch

from ollamamq_amd.ops import hip


# up to eight parts are loaded at once, nine and more are not
@pytest.mark.gpu
@pytest.mark.parametrize("ks", [*range(1, 10), 12])
@pytest.mark.parametrize("M, N", [(1, 64), (33, 448), (128, 1088), (300, 64)])
def test_parts(ks, M, N):
    hip.require()
    torch.manual_seed(ks)
    K, rows = 12 * 256, -(-M // 32) * 32

    def whole(lo, hi, *shape):
        return torch.randint(lo, hi, shape, device="cuda").bfloat16()

    def frag(t):
        return t.view(-1, 32, t.shape[1] // 8, 8).transpose(1, 2).flatten()

    def rows_of(f):
        return f.view(-1, N // 8, 32, 8).transpose(1, 2).reshape(-1, N)[:M]

    x, w, res = whole(-2, 3, rows, K), whole(-1, 2, N, K), whole(-99, 99, rows, N)
    want = x.double() @ w.double().T + res.double()
    xf, packed, y = frag(x), hip.pack_weight(w), frag(res)
    part = torch.full((ks * rows * N,), float("nan"), device="cuda")
    sq = torch.full((M, hip.TILE_FOLD), float("nan"), device="cuda")
    hip._tile_gemm(hip.TILE_PARTS, y, xf, packed, M, N, K, (4, 2, ks),
                   part=part, res=y, sq=sq)
    assert torch.equal(rows_of(y), want[:M].bfloat16())
    # sums of N squares below 2^24 each, in fp32: N roundings at most
    torch.testing.assert_close(sq.double().sum(1), want[:M].square().sum(1),
                               rtol=N * 2.0 ** -24, atol=0)
