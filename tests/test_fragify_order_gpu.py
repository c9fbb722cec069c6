"""Rows to fragments around the groups of 64 rows whose blocks change places."""
import pytest
import torch

from ollamamq_amd.ops import hip


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 63, 64, 65, 127, 128, 200])
def test_every_row(M):
    hip.require()
    torch.manual_seed(M)
    H, rows = 576, -(-M // 32) * 32
    table = torch.randint(-8, 9, (300, H), device="cuda").bfloat16()
    tokens = torch.randint(0, 300, (M,), device="cuda")
    clear = torch.ones(1000, dtype=torch.int32, device="cuda")
    xf, sq = hip.fragify_sumsq(table, tokens=tokens, clear=clear)
    x = xf.view(rows // 32, H // 8, 32, 8).transpose(1, 2).reshape(rows, H)
    want = table[tokens]
    assert torch.equal(x[:M], want) and not clear.any()
    # whole numbers below 2^24: exact in any order
    assert torch.equal(sq, want.float().square().sum(1))
