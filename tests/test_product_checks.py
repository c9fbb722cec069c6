"""What a product asks of its buffers, on the host: a kernel cannot know how
long they are."""
import pytest
import torch

from ollamamq_amd.ops import hip


@pytest.mark.parametrize("M", [1, 32, 33, 128])
def test_sums_of_whole_row_tiles(M):
    """A product writes sums of squares of 32 rows, so fewer are refused."""
    N, K, rows = 64, 64, -(-M // 32) * 32
    x, w, y = (torch.empty(n, dtype=torch.bfloat16)
               for n in (rows * K, N * K, rows * N))
    with pytest.raises(AssertionError):
        hip.linear_packed(x, w, None, N, K=K, xlds=2, M_frag=M, yfrag=1, y=y,
                          sq_out=torch.empty(rows - 1, N // 32))
