"""Streamed products of few iterations a wave, of which two are under way: all
of them, two of four, or for half of the waves two of three, and one iteration
more or less than that.  Tolerance: see test_wstream_edges_gpu.py."""
import pytest

from test_wide_batches_gpu import test_many_columns as many_columns
from test_wstream_edges_gpu import test_parts_add_themselves_up as parts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [16, 17, 32])
@pytest.mark.parametrize("ks, K", [(1, 1024), (1, 1088), (1, 1728), (1, 1792),
                                   (1, 2048), (2, 2048), (3, 5376)])
def test_depth(M, ks, K):
    parts(M, ks, 192, K)
    if ks == 1:
        many_columns(M, 6, K)
