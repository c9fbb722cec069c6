"""Products of many columns with every number of tiles a block, three to eight
in one round of blocks and the last block short of some; up to 32 rows from 25
on.  Tolerance: see test_wide_batches_gpu.py."""
import pytest

from test_wide_batches_gpu import test_many_columns as many_columns

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M, tiles, K", [
    (33, 601, 192), (128, 767, 64), (96, 700, 3136),        # four; three
    (64, 1022, 128), (97, 897, 576),                        # four
    (64, 1184, 576), (128, 1279, 64), (65, 1026, 192),      # five
    (96, 1400, 192), (33, 1535, 64), (128, 1283, 128),      # six
    (128, 1700, 64), (65, 1790, 192), (40, 1537, 576),      # seven
    (40, 2043, 192), (127, 1801, 64),                       # eight
    # up to 32 rows: the stream, and three, five and seven; eight of one round
    (24, 577, 3072), (25, 577, 3072), (32, 1183, 3136), (28, 1540, 3072),
    (32, 2051, 3072), (31, 1025, 3008), (32, 2048, 3072),
    # three of a K that takes them, and six and seven beside the others' limits
    (33, 601, 2112), (128, 767, 2048), (64, 1460, 192), (96, 1610, 1088),
    (128, 1790, 1088)])
def test_tiles(M, tiles, K):
    many_columns(M, tiles, K)
