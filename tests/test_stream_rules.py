"""Which streamed products share their rows between several tiles of columns,
and how far ahead of its sums a wave loads: no choice that is slower than the one
before it.  Each line was measured on both sides, us."""
import pytest

from ollamamq_amd.ops import hip


@pytest.mark.parametrize("M, N, K, gated, tiles", [
    # up to 32 rows: a last round of eight tiles a block that is nearly full
    (32, 73728, 4096, True, 1),         # 97, with eight 126
    (25, 65600, 4096, False, 1),        # 96, with eight 111
    (32, 102400, 4096, True, 1),        # 135, with eight 144
    (32, 81920, 3584, False, 1),        # 103, with eight 111
    (32, 139264, 4096, False, 1),       # 200, with eight 216
    (32, 128256, 4096, False, 8),       # 183, with eight 172
    (32, 152064, 3584, False, 8),       # 201, with eight 193
    (32, 102400, 3584, False, 8),       # 132, with eight 122
    (32, 65536, 3584, True, 8),         # 77, with eight 75
    (32, 22016, 4096, True, 3),         # 34, with three 32
    (24, 22016, 4096, True, 1), (32, 28672, 4096, True, 1),
    # more rows: three tiles only of a K that has them divided ...
    (33, 24576, 512, True, 4),          # 9.9, with three 11.1
    (64, 20480, 1024, True, 4),         # 14.3, with three 14.9
    (33, 24576, 1792, True, 4),         # 20.3, with three 21.3
    (64, 22016, 4096, True, 3),         # 36.9, with four 38.1
    # ... and eight where the weights' reads are what is left
    (64, 49152, 4096, True, 8),         # 68.6, with six 72.2
    (33, 57344, 3584, True, 8),         # 68.3, with seven 71.8
    (128, 53248, 4096, True, 7),        # 79.1, with eight 83.1
    (64, 49152, 1024, True, 6),         # 23.6, with eight 28.3
    (64, 37888, 3584, True, 5), (128, 28672, 4096, True, 4),
    (97, 65568, 4096, False, 4),        # 144, with eight 172
    (128, 73728, 3584, True, 4),        # 134, with eight 143
])
def test_tiles(M, N, K, gated, tiles):
    hip.require()
    assert hip._lib.wstream_wide_tiles(M, N, K, gated) == tiles


@pytest.mark.parametrize("M, N, K, parts, ahead", [
    (32, 3584, 3584, 2, 2),             # 9.7, one 9.9
    (32, 2048, 2048, 2, 2),             # 6.9, one 7.2
    (17, 4096, 1024, 1, 2), (32, 4096, 1920, 1, 2),
    (32, 8192, 1024, 1, 1),             # 5.9, two 6.1: a block a CU
    (32, 3072, 3072, 2, 1),             # 8.8, two 9.1: three iterations
    (16, 3584, 3584, 2, 1), (32, 4096, 512, 1, 1), (32, 18432, 3072, 1, 1),
    (1, 4096, 4096, 2, 4), (32, 28672, 4096, 1, 4),
])
def test_iterations_ahead(M, N, K, parts, ahead):
    hip.require()
    assert hip._lib.wstream_depth(M, N, K, parts) == ahead


def test_none():
    hip.require()
    for bad in ((0, 64, 64), (129, 64, 64), (1, 16, 64), (1, 64, 32)):
        assert hip._lib.wstream_wide_tiles(*bad, False) < 0
    for bad in ((0, 64, 64, 1), (33, 64, 64, 1), (1, 16, 64, 1),
                (1, 64, 64, 0)):
        assert hip._lib.wstream_depth(*bad) < 0


@pytest.mark.parametrize("M,N,K,ks,how", [
    # us in parts and in blocks of 16 columns ...
    (1, 4096, 4096, 2, 1), (32, 4096, 4096, 2, 1),      # 9.8 7.2, 10.6 9.7
    (8, 4096, 14336, 2, 1),                             # 22.8 21.3
    (8, 3584, 18944, 2, 1),                             # 26.0 25.7
    (32, 2048, 5632, 4, 0), (32, 2048, 2048, 2, 1),     # 9.6 11.8, 7.0 5.9
    (1, 4608, 1024, 1, 0), (16, 4096, 1024, 1, 1),      # 5.1 5.4, 5.2 4.4
    (48, 4096, 4096, 2, 1), (64, 2048, 2048, 2, 1),     # 13.9 12.3, 9.1 8.4
    (48, 2048, 5632, 4, 0), (64, 5120, 3584, 2, 0),     # 11.9 13.9, 20.5 22.2
    (65, 2048, 2048, 2, 0), (49, 1024, 1024, 1, 0), (48, 1024, 1024, 1, 1),
    # ... and of 64
    (32, 4096, 14336, 2, 4), (45, 4096, 14336, 2, 4),   # 24.3 23.1, 28.4 25.8
    (16, 3584, 18944, 2, 4), (45, 3584, 18944, 2, 4),   # 26.9 25.9, 35.2 30.6
    (1, 5120, 13824, 2, 3), (45, 4096, 11008, 2, 4),    # 33.9 27.2, 24.4 22.3
    (8, 8192, 28672, 1, 0), (32, 8192, 28672, 1, 2),    # 75.9 77.8, 80.7 75.3
    (32, 2048, 8192, 4, 0), (49, 4096, 14336, 2, 0),    # 11.5 11.7
    (32, 4128, 14336, 2, 0),
])
def test_residual(M, N, K, ks, how):
    hip.require()
    assert hip._lib.wstream_residual(M, N, K, ks) == how


@pytest.mark.parametrize("M,N,K,narrow", [
    # us in blocks of 32 columns and of 16
    (1, 8448, 4096, True), (16, 8448, 4096, True),      # 18.8 15.6, 20.2 18.0
    (1, 12288, 4096, True), (16, 12288, 8192, True),    # 20.3 17.5, 40.0 36.9
    (1, 8448, 1792, True), (16, 12288, 2048, True),     # 9.9 8.8, 12.6 11.8
    (1, 8448, 512, False), (16, 12288, 512, False),     # 4.9 7.1, 6.0 8.7
    (1, 8448, 1024, False), (16, 12288, 1024, False),   # 6.9 7.7, 8.0 9.8
    (16, 10240, 1536, False),                           # 10.3 10.6
    (16, 13312, 4096, False), (8, 15360, 5120, False),  # 21.6 23.8, 26.8 28.1
    (16, 16384, 8192, False), (8, 12416, 4096, False),  # 45.6 47.7
    (1, 8192, 4096, False), (17, 12288, 4096, False), (0, 8448, 4096, False),
    (1, 8464, 4096, False),                             # no whole tiles
])
def test_rotated(M, N, K, narrow):
    hip.require()
    assert hip._lib.wstream_rope_narrow(M, N, K) == narrow


@pytest.mark.parametrize("M,N,K,ks,how", [
    # where the weights' own time is what is left: us streamed and in 64 columns
    (9, 8192, 28672, 1, 0), (16, 8192, 28672, 1, 0),    # 69.7 71.9, 69.9 72.4
    (24, 8192, 28672, 1, 2), (16, 3584, 18944, 2, 4),   # 72.1 71.4, 24.9 25.0
    # more parts of 64 columns are more to add up
    (48, 512, 18944, 8, 0), (24, 512, 18944, 8, 0),     # 15.1 22.1, 11.7 15.9
    (48, 1024, 28672, 8, 0), (45, 1536, 8960, 8, 10),   # 20.2 22.7, 17.3 15.5
    # short K: us streamed and in 16 columns; over tiles and in 16 columns
    (32, 4096, 256, 1, 0), (24, 1536, 128, 1, 0),       # 4.5 5.1, 4.1 4.8
    (32, 3584, 512, 1, 0), (32, 1024, 1024, 1, 1),      # 5.0 5.8, 5.3 5.2
    (64, 3584, 256, 1, 0), (64, 3584, 3584, 2, 1),      # 5.2 6.8, 14.1 11.0
    # few rows: parts of few tiles
    (1, 1536, 8960, 8, 0), (9, 2048, 5632, 4, 0),       # 10.6 10.9, 9.0 9.2
])
def test_residual_sizes(M, N, K, ks, how):
    hip.require()
    assert hip._lib.wstream_residual(M, N, K, ks) == how
