"""Which kernel the expert products run on (moe_expert_tiles, host code, no
GPU), at shapes measured on both: rows an expert against the line between the
grouped GEMM (128) and the row-tile kernel (16, 32 or 64)."""
import ctypes

import pytest

from tests.helpers import expert_tiles

# (op, x, E, k, d, I, rows an expert, GEMM): µs on the GEMM and in row tiles.
MEASURED = [
    ("layer", "f16", 64, 8, 2048, 1408, 64, True),     # 229, 239
    ("layer", "f16", 64, 8, 2048, 1408, 512, True),    # 884, 1199
    ("layer", "f16", 32, 4, 2048, 5632, 64, True),     # 361, 473
    ("layer", "f16", 64, 8, 2048, 768, 96, True),      # 162, 187
    ("layer", "f16", 64, 8, 2048, 1000, 96, True),     # 205, 239
    ("layer", "f16", 64, 4, 768, 2816, 96, True),      # 205, 282
    ("layer", "f16", 64, 8, 1024, 768, 80, True),      # 92, 111
    ("layer", "f16", 64, 8, 640, 640, 96, True),       # 79, 89
    ("layer", "f16", 64, 8, 640, 640, 128, False),     # 120, 99
    ("layer", "f16", 8, 2, 640, 640, 128, False),      # 69, 46
    ("layer", "f16", 8, 2, 1024, 1024, 96, False),     # 82, 57
    ("layer", "f16", 8, 1, 768, 1024, 256, False),     # 92, 80
    ("layer", "f16", 32, 4, 512, 1024, 512, False),    # 169, 168; up alone is not the GEMM's
    ("layer", "f32", 8, 2, 2048, 1408, 96, False),     # 167, 110
    ("layer", "f32", 64, 8, 2048, 1408, 96, True),     # 366, 376
    ("layer", "f32", 64, 8, 640, 640, 192, True),      # 152, 145
    ("up", "f16", 16, 2, 2048, 5632, 96, True),        # 139, 177
    ("up", "f16", 16, 2, 1024, 768, 64, False),        # 37, 27
    ("up", "f32", 16, 2, 1024, 768, 512, True),        # 80, 100
    ("up", "f32", 64, 4, 2048, 1408, 128, False),      # 375, 299
    ("down", "f32", 16, 2, 2048, 5632, 128, True),     # 163, 219
    ("down", "f32", 64, 4, 2048, 1408, 96, True),      # 118, 135
    ("down", "f32", 64, 4, 2048, 1408, 128, False),    # 194, 169
    ("down", "f32", 128, 4, 640, 640, 512, False),     # 237, 233
]


@pytest.mark.parametrize("op,x,E,k,d,I,rows,gemm", MEASURED)
def test_grouped_gemm_where_it_is_faster(op, x, E, k, d, I, rows, gemm):
    up, down = expert_tiles(op, rows * E // k, d, I, E, k, x)
    if op != "down":
        assert (up == 128) == gemm
    # int8 down takes K = I in whole steps of 32
    if op != "up":
        assert (down == 128) == (gemm and I % 32 == 0)


@pytest.mark.parametrize("x", ["f32", "f16"])
@pytest.mark.parametrize("op", ["layer", "up", "down"])
def test_never_the_gemm_below_64_rows(op, x):
    for E, k, d, I in [(64, 8, 2048, 1408), (32, 4, 2048, 5632), (8, 2, 640, 640)]:
        for rows in (1, 8, 40, 63):
            tiles = expert_tiles(op, rows * E // k, d, I, E, k, x)
            assert 128 not in tiles, (E, k, d, I, rows)
        # calls of a batch keep to the row tiles and the decode kernels
        assert 128 not in expert_tiles(op, 256 * E // k, d, I, E, k, x, calls=2)


def test_bad_arguments_are_refused():
    from runntime_amd import _lib
    a, b = ctypes.c_int(), ctypes.c_int()
    assert _lib.load().moe_expert_tiles(3, 1, 0, 1, 8, 8, 1, 1, 8, 8, 8, a, b) != 0
    assert _lib.load().moe_expert_tiles(0, 1, 0, 1, 8, 8, 1, 1, 8, 8, 8, None, b) != 0
