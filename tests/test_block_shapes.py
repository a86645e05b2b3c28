"""Which blocks a product over a matrix in fragment order takes: what the rule names for sizes on both sides of its
lines, asked on the host (the kernels' launches go through the same functions)."""
import ctypes

import pytest

# the numbers of csrc/gemm.hip; 0: the kernel with 32 x 32 tiles
SHAPES = {"rows32": 0, "256x256": 5, "256x192": 9, "256x128": 12, "192x128": 11, "128x128": 8, "64x128": 13,
          "128x64": 14, "64x64": 15}
# whole products with bfloat16 results: M, N, K
WHOLE = {(2048, 16384, 512): "256x256", (2048, 6144, 640): "256x192", (512, 16384, 512): "256x128",
         (575, 9216, 512): "192x128", (700, 3072, 1024): "128x128", (129, 16384, 1024): "128x128",
         (160, 10240, 1024): "64x128", (575, 3072, 1024): "128x64", (417, 3072, 2048): "128x64",
         (257, 4096, 1024): "128x64", (256, 4096, 1024): "64x64", (300, 1024, 256): "64x64"}
# 25 to 128 rows: M, rows of W, K, ranges, bytes of a result, gated
FEW = {(128, 1024, 768, 3, 4, 0): "rows32", (64, 9216, 768, 1, 2, 1): "rows32",     # (a short K)
       (32, 65536, 1024, 1, 4, 0): "rows32", (32, 24576, 1792, 1, 2, 1): "rows32",  # (very wide, up to 32 rows)
       (32, 16384, 1024, 1, 2, 1): "64x64", (32, 65536, 2048, 1, 4, 0): "64x64",
       (25, 256, 1024, 4, 4, 0): "rows32", (32, 64, 1024, 1, 2, 0): "rows32",       # (the smallest)
       (25, 512, 1024, 4, 4, 0): "64x64", (33, 256, 1024, 4, 4, 0): "64x64",
       (64, 4096, 4096, 1, 2, 1): "64x64", (100, 4096, 4096, 1, 2, 1): "64x64",     # (a long K, up to 128 rows)
       (129, 4096, 4096, 1, 2, 1): "128x128", (64, 8192, 8192, 2, 4, 0): "64x64",
       (128, 8192, 8192, 2, 4, 0): "128x64", (64, 21504, 2048, 1, 2, 1): "64x128",
       (64, 40960, 2048, 1, 2, 1): "64x64", (65, 40960, 2048, 1, 2, 1): "128x128"}  # (more blocks than CUs)


def shape_of(M, n_rows, K, split, elem, gated):
    from kappai_amd.kernels.lib import library
    return library("engine").kappai_block_shape_of(*map(ctypes.c_int, (M, n_rows, K, split, elem, gated)))


@pytest.mark.parametrize("sizes", list(WHOLE))
def test_blocks_of_a_whole_product(sizes):
    assert shape_of(*sizes, 1, 2, 0) == SHAPES[WHOLE[sizes]]


def test_every_form_is_chosen():
    assert set(WHOLE.values()) == set(SHAPES) - {"rows32"}


@pytest.mark.parametrize("sizes", list(FEW))
def test_blocks_of_25_to_128_rows(sizes):
    assert shape_of(*sizes) == SHAPES[FEW[sizes]]
