"""Products on tiles of 224 and 160 rows and 256 columns: full, one row over and one short, columns that end inside a tile, short last stages;
every epilogue.  Against fp64 on the bf16 operands."""
import pytest
import torch

from tests import test_tile_rows_gpu as by_rows
from tests.test_product_tiles_cpu import tiling

#: rows, columns, K, rows of a tile
SHAPES = [(4160, 2304, 200, 160), (4161, 2304, 768, 160), (4159, 2304, 456, 160), (4200, 2288, 768, 160), (4928, 2496, 200, 224),
          (4929, 2496, 768, 224), (4927, 2496, 456, 224), (4900, 2480, 456, 224), (1345, 8832, 200, 224)]


def test_which_tiles():
    for M, N, K, rows in SHAPES:
        assert tiling(M, N, K) == ("256x256", 1) and by_rows.tile_rows(M, N, K) == rows, (M, N, K, tiling(M, N, K), by_rows.tile_rows(M, N, K))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,rows", SHAPES)
def test_against_fp64(M, N, K, rows):
    by_rows.test_against_fp64(M, N, K, rows)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,rows", SHAPES)
def test_gated(M, N, K, rows):
    by_rows.test_gated(M, N, K)
