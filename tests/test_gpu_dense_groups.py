"""Tiles of 160 to 224 rows whose last raster group would be a single tile (csrc/gemm_kernel.h gemmr_group: groups of five, of six at 21 tiles, of nine): every tile once, the bits of
256 rows as test_gpu_dense_short_tiles.py has them."""
import pytest

import test_gpu_dense_short_tiles as short

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,rows", [(1286, 5632, 160), (1605, 6144, 192), (1924, 6144, 224), (2417, 4352, 192), (4012, 2560, 192), (3606, 11008, 224)])
def test_rows(M, N, rows):
    tiles, group = -(-M // rows), 8 if N // 256 >= 32 else 4
    assert tiles > group and tiles % group == 1
    short.test_rows_by_columns(M, N, rows)


@pytest.mark.parametrize("Mp,N,rows,Tm", [(2304, 4096, 160, 768), (3328, 4096, 224, 3328), (2304, 9216, 192, 256), (5376, 5120, 224, 1792)])
def test_transposed(Mp, N, rows, Tm):
    tiles, group = Mp // 256, 8 if -(-N // rows) >= 32 else 4
    assert tiles > group and tiles % group == 1
    short.test_transposed(Mp, N, rows, Tm)
