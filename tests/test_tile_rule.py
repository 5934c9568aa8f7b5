"""The rule that picks the tile of a grouped GEMM, on the CPU: the shapes that
were fastest where it was measured (a device of 256 CUs)."""
import pytest

from hanuman_amd import _lib
from hanuman_amd import kernels as K

CUS = 256
GATE_UP = {  # (experts, d_model, d_ff): rows an expert -> rows of the tile
    (64, 2048, 1024): {1: 32, 6: 32, 42: 64, 96: 128, 256: 256, 2048: 256},
    (80, 1536, 768): {33: 64, 100: 128, 140: 256, 190: 256, 205: 256},
    (32, 4096, 2048): {16: 32, 80: 128, 140: 256, 160: 256, 190: 256},
    (16, 1024, 2048): {32: 64, 125: 256, 190: 256, 250: 256},
    # one segment: a shared expert
    (1, 1536, 768): {333: 64, 4096: 128},
    (1, 2048, 1024): {1: 32, 2000: 128, 16384: 256},
}


@pytest.mark.parametrize("shape", GATE_UP, ids=str)
def test_tile_by_rows(shape):
    n, d, f = shape
    for rows, want in GATE_UP[shape].items():
        assert K.grouped_tile(rows * n, n, 2 * d, 2 * f, CUS)[0] == want, (shape, rows)


def test_tiles_fit():
    """Every tile divides the columns, and many rows take 256 x 256."""
    for n in (2, 16, 64, 256):
        for kb, cols in ((256, 256), (4096, 2048), (8192, 4096), (1536, 768)):
            for rows in (1, 5, 40, 100, 200, 300, 400, 600, 1000, 5000, 100000):
                bm, bn = K.grouped_tile(rows * n, n, kb, cols, CUS)
                assert cols % bn == 0 and bm in (32, 64, 128, 256)
            assert (bm, bn) == (256, 256)


def test_query_checks():
    for args in ((0, 8, 128, 256, 256), (8, 0, 128, 256, 256), (8, 1025, 128, 256, 256),
                 (8, 8, 100, 256, 256), (8, 8, 128, 300, 256), (8, 8, 128, 256, 0)):
        with pytest.raises(_lib.HmoeError) as ei:
            K.grouped_tile(*args)
        assert ei.value.code == _lib.ERR_INVALID
