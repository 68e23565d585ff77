"""Where the K tile outside the pipeline of the matrix-core products is read from (``tail_chunk``, the code that the kernels inline, run on the host): every
chunk inside its operand and, shifted into place, made of the elements it stands for -- against the same in 64 bits, on operands on both sides of 2^31
and 2^32 elements.  Nothing is allocated: the arithmetic alone is looked at."""
import ctypes

import numpy as np
import pytest

from gemmkernels import _lib


def chunks(k_major, rows, cols, ld, rows_valid, tail_k):
    n = rows * cols // 8
    out = [np.empty(n, np.int32) for _ in range(3)]
    fn = _lib.lib().gk_internal_tail_chunks
    fn.restype = None
    fn(k_major, rows, cols, ctypes.c_int32(ld), ctypes.c_int32(rows_valid), tail_k, *(x.ctypes.data_as(ctypes.c_void_p) for x in out))
    return (x.astype(np.int64) for x in out)


def check(k_major, tile, block_k, extent, ld, at, tail_k):
    """The tile from row ``at`` of the ``extent`` rows (along M or N) of an operand, and its last ``tail_k`` of all k."""
    rows, cols = (tile, block_k) if k_major else (block_k, tile)
    left = extent - at
    start, shift, keep = chunks(int(k_major), rows, cols, ld, left, tail_k)
    row, col = (x.ravel().astype(np.int64) for x in np.meshgrid(np.arange(rows), np.arange(0, cols, 8), indexing="ij"))
    end = (left - 1) * ld + tail_k if k_major else (tail_k - 1) * ld + left
    where = (k_major, tile, block_k, extent, ld, at, tail_k)
    assert (shift >= 0).all() and (shift <= 7).all(), where
    assert (start + 8 <= end).all(), where
    # (the operand starts `at` rows in front of the tile, and the k in front of the tail)
    assert (start >= -(at * ld if k_major else at) - (0 if tail_k == block_k else 8 * ld if not k_major else 8)).all(), where
    k, r = (col, row) if k_major else (row, col)
    for e in range(8):
        ke, re = (k + e, r) if k_major else (k, r + e)
        stored = (ke < tail_k) & (re < left)
        kept = e < keep
        assert (kept[re < left] == (ke < tail_k)[re < left]).all(), where
        assert ((start + shift + e)[stored] == (row * ld + col + e)[stored]).all(), where
        assert ((shift + e)[stored] < 8).all(), where


# BLOCK_M or BLOCK_N, BLOCK_K, rows of the operand, its leading dimension: the products that a bound in 32 bits sent out of their operands among them
WIDE = [(256, 64, 131072, 16400), (256, 64, 65536, 50264), (64, 64, 50000, 50001), (128, 32, 131072, 16400), (128, 64, 2 ** 31 // 16392 + 1, 16392),
        (64, 64, 2 ** 31 // 4104, 4104), (64, 64, 2 ** 31 // 4104 + 1, 4104), (192, 64, 2 ** 32 // 8008, 8008), (256, 64, 2 ** 32 // 8008 + 1, 8008),
        (256, 64, 3000, 2 ** 22 - 8), (64, 64, 129, 2 ** 24 - 8), (64, 32, 2 ** 31 - 8, 8), (256, 32, 2 ** 28, 16)]


@pytest.mark.parametrize("case", range(len(WIDE)))
def test_rows_of_k_on_operands_of_any_size(case):
    tile, block_k, extent, ld = WIDE[case]
    last = (extent - 1) // tile * tile
    for at in sorted({0, tile, last // 2 // tile * tile, max(last - tile, 0), last}):
        for tail_k in (1, 7, 8, 9, 16, block_k - 1, block_k):
            if tail_k <= ld:
                check(True, tile, block_k, extent, ld, at, tail_k)


@pytest.mark.parametrize("tile,block_k", [(64, 32), (64, 64), (128, 64), (192, 64), (256, 64)])
@pytest.mark.parametrize("extent", [8, 9, 67, 255, 256, 257, 1003, 2 ** 23 - 1])
def test_both_orders(tile, block_k, extent):
    last = (extent - 1) // tile * tile
    for at in sorted({0, max(last - tile, 0), last}):
        for tail_k in (1, 5, 8, block_k - 7, block_k):
            for ld in (extent, extent + 1, extent + 5):
                check(False, tile, block_k, extent, ld, at, tail_k)
            for ld in (tail_k + 8, 1001):
                check(True, tile, block_k, extent, ld, at, tail_k)
