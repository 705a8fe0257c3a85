"""The tiles of the projection kernel (csrc/hsa_linear.hip) on the host: every result belongs to one, none reaches outside."""
import ctypes

import numpy as np
import pytest

from sparseattention_amd import _lib


class Segment(ctypes.Structure):
    _fields_ = ([(n, ctypes.c_void_p) for n in ("x", "w", "bias", "out")]
                + [(n, ctypes.c_int64) for n in ("ld_x", "ld_w", "ld_out", "batch_x", "batch_out")]
                + [(n, ctypes.c_int) for n in ("batches", "rows", "cols")])


def _segment(B, R, N, K, ld, first=0):
    """Addresses of nothing: only their alignment counts."""
    return Segment(1 << 20, 2 << 20, None, (3 << 20) + 2 * first, K, K, ld, R * K, (R + 1) * ld, B, R, N)


def _rectangles(tile, K, *segs):
    arr, room = (Segment * len(segs))(*segs), 1 << 16
    out = np.zeros((room, 8), dtype=np.int32)
    n = _lib.lib().hsa_linear_rectangles(len(segs), arr, K, 0, tile, out.ctypes.data, room)
    assert 0 < n <= room, n
    return out[:n]


def _covered(rects, *segs):
    for i, s in enumerate(segs):
        r = rects[rects[:, 0] == i]
        r = r[np.lexsort((r[:, 5], r[:, 2], r[:, 1]))]
        step, rows, width = r[0, 3], r[0, 4], r[0, 6]
        begins = np.ones(len(r), bool)  # of a row block's columns
        begins[1:] = (r[1:, 1:3] != r[:-1, 1:3]).any(1)
        ends = np.append(begins[1:], True)
        assert (r[begins, 5] == 0).all() and (r[ends, 5] + width == s.cols).all()
        assert (r[1:, 5][~begins[1:]] <= r[:-1, 5][~begins[1:]] + width).all()
        seen = np.zeros((s.batches, s.rows), bool)
        blocks = r[begins]
        at = blocks[:, 2:3] + step * np.arange(rows)[None]
        assert at.min() >= 0 and at.max() < s.rows and (blocks[:, 1] >= 0).all() and (blocks[:, 1] < s.batches).all()
        seen[np.broadcast_to(blocks[:, 1:2], at.shape), at] = True
        assert seen.all()


@pytest.mark.parametrize("period", [2, 4, 8, 16, 32, 64])
def test_rows_that_lie_alike_in_lines(period):
    """Results whose rows begin anywhere, in tiles of every period-th row: all remainders of the columns, places in a
    line and row counts around whole tiles."""
    for cols in range(7937, 7937 + 256):
        ld = next(n for n in range(cols, cols + 129) if 64 // np.gcd(n, 64) == period)
        many = cols % 37 == 0
        for first in (0, 1, 31, 58, 63) if many else (0, 63 - cols % 3):
            for rows in (256 * period, 1792 * period + 1, 7 * 257 * period + 3) if many else (256 * period,):
                s = _segment(1, rows, cols, 128, ld, first)
                r = _rectangles(4, 128, s)
                assert (r[:, 3] == period).all()
                _covered(r, s)


@pytest.mark.parametrize("rows,cols,period", [
    (32768, 50257, 64), (28672, 50257, 64), (24576, 50257, 1), (20480, 50257, 1), (16384, 50257, 64), (12288, 50257, 1),
    (8192, 50258, 32), (10240, 50258, 1), (4096, 50260, 16), (5120, 50260, 1), (7168, 50260, 16), (32768, 3001, 1),
    (32768, 8001, 64)])
def test_rows_that_lie_alike_do_not_multiply_the_tiles(rows, cols, period):
    s = _segment(1, rows, cols, 512, cols)
    r = _rectangles(4, 512, s)
    assert (r[:, 3] == period).all() and len(r) <= 1.15 * -(-rows // 256) * -(-cols // 256)
    _covered(r, s)


@pytest.mark.parametrize("tile,rows,cols", [(0, 256, 256), (1, 256, 192), (2, 128, 128), (4, 256, 256)])
def test_consecutive_rows(tile, rows, cols):
    for B, R, N in ((1, rows, cols), (3, rows + 1, cols + 8), (2, 5 * rows - 1, 3 * cols - 8), (1, 40 * rows + 7, 2 * cols)):
        segs = [_segment(B, R, N, 192, N + 8, 8), _segment(1, R + 1, N + 8, 192, N + 8)]
        _covered(_rectangles(tile, 192, *segs), *segs)


@pytest.mark.parametrize("rows,apart", [(2048, 16), (4096, 8), (5111, 8), (5120, 8), (8192, 8), (10240, 8), (14336, 8), (18432, 8),
                                        (20480, 8)])
@pytest.mark.parametrize("cols", [7001, 30001, 48305])
def test_walks_of_rows_through_the_lds_begin_apart(rows, cols, apart):
    """The eight XCDs' walks: every tile once, and at any time columns about an eighth apart (a sixteenth where two share a
    row of tiles): in step, all eight ask for the same weights at once."""
    s = _segment(1, rows, cols, 256, cols)
    r = _rectangles(4, 256, s)
    _covered(r, s)
    assert len(np.unique(r[:, [2, 5]], axis=0)) == len(r)
    starts = np.array([r[r[:, 7] == xcd][0, 5] for xcd in range(8)])
    gaps = np.diff(np.append(np.sort(starts), np.sort(starts)[0] + cols))
    assert (gaps >= cols / apart - 3 * 256).all(), starts
