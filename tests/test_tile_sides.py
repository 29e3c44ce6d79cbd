"""The extents that batches are iterated at (``newton_schulz.tile_sides``), on the CPU."""

from __future__ import annotations

import ctypes

import pytest

from dionw_amd import _lib
from dionw_amd.newton_schulz import padded_sides, prepared_orientations, tile_sides


@pytest.mark.parametrize(("blocks", "rows", "cols"), [
    (1, 1, 1), (1, 1, 128), (3, 500, 1301), (3, 1301, 500), (6, 50, 200), (6, 200, 200),
    (12, 64, 64), (5, 63, 65), (128, 352, 2048), (1, 65, 64), (64, 1408, 2048),
])
def test_sides_are_whole_tiles(blocks: int, rows: int, cols: int) -> None:
    """Multiples of 64 that hold the block, the short side no longer than the long
    one, only the wide orientation prepared, and a call that the library plans."""
    p_pad, j_pad = sides = tile_sides(blocks, rows, cols)
    assert p_pad % 64 == j_pad % 64 == 0 and 0 <= p_pad - rows < 64 and 0 <= j_pad - cols < 64
    r, c = (j_pad, p_pad) if rows > cols else (p_pad, j_pad)
    assert r <= c
    assert prepared_orientations(rows, cols, sides) == ((False, True) if rows > cols
                                                        else (True, False))
    i64 = ctypes.c_int64
    for kind in (0, 2):
        assert _lib.library().dionw_newton_schulz_group_launches(
            1, (ctypes.c_int32 * 1)(kind), (i64 * 1)(blocks), (i64 * 1)(r), (i64 * 1)(c),
            (i64 * 1)(min(rows, cols)), (i64 * 1)(max(rows, cols))) > 0


@pytest.mark.parametrize(("blocks", "rows", "cols"), [
    (100000, 8, 64), (1 << 20, 8, 8), (1, 65500, 65500), (1, 65500, 70000),
])
def test_other_batches_keep_their_sides(blocks: int, rows: int, cols: int) -> None:
    """Many thin blocks, and sides that would pass the library's limit of 65535."""
    assert tile_sides(blocks, rows, cols) == padded_sides(rows, cols)
