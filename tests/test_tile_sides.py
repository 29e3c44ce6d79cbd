"""The extents that batches are iterated at (``newton_schulz.tile_sides``), on the CPU."""

from __future__ import annotations

import ctypes

import pytest

from dionw_amd import _lib
from dionw_amd.newton_schulz import (
    PAD_SCRATCH,
    SCRATCH_PER_ELEMENT,
    NewtonSchulz,
    newton_schulz_fn,
    padded_sides,
    prepared_orientations,
    tile_sides,
)


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


def _planned(blocks: int, r: int, c: int, rows: int, cols: int) -> bool:
    """Whether the library plans a call of each kind at these extents."""
    i64 = ctypes.c_int64
    return all(_lib.library().dionw_newton_schulz_group_launches(
        1, (ctypes.c_int32 * 1)(kind), (i64 * 1)(blocks), (i64 * 1)(r), (i64 * 1)(c),
        (i64 * 1)(min(rows, cols)), (i64 * 1)(max(rows, cols))) > 0 for kind in (0, 2))


@pytest.mark.parametrize(("blocks", "rows", "cols"), [
    (100000, 8, 64), (1 << 20, 8, 8), (1, 65500, 65500), (1, 65500, 70000),
])
def test_other_batches_keep_their_sides(blocks: int, rows: int, cols: int) -> None:
    """Many thin blocks, and sides that would pass the library's limit of 65535."""
    sides = tile_sides(blocks, rows, cols)
    assert sides == padded_sides(rows, cols)
    assert min(sides) < 65536 and _planned(blocks, min(sides), max(sides), rows, cols)


def _held(blocks: int, rows: int, cols: int) -> int:
    """Bytes of a Gram call's buffers, from the library's workspace."""
    sides = tile_sides(blocks, rows, cols)
    inputs = sum(prepared_orientations(rows, cols, sides)) * 2 * blocks * sides[0] * sides[1]
    lib_kind = newton_schulz_fn(NewtonSchulz.GRAM).lib_kind
    return inputs + 2 * blocks * rows * cols + int(_lib.library().dionw_newton_schulz_workspace(
        lib_kind, blocks, min(sides), max(sides)))


@pytest.mark.parametrize(("rows", "cols"), [
    (16, 64), (64, 16), (40, 40), (40, 160), (65, 65), (72, 80), (80, 2560), (96, 96), (160, 130),
    (200, 200), (24, 1000), (8, 8), (1, 64), (250, 333),
])
def test_padding_stays_within_its_memory(rows: int, cols: int) -> None:
    """At any number of blocks up to a run's 2^30 elements the buffers stay within 20
    bytes per element (sides rounded up to 8) or 8 GiB; and thin batches that fit are
    padded."""
    plain = (rows + 7) // 8 * 8 * ((cols + 7) // 8 * 8)
    assert all(n % 64 == 0 for n in tile_sides(4, rows, cols))
    most = min(65535, 2**30 // (rows * cols))
    for blocks in sorted({*(most >> s for s in range(17)), most, most * 2 // 3} - {0}):
        assert _held(blocks, rows, cols) <= max(SCRATCH_PER_ELEMENT * blocks * plain, PAD_SCRATCH)


@pytest.mark.parametrize(("rows", "cols"), [(40, 40), (72, 65), (16, 64)])
def test_more_blocks_than_ragged_depths_take_are_padded(rows: int, cols: int) -> None:
    """Products of a depth that is no multiple of 32 take at most 65535 blocks."""
    assert all(n % 64 == 0 for n in tile_sides(100000, rows, cols))
