"""The order of LDS reads and refills in the products' quadrant tiles (CPU).

A wave passes a sync of ``quad_tile`` (gemm.hip) with some of its own LDS reads still
pending; after it, any wave may refill a slot by a direct-to-LDS load. The stages are
played here read by read, with the counts that the source gives its syncs, and no slot
may be refilled while a read of it can be pending. Reads complete in order, and a
quadrant's MFMAs wait for the fragments they use; a quadrant that is left out (past a
ragged side, below the diagonal) waits for none.
"""

from __future__ import annotations

import itertools
import re
from pathlib import Path

import pytest

SOURCE = Path(__file__).resolve().parents[1] / "dionw_amd" / "csrc" / "gemm.hip"
TILES = {"BigTile": (4, 2), "MidTile": (2, 2)}  # FI, FJ


def _pending_counts(fi: int) -> list[int]:
    """The reads that the syncs allow, in the order of the source: a stage's start, its
    middle, before the last slot's refill, and before the first stage."""
    text = SOURCE.read_text()
    counts = re.findall(r"^ *QUAD_SYNC\(.*, (2 \* FI|\d+)\)$", text, re.MULTILINE)
    assert len(counts) == 4, counts
    return [2 * fi if c == "2 * FI" else int(c) for c in counts]


class _Wave:
    """Pending LDS reads of one wave, oldest first, by the slot they read."""

    def __init__(self) -> None:
        self.pending: list[str] = []
        self.at_sync: list[str] = []

    def read(self, slot: str, count: int) -> None:
        self.pending += [slot] * count

    def use(self, slot: str) -> None:
        """MFMAs of the fragments read from ``slot``."""
        if slot in self.pending:
            last = len(self.pending) - self.pending[::-1].index(slot)
            del self.pending[:last]

    def sync(self, allowed: int) -> None:
        if len(self.pending) > allowed:
            del self.pending[:len(self.pending) - allowed]
        self.at_sync = list(self.pending)

    def refill(self, slot: str) -> None:
        """Another wave's load, issued at any time since the last sync."""
        assert slot not in self.at_sync, f"{slot} is refilled while reads of it are pending"
        assert slot not in self.pending, f"{slot} is refilled after a read of it without a sync"


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("add", [False, True], ids=["plain", "addend"])
@pytest.mark.parametrize("kn", [False, True], ids=["nk", "kn"])
@pytest.mark.parametrize("stages", [2, 3, 4, 5])
def test_no_slot_is_refilled_under_a_read(tile: str, add: bool, kn: bool, stages: int) -> None:
    fi, fj = TILES[tile]
    start, middle, last, first = _pending_counts(fi)
    reads_a, reads_b = 2 * fi, 2 * fj * (2 if kn else 1)
    four = tile == "MidTile"  # its addend needs the A slots only
    # Which of the quadrants 0 1, 1 1 and 1 0 are multiplied.
    for skip_rows, skip_cols, diagonal in itertools.product((False, True), repeat=3):
        do01, do11 = not skip_cols, not skip_rows and not skip_cols
        do10 = not skip_rows and not diagonal
        w = _Wave()

        def slot(operand: str, half: int, stage: int) -> str:
            return f"{operand}{half} of buffer {(stage + stages) % 2}"

        w.sync(first)
        w.read(slot("B", 0, 0), reads_b)
        w.read(slot("A", 0, 0), reads_a)
        for kt in range(stages):
            a0, a1, b0, b1 = (slot(o, h, kt) for o, h in ("A0", "A1", "B0", "B1"))
            o_a1 = slot("A", 1, kt + 1)
            tail = max(0, kt - (stages - 3))
            w.sync(start)
            w.use(a0), w.use(b0)
            w.read(b1, reads_b)
            if tail != 2 or add:
                w.refill(o_a1)
            if do01:
                w.use(a0), w.use(b1)
            w.read(a1, reads_a)
            if tail == 0 or (add and not four):
                w.refill(b0)
            if tail != 2 or add:
                w.sync(middle)
            if do11:
                w.use(a1), w.use(b1)
            if tail == 0 or add:
                w.refill(a0)
            if tail != 2:
                w.read(slot("B", 0, kt + 1), reads_b)
            if tail == 2 and add:
                w.sync(last)
                w.refill(a1)
            if do10:
                w.use(a1), w.use(b0)
            if tail != 2:
                w.read(slot("A", 0, kt + 1), reads_a)
            if tail == 0 or (add and not four):
                w.refill(b1)
