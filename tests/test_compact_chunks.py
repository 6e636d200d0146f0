"""Length of the chunks that the compact kernel's list cuts long block rows into, as the width of the product grows (host
function): what a wavefront's place on the device does in one panel of 64 columns, or a share of what it does in all."""
import ctypes as C

import pytest

from smat_amd._lib import lib

PLACES = 16 * 256

_fn = lib.smat_internal_compact_chunk
_fn.restype = C.c_long
_fn.argtypes = [C.c_long, C.c_size_t, C.c_long, C.c_size_t]


@pytest.mark.parametrize("steps", [0, 4096, 30 * PLACES, 120 * PLACES, 240 * PLACES])
def test_no_jump_from_one_panel_to_the_next(steps):
    rows, longest = 65536, 1 << 20
    chunks = [_fn(steps, rows, longest, 8 * n) for n in range(1, 130)]
    panels = [(8 * n + 63) // 64 for n in range(1, 130)]
    share = steps / PLACES
    for a, b, p, q in zip(chunks, chunks[1:], panels, panels[1:]):
        # a panel more is never a shorter chunk, and no longer one than its share of the steps (rounding: 1)
        assert a <= b <= a + (0.38 * share if q > p else 0) + 1
    assert chunks[7] == _fn(steps, rows, longest, 128)  # one and two panels: the chunk that ends with its panel
    assert abs(chunks[0] - max(16 + share, 2.5 * steps / rows)) <= 1


def test_which_lists_are_split():
    # not longer than four times the average (or 16 steps): whole
    assert _fn(80000, 10000, 32, 64) >= 32
    assert _fn(10000, 10000, 16, 64) >= 16
    assert _fn(9426, 967, 39, 1000) >= 39  # 4 x 9426 / 967 steps are 38.99, to the column 39
    # longer, but no longer than a chunk: whole
    assert _fn(240 * PLACES, 65536, 100, 1024) >= 100
    # longer than a chunk: split
    assert _fn(10000, 10000, 50, 64) < 50
    # too few wavefronts for the device: chunks of 56 steps at most, also of rows that are all alike
    assert _fn(500 * 100, 500, 100, 64) == 56
