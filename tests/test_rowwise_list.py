"""Work list of the row-wise kernel's plans, on the CPU: which block rows are cut, into what, and the order of the items."""
import ctypes as C

import numpy as np
import pytest

from smat_amd._lib import lib


def rowwise_list(row_ptr, N):
    """(items [n, 4]: block row, first block, end, slot or -1; cut rows; slots) of a plan of N columns."""
    rp = np.ascontiguousarray(row_ptr, np.int32)
    items, counts = np.zeros((len(rp) + int(rp[-1]), 4), np.int32), (C.c_int64 * 3)()
    fn = lib.smat_internal_rowwise_list
    fn.argtypes = [C.c_void_p, C.c_size_t, C.c_size_t, C.c_void_p, C.c_size_t, C.c_void_p]
    assert fn(rp.ctypes.data, len(rp) - 1, N, items.ctypes.data, len(items), counts) == 0
    return items[:counts[0]], counts[1], counts[2]


def row_ptr(lengths):
    return np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)


def power_law(n, top):
    return (top / np.arange(1, n + 1)).astype(int)


@pytest.mark.parametrize("N", [8, 64, 136, 1024])
@pytest.mark.parametrize("lengths", [[0], [7], [64] * 40, [60] * 1023 + [400], [100] * 511 + [570], [10, 80] * 1000 + [400], [0, 3] * 50 + [65, 66, 67, 1],
                                     power_law(4096, 9000), power_law(300, 800)], ids=lambda v: f"{len(v)}x{max(v)}")
def test_every_block_is_in_one_item(lengths, N):
    rp = row_ptr(lengths)
    items, cut, slots = rowwise_list(rp, N)
    by_place = items[np.lexsort((items[:, 1], items[:, 0]))]
    partial = by_place[by_place[:, 3] >= 0]
    assert np.array_equal(partial[:, 3], np.arange(slots)) and len(np.unique(partial[:, 0])) == cut
    whole = by_place[by_place[:, 3] < 0]
    assert np.array_equal(whole[:, 1], rp[whole[:, 0]]) and np.array_equal(whole[:, 2], rp[whole[:, 0] + 1])
    for row in np.unique(partial[:, 0]):
        of = partial[partial[:, 0] == row]
        assert len(of) > 1 and of[0, 1] == rp[row] and of[-1, 2] == rp[row + 1] and np.array_equal(of[1:, 1], of[:-1, 2])
        n = of[:, 2] - of[:, 1]
        assert np.all(n[:-1] == n[0]) and n[0] % 2 == 0 and n[-1] <= n[0]  # no pair in two pieces
    assert len(whole) + cut == len(lengths)


def test_one_long_row_does_not_cut_ordinary_ones():
    """us, ordinary rows whole and cut: 25.2 and 30.6; 19.4 and 23.9; 56 and 64; 74 and 83."""
    for lengths, N in [([60] * 1023 + [400], 128), ([50] * 2999 + [400], 32), ([10, 80] * 1024 + [400], 256), ([200] * 127 + [1070], 1024)]:
        _, cut, _ = rowwise_list(row_ptr(lengths), N)
        assert cut == 1
        assert rowwise_list(row_ptr(lengths[:-1]), N)[1:] == (0, 0)


def test_long_rows_of_a_power_law_are_cut():
    """2,048 rows from 900 blocks down, 6.6 on average: those above twice the average, and shorter ones within 5 % of the blocks."""
    lengths = power_law(2048, 900)
    items, cut, _ = rowwise_list(row_ptr(lengths), 256)
    n, partial = items[:, 2] - items[:, 1], items[:, 3] >= 0
    piece = n[partial].max()
    assert 32 <= piece < 64 and cut == np.sum(lengths > piece)
    # average 27, pieces of 44: 200 rows of 45 blocks have partial tiles of 5.3 % of the blocks' time and stay whole, 40 are cut
    lengths = np.sort(np.r_[[20] * 900, [45] * 200, 3000])
    assert rowwise_list(row_ptr(lengths), 256)[1] == 1
    lengths = np.sort(np.r_[[20] * 1008, [45] * 40, 3000])
    assert rowwise_list(row_ptr(lengths), 256)[1] == 41


def test_launches_of_a_wavefront_a_simd_cut_all_rows():
    """us, all rows cut and the longest alone: 18 and 44; 13 and 38."""
    for lengths, N in [([100] * 511 + [570], 64), ([60] * 480 + [30] * 31 + [500], 64), ([40] * 255 + [300], 256)]:
        items, cut, _ = rowwise_list(row_ptr(lengths), N)
        most = (items[:, 2] - items[:, 1]).max()
        assert most <= 40 and cut == sum(n > most for n in lengths)


def test_long_items_come_first():
    lengths = [34, 60, 1] * 400 + [200]
    items, cut, _ = rowwise_list(row_ptr(lengths), 136)
    assert cut == 1
    n, partial = items[:, 2] - items[:, 1], items[:, 3] >= 0
    longest_piece = n[partial].max()
    first_piece, last_piece = np.nonzero(partial)[0][[0, -1]]
    assert n[:first_piece].min() > longest_piece and n[last_piece + 1:].max() <= longest_piece + 8
    assert np.all(np.diff(items[partial][:, 1]) > 0)
