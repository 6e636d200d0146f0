"""Deal of a row group's block rows to the eight wavefronts of the sweep kernel: what the builder's packed counters choose is
what counters taken one by one choose (checked on the CPU)."""
import numpy as np
import pytest

from tests.test_sweep_plan import G, WAVES, random_mask_matrix, sweep_plan

S, RW, MIN_OPS = 16, 8, 4  # block columns of a chunk, block rows of a wavefront, ops of a period at least


def windows(row_ptr, col_idx, n_chunks_listed, local):
    """[row][period][length - 1]: ops of the row that may run from that period on, for so many periods"""
    win = np.zeros((G, n_chunks_listed, 3), np.int64)
    for r in range(row_ptr.size - 1):
        chunk = local[col_idx[row_ptr[r]:row_ptr[r + 1]] // 16 // S]
        q = 0
        while q < chunk.size:
            pair = q + 1 < chunk.size and chunk[q + 1] - chunk[q] <= 2
            first = max(chunk[q + pair] - 1, 0)
            last = min(chunk[q] + 1, n_chunks_listed - 1)
            win[r, first, last - first] += 1
            q += 1 + pair
    return win


def sum_of_caps(win):
    """win: [wavefront][period][length - 1]"""
    total, (due, later) = 0, np.zeros((2, WAVES), np.int64)
    for p in range(win.shape[1]):
        p0, p1, p2 = due + win[:, p, 0], later + win[:, p, 1], win[:, p, 2]
        cap = max(MIN_OPS, p0.max())
        total += cap
        room = cap - p0
        if p + 1 < win.shape[1]:
            room = np.where((room >= p1 + p2) & (p1 + p2 > 0), p1 + p2 - 1, room)
        r1 = np.minimum(room, p1)
        due, later = p1 - r1, p2 - np.minimum(room - r1, p2)
    return total


def deal(win):
    ops = win.sum((1, 2))
    wave_of, rows_of, total_of = [0] * G, [0] * WAVES, [0] * WAVES
    for r in sorted(range(G), key=lambda r: -ops[r]):
        w = min((w for w in range(WAVES) if rows_of[w] < RW), key=lambda w: total_of[w])
        wave_of[r] = w
        rows_of[w] += 1
        total_of[w] += ops[r]
    of_wave = np.zeros((WAVES,) + win.shape[1:], np.int64)
    for r in range(G):
        of_wave[wave_of[r]] += win[r]
    best = sum_of_caps(of_wave)
    for _ in range(4):
        improved = False
        for i in range(G):
            for j in range(i + 1, G):
                wi, wj = wave_of[i], wave_of[j]
                if wi == wj or (ops[i] == 0 and ops[j] == 0):
                    continue
                tried = of_wave.copy()
                tried[wi] += win[j] - win[i]
                tried[wj] += win[i] - win[j]
                now = sum_of_caps(tried)
                if now < best:
                    best, of_wave, improved = now, tried, True
                    wave_of[i], wave_of[j] = wj, wi
        if not improved:
            break
    return wave_of


@pytest.mark.parametrize("mb,kb,density,seed", [(64, 48, 0.15, 0), (64, 40, 1.0, 1), (23, 70, 0.3, 2), (64, 16, 0.4, 3), (9, 33, 0.05, 4)])
def test_deal_is_the_one_of_single_counters(mb, kb, density, seed):
    A = random_mask_matrix(mb, kb, density, seed, empty_rows=(3,), long_rows=(5,))
    plan = sweep_plan(A["b_row_ptr"], A["b_col_idx"], A["M"], A["K"])
    listed = np.unique(A["b_col_idx"] // 16 // S)
    local = np.full(kb // S + 1, -1)
    local[listed] = np.arange(listed.size)
    wave_of = deal(windows(A["b_row_ptr"], A["b_col_idx"], listed.size, local))
    want = np.full((WAVES, RW), -1)
    for w in range(WAVES):
        rows = [r for r in range(G) if wave_of[r] == w]
        want[w] = [r if r < mb else -1 for r in rows]
    np.testing.assert_array_equal(plan["row_map"].reshape(WAVES, RW), want)
