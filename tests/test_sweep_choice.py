"""Which kernel a plan of mostly full blocks takes when its values are attached, on the CPU: the choice against products
that were timed through every candidate (MI355X; three products on their own inputs in turn, us)."""
import ctypes as C

import numpy as np
import pytest

from smat_amd._lib import lib

_fn = lib.smat_internal_sweep_group_rows
_fn.restype = C.c_int
_fn.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_size_t, C.c_size_t, C.c_size_t, C.c_int]

# m, k, n, share of the blocks (or bandwidth), whether the row-wise kernel repacks B, times of the row-wise kernel and of
# the sweep kernel on row groups of 64, 32, 16
MEASURED = [
    (3088, 4112, 1000, 0.15, 1, 24.25, 27.34, 19.91, 19.92),
    (3088, 4112, 2000, 0.15, 1, 39.61, 28.05, 22.38, 34.45),
    (3088, 4112, 504, 0.15, 1, 15.76, 26.98, 19.12, 17.91),
    (1600, 2000, 512, 0.2, 0, 9.92, 20.14, 13.59, 10.87),
    (4096, 4096, 512, 0.03, 0, 9.80, 18.81, 16.93, 16.16),
    (8192, 8192, 640, 0.04, 1, 22.75, 29.83, 28.51, 49.34),
    (8192, 8192, 640, 0.10, 1, 45.57, 37.60, 28.88, 50.74),
    (8192, 8192, 128, 0.10, 0, 13.59, 36.98, 27.89, 26.16),
    (8192, 8192, 256, 0.30, 1, 38.10, 78.52, 45.01, 29.39),
    (8192, 8192, 1536, 0.10, 1, 72.10, 41.90, 56.30, 78.70),
    (768, 3072, 4096, 0.10, 1, 27.70, 16.98, 14.98, 14.04),
    (2048, 1024, 2048, 0.20, 1, 13.30, 14.40, 10.30, 9.20),
    (16384, 16384, 1024, 0.04, 1, 106.0, 61.41, 100.1, 188.7),
    (4096, 64, 128, "band", 0, 3.80, 11.27, 7.66, 6.00),
    (16384, 64, 1024, "band", 1, 43.10, 19.40, 22.80, 25.00),
    (4096, 30, 1024, "band", 1, 14.90, 12.10, 9.60, 8.90),
]


def pattern(m, k, share):
    if share == "band":
        mb, bw = m // 16, k
        lo = [max(0, 16 * i - bw) // 16 for i in range(mb)]
        hi = [min(m - 1, 16 * i + 15 + bw) // 16 + 1 for i in range(mb)]
        rp = np.concatenate([[0], np.cumsum(np.array(hi) - np.array(lo))])
        return rp.astype(np.int32), np.concatenate([np.arange(a, b) for a, b in zip(lo, hi)]).astype(np.int32) * 16, m
    mask = np.random.default_rng(1).random((m // 16, k // 16)) < share
    return np.concatenate([[0], np.cumsum(mask.sum(1))]).astype(np.int32), (np.nonzero(mask)[1] * 16).astype(np.int32), k


@pytest.mark.parametrize("m,k,n,share,packed,row_wise,t64,t32,t16", MEASURED)
def test_choice_is_worth_its_building(m, k, n, share, packed, row_wise, t64, t32, t16):
    rp, ci, K = pattern(m, k, share)
    group = _fn(rp.ctypes.data, ci.ctypes.data, m, K, ci.size, n, packed)
    times = {0: row_wise, 64: t64, 32: t32, 16: t16}
    assert group in times
    if group:  # faster, and a thousand products pay for the streams (0.11 us a block)
        assert times[group] < 0.9 * row_wise
        assert 0.11 * ci.size <= 1000 * (row_wise - times[group])
    assert times[group] <= 1.15 * min(times.values())


@pytest.mark.parametrize("m,k,n,nnzb", [(1024, 512, 4096, 600), (1024, 256, 4096, 300), (64, 1024, 4096, 1), (8192, 8192, 8, 26000)])
def test_row_wise_where_the_streams_cannot_help(m, k, n, nnzb):
    rng = np.random.default_rng(2)
    cells = np.sort(rng.choice((m // 16) * (k // 16), nnzb, replace=False))
    rp = np.concatenate([[0], np.cumsum(np.bincount(cells // (k // 16), minlength=m // 16))]).astype(np.int32)
    ci = (cells % (k // 16) * 16).astype(np.int32)
    assert _fn(rp.ctypes.data, ci.ctypes.data, m, k, nnzb, n, 1) == 0
