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
    (3088, 4112, 1000, 0.15, 1, 24.54, 27.29, 19.91, 19.61),
    (3088, 4112, 2000, 0.15, 1, 40.03, 28.34, 22.08, 34.54),
    (3088, 4112, 504, 0.15, 1, 15.27, 26.95, 19.10, 17.95),
    (1600, 2000, 512, 0.2, 0, 9.88, 19.71, 13.48, 11.01),
    (4096, 4096, 512, 0.03, 0, 9.61, 18.88, 17.03, 16.34),
    (8192, 8192, 640, 0.04, 1, 23.74, 29.95, 28.66, 49.66),
    (8192, 8192, 640, 0.10, 1, 41.69, 37.57, 29.48, 50.61),
    (8192, 8192, 128, 0.10, 1, 13.62, 37.10, 28.07, 26.41),
    (8192, 8192, 256, 0.30, 1, 37.49, 78.71, 45.07, 29.89),
    (8192, 8192, 1536, 0.10, 1, 71.40, 42.11, 55.74, 77.76),
    (5008, 3008, 800, 0.20, 1, 25.22, 26.35, 17.95, 25.66),
    (10240, 14640, 384, 0.0647, 1, 35.56, 53.32, 51.30, 51.10),
    (4560, 944, 168, 0.216, 0, 5.43, 10.76, 7.85, 6.94),
    (768, 3072, 4096, 0.10, 0, 20.66, 16.88, 15.17, 14.20),
    (2048, 1024, 2048, 0.20, 1, 13.36, 15.13, 10.91, 9.30),
    (16384, 16384, 1024, 0.04, 1, 106.17, 60.19, 99.11, 183.55),
    (4096, 64, 128, "band", 0, 3.82, 11.22, 7.63, 6.00),
    (16384, 64, 1024, "band", 0, 44.59, 19.63, 23.30, 25.51),
    (4096, 30, 1024, "band", 0, 14.96, 12.81, 10.11, 9.15),
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
    worth = [t for g, t in times.items() if not g or 0.11 * ci.size <= 1000 * (row_wise - t)]
    assert times[group] <= 1.15 * min(worth)


# rows, bandwidth, n, times of the row-wise kernel on a row-major B in place and of the sweep kernel on row groups of 64, 32, 16,
# fp16 results, and whether the sweep kernel is taken
ROW_MAJOR = [
    (12672, 225, 88, 11.39, 21.43, 13.74, 9.82, True),
    (20608, 60, 96, 7.97, 13.41, 9.43, 7.57, True),
    (37520, 233, 40, 12.44, 21.25, 14.14, 11.05, True),
    (63760, 173, 48, 15.31, 19.11, 13.87, 12.83, True),
    (57296, 65, 56, 9.70, 14.18, 10.80, 9.86, False),
    (21936, 44, 88, 9.20, 18.08, 12.63, 9.95, False),
]


@pytest.mark.parametrize("m,bandwidth,n,row_wise,t64,t32,t16,sweep", ROW_MAJOR)
def test_row_major_choice_pays_for_its_building(m, bandwidth, n, row_wise, t64, t32, t16, sweep):
    fn = lib.smat_internal_sweep_group_rows_row_major
    fn.restype, fn.argtypes = C.c_int, [C.c_void_p, C.c_void_p] + [C.c_size_t] * 4
    rp, ci, K = pattern(m, bandwidth, "band")
    group = fn(rp.ctypes.data, ci.ctypes.data, m, K, ci.size, n)
    times = {0: row_wise, 64: t64, 32: t32, 16: t16}
    assert bool(group) == sweep
    assert times[group] == min(times.values())


@pytest.mark.parametrize("m,k,n,nnzb", [(1024, 512, 4096, 600), (1024, 256, 4096, 300), (64, 1024, 4096, 1), (8192, 8192, 8, 26000)])
def test_row_wise_where_the_streams_cannot_help(m, k, n, nnzb):
    rng = np.random.default_rng(2)
    cells = np.sort(rng.choice((m // 16) * (k // 16), nnzb, replace=False))
    rp = np.concatenate([[0], np.cumsum(np.bincount(cells // (k // 16), minlength=m // 16))]).astype(np.int32)
    ci = (cells % (k // 16) * 16).astype(np.int32)
    assert _fn(rp.ctypes.data, ci.ctypes.data, m, k, nnzb, n, 1) == 0


@pytest.mark.parametrize("mb, kb, share", [(193, 257, 0.15), (33, 400, 0.30), (65, 120, 0.60), (70, 300, 0.02), (129, 96, 0.9), (64, 200, 0.25)])
@pytest.mark.parametrize("rows", [64, 32, 16])
def test_what_is_estimated_is_what_is_built(mb, kb, share, rows):
    """The chunks that the choice counts are those that the streams of its row groups list, and light where the kernel's streams are."""
    rng = np.random.default_rng(mb + rows)
    mask = rng.random((mb, kb)) < share
    rp = np.concatenate([[0], np.cumsum(mask.sum(1))]).astype(np.int32)
    ci = (np.nonzero(mask)[1] * 16).astype(np.int32)
    out = (C.c_int64 * 3)()
    ptr = lambda a: C.c_void_p(a.ctypes.data)  # noqa: E731
    lib.smat_internal_sweep_groups(ptr(rp), ptr(ci), C.c_size_t(16 * mb), C.c_size_t(16 * kb), C.c_size_t(len(ci)), C.c_size_t(rows), out)
    group, listed, light = out
    chunks = np.nonzero(mask)[1] // 16
    in_groups = lambda g: len(np.unique(np.nonzero(mask)[0] // g * kb + chunks))  # noqa: E731
    n_rg = -(-mb // rows)
    even = -(-mb // n_rg)
    assert light == (len(ci) <= 8 * 8 * in_groups(even))
    assert group == (even if light else rows) and listed == in_groups(group)
