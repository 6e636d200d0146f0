"""Rows of a row group of the sweep kernel where the tiles fill the device, on the CPU: 64 while the rounds of 256 workgroups
are full, fewer where the last one would be nearly empty; the timed products behind it (MI355X, us)."""
import ctypes as C

import numpy as np
import pytest

from smat_amd._lib import lib

_fn = lib.smat_internal_sweep_even_rounds
_fn.restype = C.c_int
_fn.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_size_t, C.c_size_t, C.c_int]


def rows(m, k, keep, n, row_major=0):
    mask = np.random.default_rng(1).random((m // 16, k // 16)) < keep
    rp = np.concatenate([[0], np.cumsum(mask.sum(1))]).astype(np.int32)
    ci = (np.nonzero(mask)[1] * 16).astype(np.int32)
    return _fn(rp.ctypes.data, ci.ctypes.data, m, k, n, row_major)


# m, k, share of the blocks, n, with 64 rows, with the rows that are taken
MEASURED = [(8192, 8192, 0.10, 2304, 74.7, 61.8), (8192, 8192, 0.10, 3072, 89.4, 82.3), (8192, 8192, 0.10, 4104, 123.9, 116.6),
            (8192, 4096, 0.25, 2600, 76.9, 64.7), (8192, 8192, 0.30, 2296, 169.5, 126.2), (16384, 8192, 0.08, 1536, 68.2, 64.8),
            (16384, 4096, 0.10, 1200, 42.6, 37.3), (16000, 3008, 0.15, 1304, 43.4, 39.8), (5008, 8000, 0.12, 3840, 85.4, 79.7)]


@pytest.mark.parametrize("m,k,keep,n,whole,taken", MEASURED)
def test_fewer_rows_where_a_round_would_be_nearly_empty(m, k, keep, n, whole, taken):
    g = rows(m, k, keep, n)
    assert 32 <= g < 64 and taken < whole
    panels = -(-n // 64)
    tiles = lambda r: -(-(m // 16) // r) * panels
    last = lambda r: (tiles(r) - 1) % 256 + 1
    assert last(g) > last(64) and tiles(g) <= -(-tiles(64) // 256) * 256  # no round more, the last one fuller


@pytest.mark.parametrize("m,k,keep,n", [(8192, 8192, 0.10, 4096), (8192, 8192, 0.10, 2048), (4096, 8192, 0.10, 4096), (16384, 16384, 0.05, 2056),
                                        (9600, 9600, 0.06, 3000), (12000, 6000, 0.07, 2000)])
def test_groups_of_64_where_that_gains_little(m, k, keep, n):
    assert rows(m, k, keep, n) == 64


def test_row_major_b_stays_in_place():
    # more row groups would have B turned first where the rows of B straddle cache lines
    assert rows(8192, 8192, 0.10, 4104) < 64 and rows(8192, 8192, 0.10, 4104, 1) == 64
    assert rows(8192, 8192, 0.10, 2304, 1) == rows(8192, 8192, 0.10, 2304)


def test_empty_and_tiny_matrices():
    assert rows(16, 16, 0.0, 64) == 64 and rows(16, 16, 1.0, 64) == 64
