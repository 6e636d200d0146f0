"""Which columns of B the windows in LDS copy, on the CPU: those that the part's products are stored from, and none past the last."""
import ctypes as C

import pytest

from smat_amd._lib import lib

_column = lib.smat_internal_window_copied_column
_column.restype = C.c_int64
_column.argtypes = [C.c_int, C.c_int64, C.c_int, C.c_int, C.c_int]


@pytest.mark.parametrize("tiles", [1, 2, 4])
def test_copies_name_columns_of_b(tiles):
    for N in range(8, 400, 8):
        parts = 2 if tiles < 4 and N > 16 * tiles else 1
        width = 16 * tiles * parts
        brought = set()
        for panel in range(-(-N // width)):
            for part in range(parts):
                columns = [_column(tiles, N, panel, part, c) for c in range(16 * tiles)]
                assert all(0 <= n < N for n in columns), (N, panel, part)
                brought.update(columns)
            assert _column(tiles, N, panel, parts, 0) == -1
        assert brought == set(range(N))  # each once, those past N apart: the panel's first instead
