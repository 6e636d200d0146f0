"""Which first drop-in calls count the widths of windows, on the CPU: those whose sizes leave windows a chance."""
import ctypes as C

import pytest

from smat_amd._lib import lib

_may = lib.smat_internal_drop_in_may_take_window
_may.argtypes = [C.c_size_t] * 4 + [C.c_int]


@pytest.mark.parametrize("M,K,N,nnzb,most,may", [
    (262144, 262144, 64, 361000, 25, True),    # 27-point stencil 64^3
    (13296, 13296, 304, 4153, 5, True),        # band of 30
    (65536, 65536, 256, 16382, 4, True),       # band of 20
    (65536, 65536, 256, 16382, 35, False),     # a row too long
    (65536, 65536, 16, 16382, 4, False),       # narrow
    (8192, 8192, 4096, 26214, 34, False),      # the sweep kernel's from the start
    (5584, 2576, 24, 7053, 34, False),         # a product of a launch's length
])
def test_widths_are_counted_where_windows_may_be_taken(M, K, N, nnzb, most, may):
    assert bool(_may(M, K, N, nnzb, most)) == may
