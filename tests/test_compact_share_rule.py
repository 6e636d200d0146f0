"""Wavefronts that share a task of the compact kernel: the host rule, on the CPU."""
import ctypes as C

import pytest

from smat_amd._lib import lib

_fn = lib.smat_internal_compact_share_rule
_fn.restype = C.c_int
_fn.argtypes = [C.c_int] + [C.c_int64] * 3


@pytest.mark.parametrize("total, steps, share", [(1, 5.9, 1), (1, 6, 2), (1, 11.9, 2), (1, 12, 4), (400, 6, 2), (400, 12, 4), (401, 5.9, 1), (401, 6, 2), (401, 100, 2),
                                                 (900, 6, 2), (900, 100, 2), (901, 100, 1), (1 << 26, 100, 1)])
def test_edges(total, steps, share):
    assert _fn(0, int(steps * 1000), 1000, total) == share
    assert _fn(1, int(steps * 1000), 1000, total) == 1  # a plan by name: the bits of mixed dispatch


def test_measured_choices():
    """us with one, two and four wavefronts a task, of `total` tasks and panels of `steps`."""
    for total, steps, times in [(448, 15, (10.5, 8.7, 8.6)), (552, 22, (13.4, 11.0, 11.4)), (177, 14, (5.65, 4.37, 4.07)), (874, 18, (12.7, 11.4, 12.0)),
                                (1083, 12, (12.2, 12.2, 12.5)), (268, 4, (3.88, 4.06, 4.11))]:
        assert times[(1, 2, 4).index(_fn(0, steps * 100, 100, total))] <= 1.02 * min(times), total
