"""Panel width of the row-wise kernel: the host rule, on the CPU."""
import ctypes as C
import itertools

import pytest

from smat_amd._lib import lib

EVEN, SPLIT, UNKNOWN = 0, 1, 2
_fn = lib.smat_internal_rowwise_panel
_fn.restype = C.c_int
_fn.argtypes = [C.c_size_t] * 4 + [C.c_int] * 2


def columns(N, K, items, avg, lengths, packed):
    return 16 * _fn(N, K, items, avg, lengths, packed)


@pytest.mark.parametrize("N", [8, 24, 32, 56, 64, 120, 128, 200, 256, 384, 504, 512, 1000, 1024, 4096])
def test_widths_that_lose_are_not_taken(N):
    for K, items, avg, packed in itertools.product([512, 8192, 16384, 1 << 20], [1, 48, 512, 1024, 4096, 65536], [1, 14, 31, 32, 87, 1000], [0, 1]):
        by_width = 256 if N >= 1024 else 128 if N >= 512 else 64
        even, split, unknown = (columns(N, K, items, avg, kind, packed) for kind in (EVEN, SPLIT, UNKNOWN))
        assert split <= 64
        # without a plan the heaviest row may be one wavefront per panel: no wider than N alone allows
        assert unknown <= by_width and unknown <= even
        if not packed:  # a panel of B in place no larger than an L2, unless N alone makes it that wide
            assert even <= by_width or K * even * 2 <= 4 << 20
        assert max(even, split, unknown) <= max(2 * N, 16)


def test_measured_choices():
    assert columns(128, 65536, 4096, 117, UNKNOWN, 0) == 64      # R-MAT scale 16: 1,406 against 2,609 us
    assert columns(512, 16384, 1024, 87, UNKNOWN, 1) == 128      # R-MAT scale 14: 806 against 975 us
    assert columns(384, 16384, 1024, 153, EVEN, 0) == 128        # the L2 holds 128 columns of B, not 256
    assert columns(128, 16384, 1024, 51, EVEN, 0) == 128         # 35.8 against 37.8 us
    assert columns(512, 8192, 512, 115, EVEN, 1) == 256          # 73 against 80 us
    assert columns(1536, 3184, 53, 18, UNKNOWN, 0) == 64         # 12.5 against 20.7 us: few wavefronts
