"""Panel width of the row-wise kernel: the host rule, on the CPU."""
import ctypes as C
import itertools

import pytest

from smat_amd._lib import lib

EVEN, SPLIT, UNKNOWN = 0, 1, 2
_fn = lib.smat_internal_rowwise_panel
_fn.restype = C.c_int
_fn.argtypes = [C.c_size_t] * 3 + [C.c_int] * 2


def columns(N, items, avg, lengths, packed):
    return 16 * _fn(N, items, avg, lengths, packed)


@pytest.mark.parametrize("N", [8, 24, 32, 56, 64, 120, 128, 200, 256, 384, 504, 512, 1000, 1024, 4096])
def test_widths_that_lose_are_not_taken(N):
    for items, avg, packed in itertools.product([1, 48, 512, 1024, 4096, 65536], [1, 14, 31, 32, 87, 1000], [0, 1]):
        even, split, unknown = (columns(N, items, avg, kind, packed) for kind in (EVEN, SPLIT, UNKNOWN))
        assert split <= 64
        if not packed:
            # without a plan the heaviest row may be one wavefront per panel
            assert unknown <= even <= 128 and unknown <= (128 if N >= 512 else 64)
        assert max(even, split, unknown) <= max(2 * N, 16)


def test_measured_choices():
    # in place
    assert columns(128, 4096, 117, UNKNOWN, 0) == 64   # R-MAT scale 16: 1,458 against 2,728 us
    assert columns(384, 1024, 51, EVEN, 0) == 128      # 96.2 against 100.8 and 133.6 us
    assert columns(1536, 53, 18, UNKNOWN, 0) == 64     # 12.5 against 20.7 us: few wavefronts
    assert columns(1152, 223, 7, EVEN, 0) == 64        # 13.5 against 14.3 and 21.6 us
    assert columns(2224, 2913, 5, EVEN, 0) == 128      # 168 against 196 us
    # repacked: us with 64, 128, 256 columns
    for N, items, avg, times in [(384, 640, 59, (39.4, 35.9, 54.6)), (512, 512, 113, (60.2, 51.3, 47.9)), (888, 284, 122, (69.9, 60.5, 96.1)),
                                 (136, 651, 155, (42.6, 62.2, 99.0)), (648, 445, 59, (52.3, 50.5, 58.7)), (1984, 506, 57, (111.8, 95.4, 86.9)),
                                 (1000, 257, 59, (51.7, 54.3, 62.5)), (784, 238, 121, (63.8, 56.5, 53.2)), (568, 199, 215, (61.5, 55.0, 81.6)),
                                 (256, 1024, 51, (33.1, 30.2, 29.0))]:
        got = columns(N, items, avg, EVEN, 1)
        assert times[(64, 128, 256).index(got)] <= 1.08 * min(times), (N, items, got)
