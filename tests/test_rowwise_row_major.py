"""Which launches of the row-wise kernel read a row-major B in place: the host rule, on the CPU."""
import ctypes as C

import pytest

from smat_amd._lib import lib

_fn = lib.smat_internal_rowwise_stays_row_major
_fn.restype = C.c_int
_fn.argtypes = [C.c_size_t] * 5 + [C.c_int]


@pytest.mark.parametrize("packed", [0, 1])
@pytest.mark.parametrize("N", [128, 136, 1000, 4096, 8192])
def test_launches_have_fewer_threads_than_the_grid_takes(N, packed):
    """64 threads for a panel of an item, less than 2^32 of them; a launch of wider panels takes what is beyond, repacked or not."""
    panels = -(-N // 64)
    items = (1 << 26) // panels  # 2^32 threads and a few less
    for n in (items, items + 1, 2 * items):
        assert not _fn(16 * n, 64, N, n, n, packed)
    n = items - (1 << 16) // panels - 1
    assert _fn(16 * n, 64, N, n, n, 0)


def test_measured_choices():
    # repacked, us in place and turned
    assert not _fn(13696, 6768, 2384, int(0.19 * 856 * 423), 856, 1)  # 391, 287
    assert not _fn(8160, 9536, 336, int(0.24 * 510 * 596), 510, 1)    # 72, 61
    # nothing is repacked: in place whatever the sizes
    assert _fn(13696, 6768, 2384, int(0.19 * 856 * 423), 856, 0)
    assert _fn(5024, 5024, 240, 314 * 3, 314, 0)
