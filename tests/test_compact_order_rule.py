"""Which lists with split rows have their tasks ordered for the L2s: the host rule, on the CPU."""
import ctypes as C

from smat_amd._lib import lib

_fn = lib.smat_internal_compact_orders
_fn.restype = C.c_int
_fn.argtypes = [C.c_size_t, C.c_size_t, C.c_int]


def test_measured_choices():
    """us in the order of the block rows and ordered (R-MAT, row-major B): scale, N."""
    for scale, N, times in [(17, 184, (96.0, 99.9)), (17, 256, (98.4, 103.3)), (17, 160, (79.3, 81.3)), (18, 256, (186.4, 190.6)), (16, 256, (52.2, 51.4)), (16, 184, (32.9, 31.0)),
                            (15, 200, (30.2, 28.2)), (19, 136, (397.1, 379.8)), (19, 200, (358.5, 337.0)), (19, 256, (315.0, 304.6)), (17, 128, (46.0, 43.9)), (17, 64, (27.7, 25.5)),
                            (15, 16, (10.0, 11.1)), (15, 32, (11.7, 12.3)), (16, 8, (13.8, 14.3)), (18, 8, (25.1, 23.7)), (17, 32, (21.4, 20.0)), (12, 256, (9.9, 9.2))]:
        assert times[_fn(1 << scale, N, 1)] == min(times), (scale, N)


def test_edges():
    for K, N, ordered in [(1 << 17, 128, True), (1 << 16, 256, True), ((1 << 16) + 16, 256, False), (1 << 17, 136, False), (1 << 18, 256, False), ((1 << 18) + 16, 256, True),
                          (1 << 15, 56, False), (1 << 15, 64, True), ((1 << 15) - 16, 64, False), (1 << 10, 72, True), (1 << 18, 8, True), ((1 << 18) - 16, 8, False)]:
        assert bool(_fn(K, N, 1)) == ordered
        assert _fn(K, N, 0)
