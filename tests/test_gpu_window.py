"""Products from windows of B in LDS: matrices whose neighbouring block rows use the same block columns."""
import ctypes

import numpy as np
import pytest

from smat_amd import generators as gen

pytestmark = pytest.mark.gpu


def to_dev(torch, a, cuda):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int16) if a.dtype == np.uint16 else np.ascontiguousarray(a)).to(cuda)


@pytest.fixture
def force(smat):
    smat.lib.smat_internal_window_force.argtypes = [ctypes.c_int, ctypes.c_int]
    smat.lib.smat_internal_window_launches.restype = ctypes.c_int64
    yield smat.lib.smat_internal_window_force
    smat.lib.smat_internal_window_force(0, 0)
    smat.lib.smat_plan_cache_clear()


def local_matrix(mb, kb, width, seed, empty=()):
    """Block row i has up to `width` blocks around column i * kb / mb, an odd and an even number of them, `empty` rows none.
    Values are small whole numbers: every order of the sums gives the same bits."""
    rng = np.random.default_rng(seed)
    rp, ci = [0], []
    for i in range(mb):
        if i not in empty:
            lo = max(0, min(i * kb // mb - width // 2, kb - width))
            n = rng.integers(1, width + 1)
            ci += sorted((lo + rng.choice(min(width, kb), n, replace=False)).tolist())
        rp.append(len(ci))
    vals = rng.integers(-3, 4, len(ci) * 256).astype(np.float16).view(np.uint16)
    return np.array(rp, np.int32), np.array(ci, np.int32) * 16, vals


def whole_b(K, N, seed):
    return np.random.default_rng(seed).integers(-4, 5, K * N).astype(np.float16).view(np.uint16)


# block rows around whole groups of 4, 8 and 16; rows of one block to the most that a wavefront holds (24 blocks on 4 tiles, 34 on 1
# and 2); N below, at and past a panel and half a panel
@pytest.mark.parametrize("mb,kb,width", [(1, 3, 2), (15, 20, 5), (33, 33, 12), (70, 64, 24), (130, 200, 34)])
@pytest.mark.parametrize("N", [8, 24, 32, 72, 136, 320])
@pytest.mark.parametrize("rows,tiles", [(4, 1), (4, 2), (8, 2), (8, 4), (16, 1), (16, 2), (16, 4)])
def test_windows_match_the_oracle(smat, cuda, oracle, force, mb, kb, width, N, rows, tiles):
    import torch
    if tiles == 4 and width > 24:
        pytest.skip("rows of more than 24 blocks")
    if width > 24 and rows == 4 and tiles == 2 or width > 20 and rows == 8 and tiles == 4:
        pytest.skip("windows wider than fit")
    rp, ci, vals = local_matrix(mb, kb, width, seed=mb + rows, empty=(0, 2) if mb > 8 else ())
    M, K, nnzb = mb * 16, kb * 16, len(ci)
    B = whole_b(K, N, seed=N)
    d = [to_dev(torch, x, cuda) for x in (vals, rp, ci, B)]
    want = oracle.spmm_bcsr(M, N, K, rp, ci, vals, B, threads=4)
    force(rows, tiles)
    for c_f32 in (False, True):
        plan = smat.Plan(rp, M, K, nnzb, N, col_idx_host=ci)
        plan.attach_values(d[0], d[1], d[2])
        assert smat.lib.smat_internal_plan_window_rows(plan.handle) == rows
        C = torch.full((M, N), float("nan"), dtype=torch.float32 if c_f32 else torch.float16, device=cuda)
        smat.spmm(d[0], d[1], d[2], d[3], C, M, N, K, nnzb, plan=plan, c_f32=c_f32)
        assert np.array_equal(C.cpu().numpy().astype(np.float32), want.astype(np.float16 if not c_f32 else np.float32).astype(np.float32))
        plan.close()


def test_many_panels_and_units(smat, cuda, oracle, force):
    """More units than workgroups, panels split among several: every group of a 40,000-row band at a width of several panels."""
    import torch
    rp, ci, vals = local_matrix(2500, 2500, 9, seed=5)
    M = K = 40000
    N = 200
    B = whole_b(K, N, seed=1)
    d = [to_dev(torch, x, cuda) for x in (vals, rp, ci, B)]
    want = oracle.spmm_bcsr(M, N, K, rp, ci, vals, B, threads=8).astype(np.float16)
    for rows, tiles in ((4, 1), (8, 2), (16, 4)):
        force(rows, tiles)
        plan = smat.Plan(rp, M, K, len(ci), N, col_idx_host=ci)
        plan.attach_values(d[0], d[1], d[2])
        C = torch.full((M, N), float("nan"), dtype=torch.float16, device=cuda)
        smat.spmm(d[0], d[1], d[2], d[3], C, M, N, K, len(ci), plan=plan)
        assert np.array_equal(C.cpu().numpy(), want)
        plan.close()


def test_infinities_stay_with_the_blocks_that_meet_them(smat, cuda, oracle, force):
    """An odd number of blocks in a row: the second half of its last pair multiplies zeros by zeros, also where the row before had infinities there."""
    import torch
    mb, kb, N = 48, 48, 64
    rp, ci = np.arange(mb + 1, dtype=np.int32) * 3, np.empty(mb * 3, np.int32)
    for i in range(mb):
        ci[3 * i:3 * i + 3] = np.array([max(0, min(i - 1, kb - 3)) + j for j in range(3)]) * 16
    vals = np.ones(mb * 3 * 256, np.float16)
    vals[3 * 20 * 256:(3 * 20 + 3) * 256] = np.inf
    vals = vals.view(np.uint16)
    M, K = mb * 16, kb * 16
    B = np.ones((N, K), np.float16)
    B[:, 30 * 16] = np.inf
    B = B.reshape(-1).view(np.uint16)
    d = [to_dev(torch, x, cuda) for x in (vals, rp, ci, B)]
    want = oracle.spmm_bcsr(M, N, K, rp, ci, vals, B, threads=4).astype(np.float16)
    for rows in (4, 8, 16):
        force(rows, 2)
        plan = smat.Plan(rp, M, K, len(ci), N, col_idx_host=ci)
        plan.attach_values(d[0], d[1], d[2])
        C = torch.zeros((M, N), dtype=torch.float16, device=cuda)
        smat.spmm(d[0], d[1], d[2], d[3], C, M, N, K, len(ci), plan=plan)
        assert np.array_equal(C.cpu().numpy(), want, equal_nan=True)
        plan.close()


def test_a_pattern_rewritten_in_place_is_multiplied_as_it_is(smat, cuda, oracle, force):
    """The drop-in call keeps the windows of the pattern it saw first; blocks that moved since are multiplied where they are now."""
    import torch
    force(8, 2)
    rp, ci, vals = local_matrix(100, 100, 7, seed=2)
    M = K = 1600
    N = 96
    B = whole_b(K, N, seed=3)
    d = [to_dev(torch, x, cuda) for x in (vals, rp, ci, B)]
    smat.lib.smat_plan_cache_clear()
    C = torch.empty((M, N), dtype=torch.float16, device=cuda)
    for seed in (None, 11, 12):
        if seed is not None:
            rng = np.random.default_rng(seed)
            for i in range(0, 100, 3):
                ci[rp[i]:rp[i + 1]] = np.sort(rng.choice(100, rp[i + 1] - rp[i], replace=False)).astype(np.int32) * 16
            d[2].copy_(torch.from_numpy(ci))
        smat.spmm(d[0], d[1], d[2], d[3], C, M, N, K, len(ci), drop_in=True)
        want = oracle.spmm_bcsr(M, N, K, rp, ci, vals, B, threads=4).astype(np.float16)
        assert np.array_equal(C.cpu().numpy(), want)


@pytest.mark.parametrize("listed", [False, True])
def test_columns_other_than_the_plan_s_are_multiplied_as_they_are(smat, cuda, oracle, force, listed):
    """The columns on the device are not those that the widths of the windows were counted in: blocks without a place in a window are multiplied from
    memory, lists of nonzeros are left to the compact kernel."""
    import torch
    force(8, 2)
    rp, ci, vals = local_matrix(96, 100, 7, seed=2)
    M, K, N, nnzb = 1536, 1600, 64, len(ci)
    if listed:
        vals = sparse_values(nnzb, 2, 1)
    rng = np.random.default_rng(3)
    moved = np.concatenate([np.sort(rng.choice(100, n, replace=False)) for n in np.diff(rp)]).astype(np.int32) * 16
    B = whole_b(K, N, seed=3)
    d = [to_dev(torch, x, cuda) for x in (vals, rp, moved, B)]
    plan = smat.Plan(rp, M, K, nnzb, N, col_idx_host=ci)
    plan.attach_values(*d[:3])
    assert smat.lib.smat_internal_plan_window_rows(plan.handle) == (0 if listed else 8)
    C = torch.full((M, N), float("nan"), dtype=torch.float16, device=cuda)
    smat.spmm(d[0], d[1], d[2], d[3], C, M, N, K, nnzb, plan=plan)
    assert np.array_equal(C.cpu().numpy(), oracle.spmm_bcsr(M, N, K, rp, moved, vals, B, threads=4).astype(np.float16))
    plan.close()


# words of the bitmap of a window: one, as many as threads, more; block rows that do and do not fill the groups, and more groups than workgroups
@pytest.mark.parametrize("mb,kb,width", [(1, 3, 2), (37, 31, 9), (1500, 8192, 12), (7133, 20011, 12)])
def test_widths_and_lists_of_windows(smat, cuda, oracle, force, mb, kb, width):
    """The widths as the device and the host count them, and products from lists that the device makes of wide bitmaps."""
    import torch
    rp, ci, vals = local_matrix(mb, kb, width, seed=mb, empty=range(20, 90) if mb > 90 else ())
    M, K, N, nnzb = mb * 16, kb * 16, 24, len(ci)
    d = [to_dev(torch, x, cuda) for x in (vals, rp, ci)]
    got = (ctypes.c_int64 * 12)()
    ptr = lambda a: ctypes.c_void_p(a.data_ptr() if torch.is_tensor(a) else a.ctypes.data)
    assert smat.lib.smat_internal_window_widths(ptr(d[1]), ptr(d[2]), ptr(rp), ptr(ci), ctypes.c_size_t(mb), ctypes.c_size_t(kb), ctypes.c_size_t(nnzb), got) == 0
    for i, rows in enumerate((4, 8, 16)):
        widths = [len(np.unique(ci[rp[g]:rp[min(g + rows, mb)]])) for g in range(0, mb, rows)]
        assert list(got)[4 * i:4 * i + 4] == [max(widths), sum(widths)] * 2
    B = whole_b(K, N, seed=N)
    d.append(to_dev(torch, B, cuda))
    want = oracle.spmm_bcsr(M, N, K, rp, ci, vals, B, threads=8).astype(np.float16)
    force(8, 1)
    plan = smat.Plan(rp, M, K, nnzb, N, col_idx_host=ci)
    plan.attach_values(*d[:3])
    smat.lib.smat_plan_cache_clear()
    for p in (plan, None):
        C = torch.full((M, N), float("nan"), dtype=torch.float16, device=cuda)
        before = smat.lib.smat_internal_window_launches()
        smat.spmm(*d, C, M, N, K, nnzb, plan=p, drop_in=p is None)
        assert smat.lib.smat_internal_window_launches() == before + 1
        assert np.array_equal(C.cpu().numpy(), want)
    plan.close()


def test_which_products_take_windows(smat, cuda):
    """Local patterns do, as the drop-in call and with values; random ones, rows too long and products of a launch's length do not."""
    import torch

    def rows(A, N, row_major=False):
        ci, rp = A["b_col_idx"].astype(np.int32), A["b_row_ptr"].astype(np.int32)
        d = [to_dev(torch, x, cuda) for x in (A["b_val"], rp, ci)]
        plan = smat.Plan(rp, A["M"], A["K"], len(ci), N, col_idx_host=ci, b_row_major=row_major)
        plan.attach_values(*d)
        r = smat.lib.smat_internal_plan_window_rows(plan.handle)
        plan.close()
        return r

    def blocked(d):
        A = smat.csr_to_bcsr(d["M"], d["K"], d["row_ptr"], d["col_idx"], d["val"])
        return {"M": A.M, "K": A.K, "b_row_ptr": A.row_ptr, "b_col_idx": A.col_idx, "b_val": A.val}

    assert rows(blocked(gen.stencil27(32)), 512) > 0
    assert rows(blocked(gen.band(8960, 120)), 48) > 0
    assert rows(blocked(gen.band(512, 16)), 32) == 0
    assert rows(blocked(gen.band(8192, 400)), 256) == 0
    assert rows(gen.random_bcsr(128, 128, 0.2, seed=1), 512) == 0


@pytest.mark.parametrize("m,bandwidth,n_hint,taken,left", [(4144, 51, 656, (656, 488), (128, 64)), (2192, 51, 584, (584,), (288, 112)),
                                                           (20064, 150, 32, (32,), (8,)), (7056, 37, 320, (320,), (64,))])
def test_launches_of_another_width_that_another_kernel_is_as_fast_for(smat, cuda, m, bandwidth, n_hint, taken, left):
    """A launch's length: not from windows, which take 5 us at least, whatever the plan's own width takes."""
    import torch
    d = gen.band(m, bandwidth)
    A = smat.csr_to_bcsr(d["M"], d["K"], d["row_ptr"], d["col_idx"], d["val"])
    smat.lib.smat_internal_window_launches.restype = ctypes.c_int64
    t = [to_dev(torch, x, cuda) for x in (A.val, A.row_ptr, A.col_idx, whole_b(A.K, n_hint, seed=1))]
    plan = smat.Plan(A.row_ptr, A.M, A.K, A.nnzb, n_hint, col_idx_host=A.col_idx)
    plan.attach_values(*t[:3])
    assert smat.lib.smat_internal_plan_window_rows(plan.handle) > 0
    C = torch.empty((A.M, n_hint), dtype=torch.float32, device=cuda)
    for n in (*taken, *left):
        for c_f32 in (False, True):
            before = smat.lib.smat_internal_window_launches()
            smat.spmm(*t, C, A.M, n, A.K, A.nnzb, plan=plan, c_f32=c_f32)
            assert (smat.lib.smat_internal_window_launches() > before) == (n in taken), (n, c_f32)
    torch.cuda.synchronize()
    plan.close()


def blocked_band(smat, m, bandwidth):
    d = gen.band(m, bandwidth)
    A = smat.csr_to_bcsr(d["M"], d["K"], d["row_ptr"], d["col_idx"], d["val"])
    return A.M, A.K, A.row_ptr, A.col_idx, A.val


def blocked_random(mb, kb, density):
    A = gen.random_bcsr(mb, kb, density, seed=1)
    return A["M"], A["K"], A["b_row_ptr"].astype(np.int32), A["b_col_idx"].astype(np.int32), A["b_val"]


@pytest.mark.parametrize("matrix,n_hint,own,others", [
    # 12.5, 15.3 and 11.4 us from windows, 8.2, 10.8 and 8.1 from memory; little is shared
    ((104, 129, 0.04), 1560, False, {}), ((84, 193, 0.0399), 1848, False, {}), ((148, 55, 0.0398), 2024, False, {}),
    # 5.6 and 5.0, one round of wavefronts of the row-wise kernel 4.5 and 4.1
    ((1248, 75), 832, False, {}), ((688, 77), 968, False, {}),
    # 4.5 and 5.8, before 5.7 and 9.0
    ((2112, 82), 216, True, {}), ((2464, 15), 912, True, {}),
    # of other widths 4.1 and 4.0, before 5.4 and 5.4; columns of B that are whole cache lines apart
    ((1536, 73), 304, True, {224: True, 120: True}), ((1472, 68), 280, True, {208: True}),
])
def test_short_products_take_windows_where_they_are_faster(smat, cuda, oracle, matrix, n_hint, own, others):
    import torch
    M, K, rp, ci, _ = blocked_band(smat, *matrix) if len(matrix) == 2 else blocked_random(*matrix)
    vals = np.random.default_rng(1).integers(-3, 4, len(ci) * 256).astype(np.float16).view(np.uint16)
    B = whole_b(K, n_hint, seed=2)
    t = [to_dev(torch, x, cuda) for x in (vals, rp, ci, B)]
    want = oracle.spmm_bcsr(M, n_hint, K, rp, ci, vals, B, threads=8).astype(np.float16)
    plan = smat.Plan(rp, M, K, len(ci), n_hint, col_idx_host=ci)
    plan.attach_values(*t[:3])
    assert (smat.lib.smat_internal_plan_window_rows(plan.handle) > 0) == own
    smat.lib.smat_internal_window_launches.restype = ctypes.c_int64
    for n, taken in {n_hint: own, **others}.items():
        C = torch.full((M, n), float("nan"), dtype=torch.float16, device=cuda)
        before = smat.lib.smat_internal_window_launches()
        smat.spmm(*t, C, M, n, K, len(ci), plan=plan)
        assert (smat.lib.smat_internal_window_launches() > before) == taken, n
        assert np.array_equal(C.cpu().numpy(), want[:, :n])
    plan.close()


def sparse_values(nnzb, seed, most):
    """Blocks of up to `most` nonzeros, some of none, small whole numbers."""
    rng = np.random.default_rng(seed)
    vals = np.zeros((nnzb, 256), np.float16)
    for b in vals:
        at = rng.choice(256, rng.integers(0, most + 1), replace=False)
        b[at] = rng.choice([-3, -2, -1, 1, 2, 3], len(at))
    return vals.reshape(-1).view(np.uint16)


# lists of a pair around 0, a lane's four and what a wavefront holds (256); the last block of odd rows alone
@pytest.mark.parametrize("mb,kb,width", [(1, 3, 2), (33, 33, 12), (130, 200, 34)])
@pytest.mark.parametrize("most", [1, 40, 127])
@pytest.mark.parametrize("rows,tiles,N", [(4, 1, 8), (8, 2, 24), (16, 1, 72), (16, 2, 136), (16, 4, 320)])
def test_windows_of_listed_nonzeros_match_the_oracle(smat, cuda, oracle, force, mb, kb, width, most, rows, tiles, N):
    import torch
    if tiles == 4 and width > 24:
        pytest.skip("rows of more than 24 blocks")
    rp, ci, _ = local_matrix(mb, kb, width, seed=mb + rows, empty=(0, 2) if mb > 8 else ())
    M, K, nnzb = mb * 16, kb * 16, len(ci)
    vals, B = sparse_values(nnzb, most, most), whole_b(K, N, seed=N)
    d = [to_dev(torch, x, cuda) for x in (vals, rp, ci, B)]
    want = oracle.spmm_bcsr(M, N, K, rp, ci, vals, B, threads=4)
    force(rows, tiles)
    plan = smat.Plan(rp, M, K, nnzb, N, col_idx_host=ci)
    plan.attach_values(d[0], d[1], d[2])
    assert smat.lib.smat_internal_plan_window_rows(plan.handle) == rows
    listed = plan.info()["kernel"] == smat.KERNEL_COMPACT
    assert listed or most > 1  # a tenth of a block's columns or most of them
    if listed:
        d[0].zero_()  # the values are the ones attached
    for n in {N, max(8, N * 3 // 4 // 8 * 8)}:
        for c_f32 in (False, True):
            for kernel in (smat.KERNEL_AUTO, smat.KERNEL_COMPACT) if listed else (smat.KERNEL_AUTO,):
                C = torch.full((M, n), float("nan"), dtype=torch.float32 if c_f32 else torch.float16, device=cuda)
                smat.spmm(d[0], d[1], d[2], d[3][:K * n], C, M, n, K, nnzb, plan=plan, c_f32=c_f32, kernel=kernel)
                assert np.array_equal(C.cpu().numpy().astype(np.float32), want[:, :n].astype(np.float16 if not c_f32 else np.float32).astype(np.float32))
    plan.close()


@pytest.mark.parametrize("N,parts", [(64, 1), (72, 2), (192, 2), (200, 4), (264, 2)])
def test_launches_of_the_compact_kernel_beside_windows_run_in_parts(smat, cuda, N, parts):
    """Halves where there are two panels and more, quarters of four; one panel in one run an XCD."""
    import torch
    d = gen.stencil27(40)
    A = smat.csr_to_bcsr(d["M"], d["K"], d["row_ptr"], d["col_idx"], d["val"])
    t = [to_dev(torch, x, cuda) for x in (A.val, A.row_ptr, A.col_idx, whole_b(A.K, N, seed=1))]
    plan = smat.Plan(A.row_ptr, A.M, A.K, A.nnzb, N, col_idx_host=A.col_idx)
    plan.attach_values(*t[:3])
    assert smat.lib.smat_internal_plan_window_rows(plan.handle) > 0 and plan.info()["kernel"] == smat.KERNEL_COMPACT
    smat.lib.smat_internal_compact_run.argtypes = [ctypes.c_int]
    C = torch.empty((A.M, N), dtype=torch.float16, device=cuda)
    runs = {}
    try:
        for force_run in (0, 1 << 24):
            smat.lib.smat_internal_compact_run(force_run)
            for row_major in (False, True):
                smat.spmm(*t, C, A.M, N, A.K, A.nnzb, plan=plan, b_row_major=row_major, kernel=smat.KERNEL_COMPACT)
                runs[force_run, row_major] = smat.lib.smat_internal_compact_last_run()
    finally:
        smat.lib.smat_internal_compact_run(0)
    torch.cuda.synchronize()
    for row_major in (False, True):
        eighth = runs[1 << 24, row_major]
        assert eighth >= 8 and runs[0, row_major] == eighth // parts
    plan.close()


def test_values_attached_again_replace_the_listed_ones(smat, cuda, oracle, force):
    """Between lists, from a list to full blocks and back, and to columns too full for a list; a launch wider than the plan is refused as before."""
    import torch
    rp, ci, full = local_matrix(60, 60, 9, seed=4)
    M = K = 960
    N = 64
    B = whole_b(K, N + 8, seed=6)
    force(8, 2)
    d = [to_dev(torch, x, cuda) for x in (full, rp, ci, B)]
    plan = smat.Plan(rp, M, K, len(ci), N, col_idx_host=ci)
    C = torch.empty((M, N), dtype=torch.float16, device=cuda)
    columns = np.where(np.arange(256) % 16 < 9, np.float16(2), np.float16(0))  # 288 nonzeros in a pair
    for vals in (sparse_values(len(ci), 6, 1), full, sparse_values(len(ci), 9, 2), np.tile(columns, len(ci)).view(np.uint16), sparse_values(len(ci), 3, 3)):
        d[0].copy_(to_dev(torch, vals, cuda))
        plan.attach_values(d[0], d[1], d[2])
        smat.spmm(d[0], d[1], d[2], d[3][:K * N], C, M, N, K, len(ci), plan=plan)
        assert np.array_equal(C.cpu().numpy(), oracle.spmm_bcsr(M, N, K, rp, ci, vals, B[:K * N], threads=4).astype(np.float16))
    with pytest.raises(smat.SmatError):
        smat.spmm(d[0], d[1], d[2], d[3], torch.empty((M, N + 8), dtype=torch.float16, device=cuda), M, N + 8, K, len(ci), plan=plan)
    plan.close()


def test_plans_for_the_sweep_kernel_may_multiply_from_windows(smat, cuda, oracle, force):
    """A narrow band: the plan says the sweep kernel and takes launches for it, launches that leave the choice take windows, attached twice or not."""
    import torch
    d = gen.band(13296, 30)
    A = smat.csr_to_bcsr(d["M"], d["K"], d["row_ptr"], d["col_idx"], d["val"])
    N, nnzb = 304, len(A.col_idx)
    vals = np.random.default_rng(1).integers(-3, 4, nnzb * 256).astype(np.float16).view(np.uint16)
    B = whole_b(A.K, N, seed=2)
    t = [to_dev(torch, x, cuda) for x in (vals, A.row_ptr, A.col_idx, B)]
    want = oracle.spmm_bcsr(A.M, N, A.K, A.row_ptr, A.col_idx, vals, B, threads=8).astype(np.float16)
    plan = smat.Plan(A.row_ptr, A.M, A.K, nnzb, N, col_idx_host=A.col_idx)
    for _ in range(2):
        plan.attach_values(*t[:3])
        assert plan.info()["kernel"] == smat.KERNEL_SWEEP and smat.lib.smat_internal_plan_window_rows(plan.handle) > 0
        for n in (N, 128):
            for kernel in (smat.KERNEL_AUTO, smat.KERNEL_SWEEP):
                C = torch.full((A.M, n), float("nan"), dtype=torch.float16, device=cuda)
                smat.spmm(t[0], t[1], t[2], t[3][:A.K * n], C, A.M, n, A.K, nnzb, plan=plan, kernel=kernel)
                assert np.array_equal(C.cpu().numpy(), want[:, :n])
    plan.close()


@pytest.mark.parametrize("rows,tiles,N", [(4, 1, 24), (8, 2, 136), (16, 2, 72), (16, 4, 64)])
@pytest.mark.parametrize("listed", [False, True])
def test_groups_without_blocks(smat, cuda, oracle, force, rows, tiles, N, listed):
    """The first groups, some in the middle and the last one have no blocks: their rows of C are zeros."""
    import torch
    rp, ci, vals = local_matrix(200, 90, 7, seed=rows, empty=(*range(32), *range(64, 97), *range(160, 200)))
    if listed:
        vals = sparse_values(len(ci), 2, 1)
    M, K, nnzb = 3200, 1440, len(ci)
    B = whole_b(K, N, seed=N)
    d = [to_dev(torch, x, cuda) for x in (vals, rp, ci, B)]
    want = oracle.spmm_bcsr(M, N, K, rp, ci, vals, B, threads=4).astype(np.float16)
    force(rows, tiles)
    plan = smat.Plan(rp, M, K, nnzb, N, col_idx_host=ci)
    plan.attach_values(*d[:3])
    assert smat.lib.smat_internal_plan_window_rows(plan.handle) == rows and (plan.info()["kernel"] == smat.KERNEL_COMPACT) == listed
    C = torch.full((M, N), float("nan"), dtype=torch.float16, device=cuda)
    smat.spmm(d[0], d[1], d[2], d[3], C, M, N, K, nnzb, plan=plan)
    assert np.array_equal(C.cpu().numpy(), want)
    plan.close()


@pytest.mark.parametrize("kind", ["blocks", "nonzeros", "columns"])
def test_block_columns_in_any_order_and_twice(smat, cuda, oracle, force, kind):
    """A block row whose columns do not ascend, some of them listed twice: windows of whole blocks, of listed nonzeros, and columns of B in LDS."""
    import torch
    rp, ci, vals = local_matrix(45, 50, 10, seed=31)
    rng = np.random.default_rng(5)
    for i in range(45):
        row = ci[rp[i]:rp[i + 1]]
        rng.shuffle(row)
        if len(row) > 2:
            row[1] = row[0]
    M, K, N, nnzb = 720, 800, 72, len(ci)
    if kind != "blocks":
        vals = sparse_values(nnzb, 3, 4)
    B = whole_b(K, N, seed=3)
    d = [to_dev(torch, x, cuda) for x in (vals, rp, ci, B)]
    want = oracle.spmm_bcsr(M, N, K, rp, ci, vals, B, threads=4).astype(np.float16)
    smat.lib.smat_internal_resident_force.argtypes = [ctypes.c_int, ctypes.c_int]
    try:
        force(*((-1, 0) if kind == "columns" else (8, 2)))
        smat.lib.smat_internal_resident_force(4 if kind == "columns" else -1, 0)
        plan = smat.Plan(rp, M, K, nnzb, N, col_idx_host=ci)
        plan.attach_values(*d[:3])
        assert (smat.lib.smat_internal_plan_window_rows(plan.handle), smat.lib.smat_internal_plan_resident(plan.handle)) == ((0, 1) if kind == "columns" else (8, 0))
        C = torch.full((M, N), float("nan"), dtype=torch.float16, device=cuda)
        smat.spmm(d[0], d[1], d[2], d[3], C, M, N, K, nnzb, plan=plan)
        assert np.array_equal(C.cpu().numpy(), want)
        plan.close()
        if kind == "blocks":
            smat.lib.smat_plan_cache_clear()
            C.fill_(float("nan"))
            smat.spmm(d[0], d[1], d[2], d[3], C, M, N, K, nnzb, drop_in=True)
            assert np.array_equal(C.cpu().numpy(), want)
    finally:
        smat.lib.smat_internal_resident_force(0, 0)


def octets_fit(row, steps):
    """Whether a block row, nonzeros of its octets in order, fits a wavefront's lists: rounds of 16 octets and 252 nonzeros, ended where the next pair of
    blocks does not fit, and `steps` of four octets in all."""
    places = n = 0
    for pair in range(0, len(row), 4):
        used = [k for k in row[pair:pair + 4] if k]
        here = used[:16 - places % 16]
        if n and n + sum(here) > 252:
            places, n, here = -(-places // 16) * 16, 0, used
        end = n + sum(here)
        if end > 252:
            return False
        full = (places % 16 + len(used)) // 16
        places, n = places + len(used), sum(used) - sum(here) if full else end
    return -(-places // 4) <= steps


# (nonzeros per octet of 8 columns, those of even and of odd ones): 16 octets a round and 252 nonzeros in its list are the edges
@pytest.mark.parametrize("width", [1, 3, 7, 12, 15, 16, 17, 24])
@pytest.mark.parametrize("octets", [(5, 0), (0, 3), (15, 0), (16, 0), (21, 0), (60, 0), (23, 20), (1, 1)])
def test_octets_without_a_nonzero_are_left_out(smat, cuda, oracle, force, width, octets):
    """Rounds that are full to the last place, end early and hold one octet; B is infinite where no octet holds a nonzero, places of none included."""
    import torch
    rng = np.random.default_rng(width)
    mb, kb, N = 40, 40, 40
    rp, ci, _ = local_matrix(mb, kb, width, seed=width, empty=(5,))
    M, K, nnzb = mb * 16, kb * 16, len(ci)
    vals = np.zeros((nnzb, 16, 2, 8), np.float16)  # row, octet, column
    for b in vals:
        for h, n in enumerate(octets):
            for at in rng.choice(64, n, replace=False):
                b[at // 4, h, at % 4 * 2 + h] = rng.choice([-2, -1, 1, 2])
    vals = vals.reshape(-1).view(np.uint16)
    B = whole_b(K, N, seed=3).view(np.float16).reshape(N, kb, 2, 8).copy()
    for h, n in enumerate(octets):
        if n == 0:
            B[:, :, h] = 0
    want = oracle.spmm_bcsr(M, N, K, rp, ci, vals, B.reshape(-1).view(np.uint16), threads=4).astype(np.float16)
    for h, n in enumerate(octets):
        if n == 0:
            B[:, :, h] = np.inf
    d = [to_dev(torch, x, cuda) for x in (vals, rp, ci, B.reshape(-1).view(np.uint16))]
    kinds = vals.view(np.float16).reshape(nnzb, 16, 16) != 0
    listed = kinds.any(1).sum() < 0.6 * 16 * nnzb  # else the blocks are multiplied whole
    held = 12 if width <= 24 else 17
    fits = all(octets_fit(kinds[rp[i]:rp[i + 1]].reshape(-1, 16, 2, 8).sum((1, 3)).reshape(-1).tolist(), held) for i in range(mb))
    for rows, tiles in ((4, 1), (8, 2), (16, 4)):
        force(rows, tiles)
        plan = smat.Plan(rp, M, K, nnzb, N, col_idx_host=ci)
        plan.attach_values(d[0], d[1], d[2])
        assert (plan.info()["kernel"] == smat.KERNEL_COMPACT) == listed
        assert smat.lib.smat_internal_plan_window_rows(plan.handle) == (rows if fits or not listed else 0)
        C = torch.full((M, N), float("nan"), dtype=torch.float16, device=cuda)
        smat.spmm(d[0], d[1], d[2], d[3], C, M, N, K, nnzb, plan=plan)
        assert np.array_equal(C.cpu().numpy(), want)
        plan.close()


@pytest.mark.parametrize("rows,tiles", [(4, 1), (8, 2), (16, 4)])
@pytest.mark.parametrize("most", [1, 40, 62])  # rounds of 16 octets; ended early by the entries of 6 and of 4
def test_infinities_under_the_first_octet_of_a_row(smat, cuda, oracle, force, rows, tiles, most):
    """Octets, one a block, that do not fill a step or a round: the places left over do not multiply the row's first octet again.  A row whose own
    nonzeros alone meet an infinity has that infinity, as block by block."""
    import torch
    rng = np.random.default_rng(most)
    mb, kb, N = 41, 60, 24
    rp = np.concatenate([[0], np.cumsum(np.arange(mb) % (18 if most == 1 else 8) + 1)]).astype(np.int32)
    ci = np.concatenate([min(i, kb - rp[i + 1] + rp[i]) + np.arange(rp[i + 1] - rp[i]) for i in range(mb)]).astype(np.int32) * 16
    M, K, nnzb = mb * 16, kb * 16, len(ci)
    vals = np.zeros((nnzb, 16, 16), np.float16)
    vals[:, 3, 0] = 2  # every block meets the infinities of its first column in this row
    for b in vals:
        at = rng.choice(np.delete(np.arange(1, 128), 3 * 8 - 1), most - 1, replace=False)
        b[at // 8, at % 8] = 1
    vals = vals.reshape(-1).view(np.uint16)
    B = whole_b(K, N, seed=3).view(np.float16).reshape(N, K).copy()
    first = ci[rp[:-1]]
    B[:, first[rng.permutation(mb)[:5]]] = np.inf
    B = B.reshape(-1).view(np.uint16)
    d = [to_dev(torch, x, cuda) for x in (vals, rp, ci, B)]
    want = oracle.spmm_bcsr(M, N, K, rp, ci, vals, B, threads=4).astype(np.float16)
    assert np.isinf(want).any() and np.isfinite(want).any()
    force(rows, tiles)
    plan = smat.Plan(rp, M, K, nnzb, N, col_idx_host=ci)
    plan.attach_values(d[0], d[1], d[2])
    assert plan.info()["kernel"] == smat.KERNEL_COMPACT and smat.lib.smat_internal_plan_window_rows(plan.handle) == rows
    C = torch.zeros((M, N), dtype=torch.float16, device=cuda)
    smat.spmm(d[0], d[1], d[2], d[3], C, M, N, K, nnzb, plan=plan)
    assert np.array_equal(C.cpu().numpy(), want, equal_nan=True)
    plan.close()


def test_row_major_b_is_turned_only_for_windows_that_are_taken(smat, cuda, oracle, force):
    """A launch that names the row-wise kernel takes no windows, and one without windows reads B in place: no pass over B before either."""
    import torch
    counts = smat.lib.smat_internal_window_launches, smat.lib.smat_internal_turned_launches
    counts[1].restype = ctypes.c_int64
    rng = np.random.default_rng(9)
    groups = [rng.choice(1000, 10, replace=False) for _ in range(250)]  # the block columns of 16 block rows, all over B: not for the sweep kernel
    ci = np.concatenate([np.sort(rng.permutation(groups[i // 16])[:8]) for i in range(4000)]).astype(np.int32) * 16
    rp = np.arange(0, len(ci) + 1, 8, dtype=np.int32)
    vals = rng.integers(-3, 4, len(ci) * 256).astype(np.float16).view(np.uint16)
    M, K, n_hint, nnzb = 64000, 16000, 256, len(ci)
    d = [to_dev(torch, x, cuda) for x in (vals, rp, ci)]
    force(16, 0)
    plan = smat.Plan(rp, M, K, nnzb, n_hint, col_idx_host=ci, b_row_major=True)
    plan.attach_values(*d)
    assert smat.lib.smat_internal_plan_window_rows(plan.handle) == 16
    force(0, 0)
    taken = set()
    for kernel in (smat.KERNEL_AUTO, smat.KERNEL_ROWWISE_DIRECT):
        for N in (256, 200, 136, 64, 24, 8):
            B = whole_b(K, N, seed=N)
            want = oracle.spmm_bcsr(M, N, K, rp, ci, vals, B, threads=8).astype(np.float16)
            rows = to_dev(torch, np.ascontiguousarray(B.reshape(N, K).T), cuda)
            C = torch.full((M, N), float("nan"), dtype=torch.float16, device=cuda)
            before = [count() for count in counts]
            smat.spmm(*d, rows, C, M, N, K, nnzb, plan=plan, kernel=kernel, b_row_major=True)
            windows, turned = (count() - b for count, b in zip(counts, before))
            assert np.array_equal(C.cpu().numpy(), want), N
            assert turned == windows, N
            taken.add((kernel, windows))
    assert taken == {(smat.KERNEL_AUTO, 0), (smat.KERNEL_AUTO, 1), (smat.KERNEL_ROWWISE_DIRECT, 0)}
    plan.close()
