"""The compact kernel on a copy of B that holds only the rows of B which meet a nonzero."""
import ctypes

import numpy as np
import pytest

from smat_amd import generators as gen

pytestmark = pytest.mark.gpu


def to_dev(torch, a, cuda):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int16) if a.dtype == np.uint16 else np.ascontiguousarray(a)).to(cuda)


def matrix(mb, K, used, seed):
    """Block rows of up to 40 nonzeros (one in eight without any) in the given columns of K."""
    rng = np.random.default_rng(seed)
    rp, ci, val = [0], [], []
    for b in range(mb):
        n = 0 if b % 8 == 3 else int(rng.integers(1, 41))
        cols = rng.choice(used, n, replace=False) if n else np.zeros(0, np.int64)
        blocks = np.unique(cols // 16)
        v = np.zeros((blocks.size, 16, 16), np.float16)
        for c in cols:
            v[np.searchsorted(blocks, c // 16), rng.integers(0, 16), c % 16] = rng.normal()
        ci.append(blocks * 16)
        val.append(v.reshape(-1))
        rp.append(rp[-1] + blocks.size)
    return {"M": mb * 16, "K": K, "nnzb": rp[-1], "b_row_ptr": np.array(rp, np.int32), "b_col_idx": np.concatenate(ci).astype(np.int32),
            "b_val": np.concatenate(val).view(np.uint16)}


# which columns have nonzeros: the first and the last among them or not, all (then nothing is left out), few
@pytest.mark.parametrize("used,placed", [("odd", True), ("even", True), ("all", False), ("middle", True)])
@pytest.mark.parametrize("N", [136, 256])
@pytest.mark.parametrize("c_f32,whole_columns", [(False, False), (True, True)])
def test_products_on_the_placed_rows(smat, cuda, oracle, used, placed, N, c_f32, whole_columns):
    import torch
    K, mb = 65536, 60
    columns = {"odd": np.arange(1, K, 2), "even": np.arange(0, K, 2), "all": np.arange(K), "middle": np.arange(K // 2, K // 2 + 300)}[used]
    if used == "all":
        mb, K = 2000, 65536
        columns = np.arange(0, K)
    A = matrix(mb, K, columns, 5)
    if used == "all":
        # 2000 block rows of 20 on average leave too many columns out: one more block row of full blocks names them all
        v = np.zeros((K // 16, 16, 16), np.float16)
        v[:, 0, :] = 0.5
        A["b_row_ptr"] = np.append(A["b_row_ptr"], A["b_row_ptr"][-1] + K // 16).astype(np.int32)
        A["b_col_idx"] = np.append(A["b_col_idx"], np.arange(0, K, 16)).astype(np.int32)
        A["b_val"] = np.append(A["b_val"], v.reshape(-1).view(np.uint16))
        A["M"], A["nnzb"] = A["M"] + 16, A["nnzb"] + K // 16
    M, nnzb = A["M"], A["nnzb"]
    B = gen.dense_b(K, N, seed=N)
    vals, rp, ci = (to_dev(torch, x, cuda) for x in (A["b_val"], A["b_row_ptr"], A["b_col_idx"]))
    Bd = to_dev(torch, B, cuda)
    Brm = Bd.view(N, K).t().contiguous()
    smat.lib.smat_internal_compact_list(1 if whole_columns else 2)
    try:
        plan = smat.Plan(A["b_row_ptr"], M, K, nnzb, N, col_idx_host=A["b_col_idx"], kernel=smat.KERNEL_COMPACT)
        plan.attach_values(vals, rp, ci)
        in_place = smat.Plan(A["b_row_ptr"], M, K, nnzb, N, col_idx_host=A["b_col_idx"], kernel=smat.KERNEL_COMPACT, b_row_major=True)
        in_place.attach_values(vals, rp, ci)
    finally:
        smat.lib.smat_internal_compact_list(0)
    fn = smat.lib.smat_internal_compact_placed_rows
    fn.restype = ctypes.c_int64
    assert (0 < fn(plan.handle) < K) == placed and fn(in_place.handle) == 0

    def product(p, n, row_major):
        C = torch.full((M, n), float("nan"), dtype=torch.float32 if c_f32 else torch.float16, device=cuda)
        b = Brm[:, :n].contiguous() if row_major else Bd[:n * K]
        smat.spmm(vals, rp, ci, b, C, M, n, K, nnzb, plan=p, kernel=smat.KERNEL_COMPACT, c_f32=c_f32, b_row_major=row_major)
        torch.cuda.synchronize()
        return C.cpu().numpy()

    want = oracle.spmm_bcsr(M, N, K, A["b_row_ptr"], A["b_col_idx"], A["b_val"], B, threads=4)
    got = product(plan, N, False)
    if c_f32:
        oracle.assert_fp32_close(got, want, N, K, A, B)
    else:
        assert oracle.compare(got.view(np.uint16), want)[0] <= 1e-3
    # the same lists on B in place, through either plan, and narrower than the plan: the same bits
    assert np.array_equal(got, product(in_place, N, True)) and np.array_equal(got, product(plan, N, True))
    assert np.array_equal(got[:, :72], product(plan, 72, False))


@pytest.mark.parametrize("whole_columns", [False, True])
@pytest.mark.parametrize("K,used", [(65536, "odd"), (65552, "odd"), (262160, "last"), (65536, "all")])
def test_used_rows_are_counted_on_the_way(smat, cuda, whole_columns, K, used):
    """The copy holds the rows that the list names and row 0, which padding names; to find that none can be left out takes one
    allocation and no list, scan or copy of its own."""
    import torch
    columns = {"odd": np.arange(1, K, 2), "last": np.arange(K - 700, K), "all": np.arange(K)}[used]
    A = matrix(60 if used != "all" else 1, K, columns, 5)
    if used == "all":
        v = np.zeros((K // 16, 16, 16), np.float16)
        v[:, 0, :] = 0.5
        A["b_row_ptr"] = np.append(A["b_row_ptr"], A["b_row_ptr"][-1] + K // 16).astype(np.int32)
        A["b_col_idx"] = np.append(A["b_col_idx"], np.arange(0, K, 16)).astype(np.int32)
        A["b_val"] = np.append(A["b_val"], v.reshape(-1).view(np.uint16))
        A["M"], A["nnzb"] = A["M"] + 16, A["nnzb"] + K // 16
    M, nnzb = A["M"], A["nnzb"]
    vals, rp, ci = (to_dev(torch, x, cuda) for x in (A["b_val"], A["b_row_ptr"], A["b_col_idx"]))
    nonzero = (A["b_val"].reshape(-1, 16, 16) & 0x7fff != 0).any(axis=1)
    named = np.zeros(K, bool)
    np.logical_or.at(named, (A["b_col_idx"][:, None] + np.arange(16)).reshape(-1), nonzero.reshape(-1))
    named[0] = True
    counts, allocated = (ctypes.c_int64 * 2)(), []
    fn = smat.lib.smat_internal_compact_placed_rows
    fn.restype, fn.argtypes = ctypes.c_int64, [ctypes.c_void_p]
    smat.lib.smat_internal_compact_list(1 if whole_columns else 2)
    smat.lib.smat_internal_compact_tune(0)
    try:
        for N in (8, 256):  # a B that is too small to look, and one that is not
            plan = smat.Plan(A["b_row_ptr"], M, K, nnzb, N, col_idx_host=A["b_col_idx"], kernel=smat.KERNEL_COMPACT)
            plan.attach_values(vals, rp, ci)
            smat.lib.smat_internal_alloc_counts(counts)
            before = counts[0]
            plan.attach_values(vals, rp, ci)
            smat.lib.smat_internal_alloc_counts(counts)
            allocated.append(counts[0] - before)
            assert fn(plan.handle) == (named.sum() if N == 256 and used != "all" else 0)
    finally:
        smat.lib.smat_internal_compact_list(0)
        smat.lib.smat_internal_compact_tune(1)
    if used == "all":
        assert allocated[1] <= allocated[0] + 1
