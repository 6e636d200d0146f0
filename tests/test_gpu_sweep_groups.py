"""Sweep kernel on row groups of fewer than 64 block rows: what a plan takes where groups of 64 would leave compute units idle."""
import numpy as np
import pytest

from smat_amd import generators as gen

pytestmark = pytest.mark.gpu


def to_dev(torch, a, cuda):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int16) if a.dtype == np.uint16 else np.ascontiguousarray(a)).to(cuda)


def check(oracle, C, want, N, K, A, B):
    C = C.cpu().numpy()
    if C.dtype == np.float32:
        oracle.assert_fp32_close(C, want, N, K, A, B)
    else:
        assert oracle.compare(C.view(np.uint16), want)[0] <= 1e-3


# block rows around one, two and four groups of 16 and 32, a last group of one row, K not a multiple of a chunk
@pytest.mark.parametrize("mb,kb,density,N", [(48, 64, 0.3, 4096), (49, 33, 0.5, 2048), (17, 64, 0.4, 8192), (65, 49, 0.4, 2504), (193, 64, 0.1, 1608)])
@pytest.mark.parametrize("c_f32", [False, True])
def test_small_row_groups_match_the_oracle(smat, cuda, oracle, mb, kb, density, N, c_f32):
    import torch
    A = gen.random_bcsr(mb, kb, density, seed=mb + kb)
    M, K, nnzb = A["M"], A["K"], A["nnzb"]
    B = gen.dense_b(K, N, seed=N)
    vals, rp, ci, Bd = (to_dev(torch, x, cuda) for x in (A["b_val"], A["b_row_ptr"].astype(np.int32), A["b_col_idx"].astype(np.int32), B))
    plan = smat.Plan(A["b_row_ptr"], M, K, nnzb, N, col_idx_host=A["b_col_idx"])
    plan.attach_values(vals, rp, ci)
    assert plan.info()["kernel"] == smat.KERNEL_SWEEP
    want = oracle.spmm_bcsr(M, N, K, A["b_row_ptr"], A["b_col_idx"], A["b_val"], B, threads=4)
    C = torch.full((M, N), float("nan"), dtype=torch.float32 if c_f32 else torch.float16, device=cuda)
    smat.spmm(vals, rp, ci, Bd, C, M, N, K, nnzb, plan=plan, c_f32=c_f32)
    torch.cuda.synchronize()
    check(oracle, C, want, N, K, A, B)
    # the same plan at another width: the first columns of the same product, through whichever kernel that width takes
    n = 64
    C2 = torch.full((M, n), float("nan"), dtype=C.dtype, device=cuda)
    smat.spmm(vals, rp, ci, Bd, C2, M, n, K, nnzb, plan=plan, c_f32=c_f32)
    torch.cuda.synchronize()
    first = oracle.spmm_bcsr(M, n, K, A["b_row_ptr"], A["b_col_idx"], A["b_val"], B[:n * K], threads=4)
    check(oracle, C2, first, n, K, A, B[:n * K])


# bands: few blocks of the matrix, few chunks for a row group; a last group of one block row, edges cut off
@pytest.mark.parametrize("m,bandwidth,N", [(4096, 30, 1024), (4112, 64, 1000), (8192, 100, 520)])
def test_bands_match_the_oracle(smat, cuda, oracle, m, bandwidth, N):
    import torch
    d = gen.band(m, bandwidth)
    A = smat.csr_to_bcsr(d["M"], d["K"], d["row_ptr"], d["col_idx"], d["val"])
    B = gen.dense_b(A.K, N, seed=m)
    vals, rp, ci, Bd = (to_dev(torch, x, cuda) for x in (A.val, A.row_ptr, A.col_idx, B))
    plan = smat.Plan(A.row_ptr, A.M, A.K, A.nnzb, N, col_idx_host=A.col_idx)
    plan.attach_values(vals, rp, ci)
    assert plan.info()["kernel"] == smat.KERNEL_SWEEP
    C = torch.full((A.M, N), float("nan"), dtype=torch.float16, device=cuda)
    smat.spmm(vals, rp, ci, Bd, C, A.M, N, A.K, A.nnzb, plan=plan)
    torch.cuda.synchronize()
    want = oracle.spmm_bcsr(A.M, N, A.K, A.row_ptr, A.col_idx, A.val, B, threads=4)
    assert oracle.compare(C.cpu().numpy().view(np.uint16), want)[0] <= 1e-3


def block_diagonal(mb, width):
    """Block row i holds the `width` block columns around i: a row group lists one or two chunks of 16 block columns."""
    cols = [range(max(0, i - width // 2), min(mb, i + (width + 1) // 2)) for i in range(mb)]
    rp = np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.int32)
    ci = np.concatenate([np.array(c) for c in cols]).astype(np.int32) * 16
    val = gen.f16_bits(np.random.default_rng(mb).normal(size=ci.size * 256))
    return {"M": mb * 16, "K": mb * 16, "b_row_ptr": rp, "b_col_idx": ci, "b_val": val, "nnzb": ci.size}


# groups that list one or two chunks, fewer than the entry fetches; a last group of one block row
@pytest.mark.parametrize("group_rows", [64, 32, 16])
@pytest.mark.parametrize("mb,width", [(64, 1), (49, 1), (65, 2), (81, 3)])
@pytest.mark.parametrize("c_f32", [False, True])
def test_groups_of_few_chunks_match_the_oracle(smat, cuda, oracle, group_rows, mb, width, c_f32):
    import torch
    A = block_diagonal(mb, width)
    M, K, nnzb, N = A["M"], A["K"], A["nnzb"], 200
    B = gen.dense_b(K, N, seed=mb)
    vals, rp, ci, Bd = (to_dev(torch, x, cuda) for x in (A["b_val"], A["b_row_ptr"], A["b_col_idx"], B))
    smat.lib.smat_internal_sweep_force_groups(group_rows)
    try:
        plan = smat.Plan(A["b_row_ptr"], M, K, nnzb, N, col_idx_host=A["b_col_idx"])
        plan.attach_values(vals, rp, ci)
    finally:
        smat.lib.smat_internal_sweep_force_groups(0)
    assert plan.info()["kernel"] == smat.KERNEL_SWEEP
    C = torch.full((M, N), float("nan"), dtype=torch.float32 if c_f32 else torch.float16, device=cuda)
    smat.spmm(vals, rp, ci, Bd, C, M, N, K, nnzb, plan=plan, kernel=smat.KERNEL_SWEEP, c_f32=c_f32)
    torch.cuda.synchronize()
    check(oracle, C, oracle.spmm_bcsr(M, N, K, A["b_row_ptr"], A["b_col_idx"], A["b_val"], B, threads=4), N, K, A, B)


@pytest.mark.parametrize("c_f32", [False, True])
def test_row_groups_without_a_block_give_zeros(smat, cuda, oracle, c_f32):
    import torch
    lengths = [0 if 64 <= r < 128 else 3 for r in range(16 * 64)]  # the second of 16 groups of 64 block rows is empty
    A = gen.random_bcsr(len(lengths), 33, 0.0, seed=5, row_lengths=lengths)
    M, K, nnzb, N = A["M"], A["K"], A["nnzb"], 136
    B = gen.dense_b(K, N, seed=N)
    vals, rp, ci, Bd = (to_dev(torch, x, cuda) for x in (A["b_val"], A["b_row_ptr"].astype(np.int32), A["b_col_idx"].astype(np.int32), B))
    plan = smat.Plan(A["b_row_ptr"], M, K, nnzb, N, col_idx_host=A["b_col_idx"], kernel=smat.KERNEL_SWEEP)
    C = torch.full((M, N), float("nan"), dtype=torch.float32 if c_f32 else torch.float16, device=cuda)
    smat.spmm(vals, rp, ci, Bd, C, M, N, K, nnzb, plan=plan, kernel=smat.KERNEL_SWEEP, c_f32=c_f32)
    torch.cuda.synchronize()
    want = oracle.spmm_bcsr(M, N, K, A["b_row_ptr"], A["b_col_idx"], A["b_val"], B, threads=4)
    assert (C[64 * 16:128 * 16] == 0).all()
    check(oracle, C, want, N, K, A, B)
