"""Compact kernel: the last panel of the copy of a column-major B is as narrow as its columns."""
import numpy as np
import pytest

from tests.test_gpu_compact_narrow import hooks, sparse, to_dev  # noqa: F401

pytestmark = pytest.mark.gpu


# one column of eight past a panel, and every width of the last panel: 8, 16, 32 and 64 (panels of 128: 128) halves
@pytest.mark.parametrize("N", [72, 80, 88, 96, 104, 136, 168, 200, 264])
@pytest.mark.parametrize("panel", [1, 2])
@pytest.mark.parametrize("M,K,per_row,heavy", [(304, 528, 3, False), (1040, 2064, 12, True)])
@pytest.mark.parametrize("c_f32", [False, True])
def test_last_panels_match_the_oracle(smat, cuda, oracle, hooks, M, K, per_row, heavy, N, panel, c_f32):  # noqa: F811
    import torch
    rp, ci, val = sparse(M, K, per_row, seed=M + N, heavy=heavy)
    A = smat.csr_to_bcsr(M, K, rp, ci, val)
    B = np.random.default_rng(N).integers(-4, 5, (N, K)).astype(np.float16).reshape(-1).view(np.uint16)
    hooks.smat_internal_compact_panel(panel)
    vals, brp, bci, Bd = (to_dev(torch, x, cuda) for x in (A.val, A.row_ptr, A.col_idx, B))
    plan = smat.Plan(A.row_ptr, M, K, A.nnzb, N, col_idx_host=A.col_idx, kernel=smat.KERNEL_COMPACT)
    plan.attach_values(vals, brp, bci)
    want = oracle.spmm_bcsr(M, N, K, A.row_ptr, A.col_idx, A.val, B, threads=4)
    C = torch.full((M, N), float("nan"), dtype=torch.float32 if c_f32 else torch.float16, device=cuda)
    smat.spmm(vals, brp, bci, Bd, C, M, N, K, A.nnzb, plan=plan, c_f32=c_f32, kernel=smat.KERNEL_COMPACT)
    # whole numbers: the sums are exact in fp32
    assert np.array_equal(C.cpu().numpy(), want if c_f32 else want.astype(np.float16))
    plan.close()
