"""Row-wise launches of few long items: the four wavefronts of a workgroup share one (block row, panel)."""
import numpy as np
import pytest

from smat_amd import generators as gen

pytestmark = pytest.mark.gpu


def to_dev(torch, a, cuda):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int16) if a.dtype == np.uint16 else np.ascontiguousarray(a)).to(cuda)


# rows of no block, of fewer blocks than wavefronts, around a batch of pairs, around the window of 64 column indices
LENGTHS = [0, 1, 2, 7, 8, 9, 23, 24, 25, 63, 64, 65, 127, 128, 129, 140]


@pytest.mark.parametrize("N", [8, 24, 40, 64, 200])
@pytest.mark.parametrize("kernel", [3, 4])
@pytest.mark.parametrize("c_f32", [False, True])
def test_shared_items_match_the_oracle(smat, cuda, oracle, N, kernel, c_f32):
    import torch
    A = gen.random_bcsr(len(LENGTHS), 144, 0.0, seed=N, row_lengths=LENGTHS)
    M, K, nnzb = A["M"], A["K"], A["nnzb"]
    B = gen.dense_b(K, N, seed=N + 1)
    vals, rp, ci, Bd = (to_dev(torch, x, cuda) for x in (A["b_val"], A["b_row_ptr"].astype(np.int32), A["b_col_idx"].astype(np.int32), B))
    C = torch.full((M, N), float("nan"), dtype=torch.float32 if c_f32 else torch.float16, device=cuda)
    plan = smat.Plan(A["b_row_ptr"], M, K, nnzb, N, col_idx_host=A["b_col_idx"], kernel=kernel)
    smat.spmm(vals, rp, ci, Bd, C, M, N, K, nnzb, plan=plan, kernel=kernel, c_f32=c_f32)
    torch.cuda.synchronize()
    want = oracle.spmm_bcsr(M, N, K, A["b_row_ptr"], A["b_col_idx"], A["b_val"], B, threads=4)
    if c_f32:
        oracle.assert_fp32_close(C.cpu().numpy(), want, N, K, A, B)
    else:
        assert oracle.compare(C.cpu().numpy().view(np.uint16), want)[0] <= 1e-3
    # the plan-less launch works on whole block rows too: the same sums
    if kernel == 3:
        C2 = torch.full_like(C, float("nan"))
        smat.spmm(vals, rp, ci, Bd, C2, M, N, K, nnzb, kernel=kernel, c_f32=c_f32)
        torch.cuda.synchronize()
        if plan.info()["split_rows"] == 0:
            assert torch.equal(C, C2)


# even numbers of blocks: every pair is complete, so a column of B that is Inf gives Inf (the values of A are positive)
@pytest.mark.parametrize("lengths", [[2, 4, 6, 8, 10, 0, 4, 2] * 8, [2, 4, 14, 24, 26, 30, 46, 64, 66, 126, 128, 140]])
@pytest.mark.parametrize("N", [8, 40, 72, 200])
@pytest.mark.parametrize("kernel", [3, 4])
def test_infinities_under_complete_pairs_stay_infinities(smat, cuda, lengths, N, kernel):
    import torch
    A = gen.random_bcsr(len(lengths), 144, 0.0, seed=N, row_lengths=lengths)
    M, K, nnzb = A["M"], A["K"], A["nnzb"]
    val = np.full(nnzb * 256, np.float16(0.5)).view(np.uint16)
    B = np.full((N, K), np.float16(0.25))
    B[3] = np.inf
    vals, rp, ci, Bd = (to_dev(torch, x, cuda) for x in (val, A["b_row_ptr"].astype(np.int32), A["b_col_idx"].astype(np.int32), B.view(np.uint16)))
    plan = smat.Plan(A["b_row_ptr"], M, K, nnzb, N, col_idx_host=A["b_col_idx"], kernel=kernel)
    want = np.repeat(2.0 * np.array(lengths, np.float32), 16)[:, None].repeat(N, 1)  # 16 products of 0.5 * 0.25 a block
    want[:, 3] = np.where(np.repeat(lengths, 16) > 0, np.inf, 0)
    for p in (plan, None) if kernel == 3 else (plan,):
        C = torch.full((M, N), float("nan"), dtype=torch.float32, device=cuda)
        smat.spmm(vals, rp, ci, Bd, C, M, N, K, nnzb, plan=p, kernel=kernel, c_f32=True)
        torch.cuda.synchronize()
        assert np.array_equal(C.cpu().numpy(), want)
