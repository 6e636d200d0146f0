"""The row-wise kernels at every number of block pairs that is left over: rows of 0 to 10 blocks (all pairs asked for at once), rows that four wavefronts
share (runs of 1 to 9 pairs, some empty), and rows that one wavefront takes two pairs at a time, past the 64 blocks of one load of indices; rows cut
in chunks; on either layout of B."""
import numpy as np
import pytest

from smat_amd import generators as gen

pytestmark = pytest.mark.gpu

LENGTHS = {"short": list(range(11)) * 2, "shared": list(range(12, 76)), "whole": list(range(1, 71)) * 10,
           "split": [1, 300, 0, 2, 32, 33, 34, 35, 500, 0] + [3] * 60,  # pieces of at most 32 blocks
          "outlier": [34, 60, 1] * 120 + [200]}                        # N = 136: one row is cut, and whole ones are longer than its pieces


@pytest.mark.parametrize("rows", sorted(LENGTHS))
@pytest.mark.parametrize("N", [8, 24, 40, 64, 136])
@pytest.mark.parametrize("packed", [False, True])
def test_every_remainder(smat, cuda, oracle, rows, N, packed):
    import torch
    lengths = [n for n in LENGTHS[rows] if not (rows == "shared" and n > 64)]  # not split
    A = gen.random_bcsr(len(lengths), max(90, max(lengths)), 0.0, seed=5 + N, row_lengths=lengths)
    M, K, nnzb = A["M"], A["K"], A["nnzb"]
    B = gen.dense_b(K, N, seed=N + 2)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a).view(np.int16) if a.dtype == np.uint16 else np.ascontiguousarray(a)).to(cuda)  # noqa: E731
    vals, rp, ci, Bd = dev(A["b_val"]), dev(A["b_row_ptr"].astype(np.int32)), dev(A["b_col_idx"].astype(np.int32)), dev(B)
    kernel = smat.KERNEL_ROWWISE_PACKED if packed else smat.KERNEL_ROWWISE_DIRECT
    plan = smat.Plan(A["b_row_ptr"], M, K, nnzb, N, col_idx_host=A["b_col_idx"], kernel=kernel)
    assert (plan.info()["split_rows"] > 0) == (rows in ("split", "outlier"))
    C = torch.full((M, N), float("nan"), dtype=torch.float32, device=cuda)
    smat.spmm(vals, rp, ci, Bd, C, M, N, K, nnzb, plan=plan, kernel=kernel, c_f32=True)
    torch.cuda.synchronize()
    if not packed:  # B as rows, read in place, gives the same bits
        plan = smat.Plan(A["b_row_ptr"], M, K, nnzb, N, col_idx_host=A["b_col_idx"], kernel=kernel, b_row_major=True)
        rows_of_b = Bd.view(N, K).t().contiguous()
        for c_f32, same in ((True, C), (False, C.half())):
            R = torch.full((M, N), float("nan"), dtype=same.dtype, device=cuda)
            smat.spmm(vals, rp, ci, rows_of_b, R, M, N, K, nnzb, plan=plan, kernel=kernel, c_f32=c_f32, b_row_major=True)
            torch.cuda.synchronize()
            assert torch.equal(R, same)
    # fp32 sums of exact products in another order: n roundings of 2^-24 of what the terms add up to, n <= 500 * 16
    dense = np.zeros((M, K))
    v = A["b_val"].view(np.float16).astype(np.float64).reshape(-1, 16, 16)
    for i in range(M // 16):
        for p in range(A["b_row_ptr"][i], A["b_row_ptr"][i + 1]):
            dense[16 * i:16 * i + 16, A["b_col_idx"][p]:A["b_col_idx"][p] + 16] = v[p]
    b = B.view(np.float16).astype(np.float64).reshape(N, K).T
    err = np.abs(C.cpu().numpy() - dense @ b)
    assert np.all(err <= max(lengths) * 16 * 2.0 ** -24 * (np.abs(dense) @ np.abs(b)))
