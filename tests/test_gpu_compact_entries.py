"""The compact kernel on lists of single nonzeros: steps with more entries than are asked for at once, items put together
into tasks, empty block rows between and around them."""
import numpy as np
import pytest

from smat_amd import generators as gen

pytestmark = pytest.mark.gpu


def to_dev(torch, a, cuda):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int16) if a.dtype == np.uint16 else np.ascontiguousarray(a)).to(cuda)


def matrix(fill, seed):
    """Block rows of 0 .. 70 blocks, K above 4096 (lists of nonzeros), fill nonzeros per nonzero column on average:
    one row or several of a column; some block rows hold full columns, so that a step has up to 512 entries."""
    rng = np.random.default_rng(seed)
    mb, kb = 40, 300
    lengths = [0, 1, 2, 3, 31, 32, 33, 0, 0, 70] + list(rng.integers(0, 40, mb - 11)) + [0]
    A = gen.random_bcsr(mb, kb, 0.0, seed=seed, row_lengths=lengths)
    v = A["b_val"].reshape(-1, 16, 16).copy()
    keep = np.zeros(v.shape, bool)
    for p in range(v.shape[0]):
        cols = rng.choice(16, int(rng.integers(1, 5)), replace=False)
        for c in cols:
            n = 16 if p % 37 == 0 else min(16, max(1, int(rng.poisson(fill - 1)) + 1))
            keep[p, rng.choice(16, n, replace=False), c] = True
    v[~keep] = 0
    A["b_val"] = v.reshape(-1)
    return A


@pytest.mark.parametrize("fill", [1.0, 2.5])
@pytest.mark.parametrize("N", [8, 64, 136])
@pytest.mark.parametrize("c_f32,row_major", [(False, False), (True, False), (False, True)])
def test_lists_of_nonzeros_match_the_oracle(smat, cuda, oracle, fill, N, c_f32, row_major):
    import torch
    A = matrix(fill, 7 + N)
    M, K, nnzb = A["M"], A["K"], A["nnzb"]
    B = gen.dense_b(K, N, seed=N + 1)
    vals, rp, ci, Bd = (to_dev(torch, x, cuda) for x in (A["b_val"], A["b_row_ptr"].astype(np.int32), A["b_col_idx"].astype(np.int32), B))
    if row_major:
        Bd = Bd.view(N, K).t().contiguous()
    want = oracle.spmm_bcsr(M, N, K, A["b_row_ptr"], A["b_col_idx"], A["b_val"], B, threads=4)
    for tq in (1, 2):  # panels of 64 and of 128 columns
        smat.lib.smat_internal_compact_panel(tq)
        try:
            C = torch.full((M, N), float("nan"), dtype=torch.float32 if c_f32 else torch.float16, device=cuda)
            plan = smat.Plan(A["b_row_ptr"], M, K, nnzb, N, col_idx_host=A["b_col_idx"], kernel=5, b_row_major=row_major)
            plan.attach_values(vals, rp, ci)
            smat.spmm(vals, rp, ci, Bd, C, M, N, K, nnzb, plan=plan, kernel=5, c_f32=c_f32, b_row_major=row_major)
            torch.cuda.synchronize()
        finally:
            smat.lib.smat_internal_compact_panel(0)
        assert oracle.compare(C.half().cpu().numpy().view(np.uint16), want)[0] <= 1e-3
