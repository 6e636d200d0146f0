"""The compact kernel's tasks in the order that lists with split rows get (chunks by where they begin in their rows, whole rows by classes of length, empty
places where an XCD has fewer workgroups than another): the bits of the order of the items, and the oracle's product."""
import numpy as np
import pytest

from smat_amd import generators as gen

pytestmark = pytest.mark.gpu


def to_dev(torch, a, cuda):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int16) if a.dtype == np.uint16 else np.ascontiguousarray(a)).to(cuda)


def matrix(shape, seed):
    """Blocks of one nonzero; block rows of these numbers of blocks."""
    rng = np.random.default_rng(seed)
    kb = 2400
    lengths = {"one": [2300] + [2] * 30,                                          # chunks and one workgroup of whole rows
               "few": [0, 2100, 0, 5, 1500, 1] + [0, 3] * 20,                     # empty rows beside them
               "skewed": list(rng.integers(0, 12, 700)) + [2400, 1640, 2000, 0] + list(rng.integers(0, 150, 200)),
               "even": [1900] * 33}[shape]                                        # too few wavefronts: all rows are cut
    A = gen.random_bcsr(len(lengths), kb, 0.0, seed=seed, row_lengths=lengths)
    v = A["b_val"].reshape(-1, 256).copy()
    keep = np.zeros(v.shape, bool)
    keep[np.arange(v.shape[0]), rng.integers(0, 256, v.shape[0])] = True
    v[~keep] = 0
    A["b_val"] = v.reshape(-1)
    return A


@pytest.mark.parametrize("shape", ["one", "few", "skewed", "even"])
@pytest.mark.parametrize("N,c_f32,row_major", [(8, False, False), (64, True, False), (136, False, False), (200, False, True)])
def test_the_order_of_the_tasks_moves_no_bit(smat, cuda, oracle, shape, N, c_f32, row_major):
    import torch
    A = matrix(shape, 3 + N)
    M, K, nnzb = A["M"], A["K"], A["nnzb"]
    B = gen.dense_b(K, N, seed=N + 1)
    vals, rp, ci, Bd = (to_dev(torch, x, cuda) for x in (A["b_val"], A["b_row_ptr"].astype(np.int32), A["b_col_idx"].astype(np.int32), B))
    if row_major:
        Bd = Bd.view(N, K).t().contiguous()
    got = []
    for what in (1, 2):
        smat.lib.smat_internal_compact_order(what)
        try:
            plan = smat.Plan(A["b_row_ptr"], M, K, nnzb, N, col_idx_host=A["b_col_idx"], kernel=5, b_row_major=row_major)
            plan.attach_values(vals, rp, ci)
        finally:
            smat.lib.smat_internal_compact_order(0)
        assert smat.lib.smat_internal_compact_split_rows(plan.handle) > 0
        for n in (N, 8):  # the plan's width, and one of another number of panels
            C = torch.full((M, n), float("nan"), dtype=torch.float32 if c_f32 else torch.float16, device=cuda)
            b = Bd if n == N else (Bd[:, :n].contiguous() if row_major else Bd)
            smat.spmm(vals, rp, ci, b, C, M, n, K, nnzb, plan=plan, kernel=5, c_f32=c_f32, b_row_major=row_major)
            got.append(C)
    torch.cuda.synchronize()
    assert torch.equal(got[0], got[2]) and torch.equal(got[1], got[3])
    want = oracle.spmm_bcsr(M, N, K, A["b_row_ptr"], A["b_col_idx"], A["b_val"], B, threads=4)
    out = got[2].half().cpu().numpy().view(np.uint16)
    assert oracle.compare(out, want)[0] <= 1e-3
