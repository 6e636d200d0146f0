"""The compact kernel with entries staged in LDS by blocks of 256: the bits of the loads step by step, and the oracle's result."""
import numpy as np
import pytest

from smat_amd import generators as gen
from tests.test_gpu_compact_entries import STEPS, matrix, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture
def hooks(smat):
    yield smat.lib
    for hook in (smat.lib.smat_internal_compact_list, smat.lib.smat_internal_compact_staged, smat.lib.smat_internal_compact_panel):
        hook(0)


def long_rows(per_column, seed):
    """Block rows of 1 to 260 steps, per_column nonzeros in every column."""
    rng = np.random.default_rng(seed)
    A = gen.random_bcsr(len(STEPS), 528, 0.0, seed=seed, row_lengths=[2 * s for s in STEPS])
    v = A["b_val"].reshape(-1, 16, 16).copy()
    keep = np.zeros(v.shape, bool)
    for _ in range(per_column):
        keep[np.arange(v.shape[0])[:, None], rng.integers(0, 16, (v.shape[0], 16)), np.arange(16)[None, :]] = True
    v[~keep] = 0
    A["b_val"] = v.reshape(-1)
    return A


# one nonzero a column (a block of entries lasts eight steps) to sixteen in some (a step takes half of one), tasks of several
# items with empty block rows between them, tasks longer than one load of entry ranges, rows whole and split
@pytest.mark.parametrize("A", [matrix(1.0, 1), matrix(2.5, 2), matrix(6.0, 3), long_rows(1, 4), long_rows(3, 5)], ids=["one", "few", "many", "long", "long_3"])
@pytest.mark.parametrize("N,n_hint", [(64, 64), (136, 4096)])
@pytest.mark.parametrize("c_f32,row_major", [(False, False), (True, True)])
def test_staged_entries_give_the_same_bits(smat, cuda, oracle, hooks, A, N, n_hint, c_f32, row_major):
    import torch
    hooks.smat_internal_compact_list(2)
    M, K, nnzb = A["M"], A["K"], A["nnzb"]
    B = gen.dense_b(K, N, seed=N)
    vals, rp, ci, Bd = (to_dev(torch, x, cuda) for x in (A["b_val"], A["b_row_ptr"].astype(np.int32), A["b_col_idx"].astype(np.int32), B))
    if row_major:
        Bd = Bd.view(N, K).t().contiguous()
    plan = smat.Plan(A["b_row_ptr"], M, K, nnzb, n_hint, col_idx_host=A["b_col_idx"], kernel=smat.KERNEL_COMPACT, b_row_major=row_major)
    plan.attach_values(vals, rp, ci)
    want = oracle.spmm_bcsr(M, N, K, A["b_row_ptr"], A["b_col_idx"], A["b_val"], B, threads=4)
    for tq in (1, 2):
        hooks.smat_internal_compact_panel(tq)
        out = []
        for staged in (2, 1):
            hooks.smat_internal_compact_staged(staged)
            C = torch.full((M, N), float("nan"), dtype=torch.float32 if c_f32 else torch.float16, device=cuda)
            smat.spmm(vals, rp, ci, Bd, C, M, N, K, nnzb, plan=plan, kernel=smat.KERNEL_COMPACT, c_f32=c_f32, b_row_major=row_major)
            torch.cuda.synchronize()
            out.append(C.cpu().numpy())
        assert np.array_equal(out[0], out[1])
        if c_f32:
            oracle.assert_fp32_close(out[1], want, N, K, A, B)
        else:
            assert oracle.compare(out[1].view(np.uint16), want)[0] <= 1e-3
