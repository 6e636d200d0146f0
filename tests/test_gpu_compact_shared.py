"""Compact kernel: tasks whose steps are shared by the wavefronts of a workgroup."""
import ctypes

import numpy as np
import pytest

from tests.test_gpu_compact_narrow import to_dev

pytestmark = pytest.mark.gpu

HOOKS = ("panel", "list", "staged", "share")


@pytest.fixture
def hooks(smat):
    lib = smat.lib
    for f in HOOKS:
        getattr(lib, "smat_internal_compact_" + f).argtypes = [ctypes.c_int]
    yield lib
    for f in HOOKS:
        getattr(lib, "smat_internal_compact_" + f)(0)


# columns of the block rows: steps of 32 that two and four wavefronts share evenly, unevenly, and fewer than the wavefronts; 0 = an empty row
ROWS = [(1,), (31, 33, 0, 64), (97, 128, 129, 160, 0, 257, 5), (1500, 0, 2064, 700), (2064,) + (40,) * 30]  # the last: a row that is split


def rows_of(lengths, K, per_column, seed):
    """CSR with the given number of nonzero columns in every block row, per_column nonzeros each, small whole numbers."""
    rng = np.random.default_rng(seed)
    keys = []
    for i, n in enumerate(lengths):
        for c in rng.permutation(K)[:n]:
            for r in rng.permutation(16)[:per_column]:
                keys.append((16 * i + r) * K + c)
    key = np.sort(np.array(keys, np.int64))
    rp = np.zeros(16 * len(lengths) + 1, np.int32)
    np.add.at(rp, key // K + 1, 1)
    return np.cumsum(rp).astype(np.int32), (key % K).astype(np.int32), rng.integers(1, 4, key.size).astype(np.float16).view(np.uint16)


@pytest.mark.parametrize("lengths", ROWS)
@pytest.mark.parametrize("N,panel", [(8, 0), (32, 0), (72, 1), (136, 2)])
@pytest.mark.parametrize("lists,staged,per_column", [(1, 2, 3), (2, 2, 1), (2, 1, 1), (2, 1, 3)])
@pytest.mark.parametrize("row_major,c_f32", [(False, False), (True, True)])
def test_shared_tasks_match_the_oracle(smat, cuda, oracle, hooks, lengths, N, panel, lists, staged, per_column, row_major, c_f32):
    import torch
    M, K = 16 * len(lengths), 2064
    may = per_column > 1 or row_major  # columns of one nonzero, column-major: one wavefront a task
    rp, ci, val = rows_of(lengths, K, per_column, seed=N + per_column)
    A = smat.csr_to_bcsr(M, K, rp, ci, val)
    b = np.random.default_rng(N).integers(-4, 5, (N, K)).astype(np.float16)
    want = oracle.spmm_bcsr(M, N, K, A.row_ptr, A.col_idx, A.val, b.reshape(-1).view(np.uint16), threads=4)
    want = want if c_f32 else want.astype(np.float16)
    hooks.smat_internal_compact_list(lists)
    hooks.smat_internal_compact_staged(staged)
    hooks.smat_internal_compact_panel(panel)
    vals, brp, bci = to_dev(torch, A.val, cuda), to_dev(torch, A.row_ptr, cuda), to_dev(torch, A.col_idx, cuda)
    Bd = to_dev(torch, (np.ascontiguousarray(b.T) if row_major else b).reshape(-1).view(np.uint16), cuda)
    plan = smat.Plan(A.row_ptr, M, K, A.nnzb, N, col_idx_host=A.col_idx, kernel=smat.KERNEL_COMPACT, b_row_major=row_major)
    plan.attach_values(vals, brp, bci)
    for share in (1, 2, 4):  # whole numbers: the sums are exact in fp32 in any order
        hooks.smat_internal_compact_share(share)
        C = torch.full((M, N), float("nan"), dtype=torch.float32 if c_f32 else torch.float16, device=cuda)
        smat.spmm(vals, brp, bci, Bd, C, M, N, K, A.nnzb, plan=plan, c_f32=c_f32, kernel=smat.KERNEL_COMPACT, b_row_major=row_major)
        assert hooks.smat_internal_compact_last_share() == (share if may else 1)
        assert np.array_equal(C.cpu().numpy(), want)
    plan.close()


def full_blocks_and_pairs(mb, kb, keep, per_row, seed):
    """BCSR of full blocks, and between them nonzeros in pairs, one below the other, small whole numbers."""
    rng = np.random.default_rng(seed)
    blocks = np.zeros((mb, kb, 16, 16), np.float16)
    full = rng.random((mb, kb)) < keep
    blocks[full] = rng.integers(1, 3, (full.sum(), 16, 16))
    row = np.repeat(np.arange(16 * mb), per_row)
    col = rng.integers(0, 16 * kb, row.size)
    for r in (row, row ^ 1):
        blocks[r // 16, col // 16, r % 16, col % 16] = 1
    there = blocks.any((2, 3))
    rp = np.concatenate([[0], np.cumsum(there.sum(1))]).astype(np.int32)
    return rp, (np.nonzero(there)[1] * 16).astype(np.int32), np.ascontiguousarray(blocks[there]).reshape(-1).view(np.uint16)


# One kernel for all blocks, as the rule says by itself; and the list added to what the sweep kernel wrote of the full blocks, where a plan asks for that by name and only the hook
# shares tasks.
@pytest.mark.parametrize("mb,kb,keep,per_row,N,kernel,share", [(224, 257, 0.08, 5, 96, 0, 2), (100, 2600, 0.0, 32, 48, 0, 4), (2, 256, 0.30, 12, 16384, 6, 1)])
@pytest.mark.parametrize("row_major", [False, True])
def test_plans_that_attach_values_share_tasks(smat, cuda, oracle, hooks, mb, kb, keep, per_row, N, kernel, share, row_major):
    import torch
    M, K = 16 * mb, 16 * kb
    rp, ci, val = full_blocks_and_pairs(mb, kb, keep, per_row, seed=N)
    nnzb = len(ci)
    b = np.random.default_rng(N).integers(-1, 2, (N, K)).astype(np.float16)
    want = oracle.spmm_bcsr(M, N, K, rp, ci, val, b.reshape(-1).view(np.uint16), threads=8)
    assert np.abs(want).max() <= 2048  # whole numbers in fp16
    vals, brp, bci = to_dev(torch, val, cuda), to_dev(torch, rp, cuda), to_dev(torch, ci, cuda)
    Bd = to_dev(torch, (np.ascontiguousarray(b.T) if row_major else b).reshape(-1).view(np.uint16), cuda)
    plan = smat.Plan(rp, M, K, nnzb, N, col_idx_host=ci, kernel=kernel, b_row_major=row_major)
    plan.attach_values(vals, brp, bci)
    assert plan.info()["kernel"] == (kernel or smat.KERNEL_COMPACT)
    for forced in (0, 2, 4, 1):
        hooks.smat_internal_compact_share(forced)
        for c_f32 in (False, True):
            C = torch.full((M, N), float("nan"), dtype=torch.float32 if c_f32 else torch.float16, device=cuda)
            smat.spmm(vals, brp, bci, Bd, C, M, N, K, nnzb, plan=plan, c_f32=c_f32, b_row_major=row_major, kernel=kernel)
            assert np.array_equal(C.cpu().numpy(), want if c_f32 else want.astype(np.float16)), forced
            assert hooks.smat_internal_compact_last_share() == (forced or share)
    plan.close()
