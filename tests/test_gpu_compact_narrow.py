"""Compact kernel on products of up to 32 columns: panels of 16 and 32 columns."""
import ctypes

import numpy as np
import pytest

from smat_amd import generators as gen

pytestmark = pytest.mark.gpu


def to_dev(torch, a, cuda):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int16) if a.dtype == np.uint16 else np.ascontiguousarray(a)).to(cuda)


@pytest.fixture
def hooks(smat):
    lib = smat.lib
    for f in ("panel", "list", "staged"):
        getattr(lib, "smat_internal_compact_" + f).argtypes = [ctypes.c_int]
    yield lib
    for f in ("panel", "list", "staged"):
        getattr(lib, "smat_internal_compact_" + f)(0)


def sparse(M, K, per_row, seed, heavy=False):
    """About per_row nonzeros a row, small whole numbers; heavy: one block row with a nonzero in every column."""
    rng = np.random.default_rng(seed)
    r, c = rng.integers(0, M, M * per_row), rng.integers(0, K, M * per_row)
    if heavy:
        r, c = np.concatenate([r, np.full(K, 3)]), np.concatenate([c, np.arange(K)])
    key = np.unique(r * K + c)
    rp = np.zeros(M + 1, np.int32)
    np.add.at(rp, key // K + 1, 1)
    return np.cumsum(rp).astype(np.int32), (key % K).astype(np.int32), rng.integers(1, 4, key.size).astype(np.float16).view(np.uint16)


# K around tiles of 128 and 256 rows of the transposition; a row that is split
@pytest.mark.parametrize("M,K,per_row,heavy", [(16, 16, 2, False), (304, 528, 3, False), (1040, 2064, 12, False), (4096, 20000, 4, True)])
@pytest.mark.parametrize("N", [8, 16, 24, 32])
@pytest.mark.parametrize("lists,staged", [(1, 2), (2, 2), (2, 1)])
@pytest.mark.parametrize("row_major,c_f32", [(False, False), (True, True)])
def test_narrow_panels_match_the_oracle(smat, cuda, oracle, hooks, M, K, per_row, heavy, N, lists, staged, row_major, c_f32):
    import torch
    rp, ci, val = sparse(M, K, per_row, seed=M + N, heavy=heavy)
    A = smat.csr_to_bcsr(M, K, rp, ci, val)
    b = np.random.default_rng(N).integers(-4, 5, (N, K)).astype(np.float16)
    B = b.reshape(-1).view(np.uint16)
    hooks.smat_internal_compact_list(lists)
    hooks.smat_internal_compact_staged(staged)
    vals, brp, bci = to_dev(torch, A.val, cuda), to_dev(torch, A.row_ptr, cuda), to_dev(torch, A.col_idx, cuda)
    Bd = to_dev(torch, np.ascontiguousarray(b.T).reshape(-1).view(np.uint16) if row_major else B, cuda)
    plan = smat.Plan(A.row_ptr, M, K, A.nnzb, N, col_idx_host=A.col_idx, kernel=smat.KERNEL_COMPACT, b_row_major=row_major)
    plan.attach_values(vals, brp, bci)
    want = oracle.spmm_bcsr(M, N, K, A.row_ptr, A.col_idx, A.val, B, threads=4)
    want = want if c_f32 else want.astype(np.float16)
    for panel in (0, 1):  # whole numbers: the sums are exact in fp32 whatever the panel
        hooks.smat_internal_compact_panel(panel)
        C = torch.full((M, N), float("nan"), dtype=torch.float32 if c_f32 else torch.float16, device=cuda)
        smat.spmm(vals, brp, bci, Bd, C, M, N, K, A.nnzb, plan=plan, c_f32=c_f32, kernel=smat.KERNEL_COMPACT, b_row_major=row_major)
        assert np.array_equal(C.cpu().numpy(), want)
    plan.close()


@pytest.mark.parametrize("width,most", [(16, 64), (32, 72), (64, 128), (128, 168)])
@pytest.mark.parametrize("c_f32", [0, 1])
def test_registers_leave_room_for_the_wavefronts(smat, cuda, width, most, c_f32):
    """512 registers a SIMD: eight wavefronts of panels of 16 columns, seven of 32, four of 64 and three of 128."""
    registers = smat.lib.smat_internal_compact_registers(width, c_f32)
    assert 0 < registers <= most
