"""Sweep kernel on row-major B read in place: the bits that it writes for the column-major copy of the same B."""
import ctypes

import numpy as np
import pytest

from smat_amd import generators as gen

pytestmark = pytest.mark.gpu


def to_dev(torch, a, cuda):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int16) if a.dtype == np.uint16 else np.ascontiguousarray(a)).to(cuda)


# one panel and a part of one, N of one 8-column piece, K of one block column, of whole chunks and of chunks and a rest, one row
# group and several, rows of B that start at every multiple of 16 bytes of a cache line
@pytest.mark.parametrize("mb,kb,density,N", [(64, 64, 0.1, 64), (20, 17, 0.3, 8), (70, 33, 0.2, 1000), (5, 100, 0.5, 72), (64, 16, 0.4, 200),
                                             (3, 1, 1.0, 136), (130, 47, 0.03, 520), (257, 64, 0.1, 4104)])
@pytest.mark.parametrize("c_f32", [False, True])
def test_row_major_b_gives_the_bits_of_column_major_b(smat, cuda, oracle, mb, kb, density, N, c_f32):
    import torch
    A = gen.random_bcsr(mb, kb, density, seed=mb + kb)
    M, K, nnzb = A["M"], A["K"], A["nnzb"]
    B = gen.dense_b(K, N, seed=N)
    vals, rp, ci = (to_dev(torch, x, cuda) for x in (A["b_val"], A["b_row_ptr"].astype(np.int32), A["b_col_idx"].astype(np.int32)))
    out = []
    for row_major in (False, True):
        plan = smat.Plan(A["b_row_ptr"], M, K, nnzb, N, col_idx_host=A["b_col_idx"], kernel=smat.KERNEL_SWEEP, b_row_major=row_major)
        Bd = to_dev(torch, np.ascontiguousarray(B.reshape(N, K).T) if row_major else B, cuda)
        C = torch.full((M, N), float("nan"), dtype=torch.float32 if c_f32 else torch.float16, device=cuda)
        smat.spmm(vals, rp, ci, Bd, C, M, N, K, nnzb, plan=plan, kernel=smat.KERNEL_SWEEP, c_f32=c_f32, b_row_major=row_major)
        torch.cuda.synchronize()
        out.append(C.cpu().numpy())
        if row_major:  # the plan still takes a column-major B
            C.fill_(float("nan"))
            smat.spmm(vals, rp, ci, to_dev(torch, B, cuda), C, M, N, K, nnzb, plan=plan, kernel=smat.KERNEL_SWEEP, c_f32=c_f32)
            torch.cuda.synchronize()
            out.append(C.cpu().numpy())
    bits = np.uint32 if c_f32 else np.uint16
    assert np.array_equal(out[0].view(bits), out[1].view(bits)) and np.array_equal(out[0].view(bits), out[2].view(bits))
    want = oracle.spmm_bcsr(M, N, K, A["b_row_ptr"], A["b_col_idx"], A["b_val"], B, threads=4)
    if c_f32:
        oracle.assert_fp32_close(out[1], want, N, K, A, B)
    else:
        assert oracle.compare(out[1].view(np.uint16), want)[0] <= 1e-3


def test_infinities_in_row_major_b_stay_in_their_column(smat, cuda):
    """An Inf next to the blocks of a row (in the block column behind an unpaired one, in the rows past the last chunk's blocks)
    must not reach C."""
    import torch
    mb, kb, N = 64, 40, 64
    rng = np.random.default_rng(1)
    ci = np.sort(rng.choice(kb // 2, (mb, 3)), axis=1) * 2 * 16  # even block columns only, some twice: made unique below
    rows = [np.unique(c) for c in ci]
    rp = np.concatenate([[0], np.cumsum([r.size for r in rows])]).astype(np.int32)
    ci = np.concatenate(rows).astype(np.int32)
    val = gen.f16_bits(rng.normal(size=ci.size * 256))
    B = rng.normal(size=(kb * 16, N)).astype(np.float16)
    B.reshape(kb, 16, N)[1::2] = np.inf
    plan = smat.Plan(rp, mb * 16, kb * 16, ci.size, N, col_idx_host=ci, kernel=smat.KERNEL_SWEEP, b_row_major=True)
    vals, rpd, cid, Bd = (to_dev(torch, x, cuda) for x in (val, rp, ci, B.view(np.uint16)))
    C = torch.full((mb * 16, N), float("nan"), dtype=torch.float16, device=cuda)
    smat.spmm(vals, rpd, cid, Bd, C, mb * 16, N, kb * 16, ci.size, plan=plan, kernel=smat.KERNEL_SWEEP, b_row_major=True)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(C).all())


# row groups of fewer than 64 block rows chosen for the rounds (29 to 43): blocks of three and four row groups in the
# order of the tiles, a last group that is not full
@pytest.mark.parametrize("mb,N", [(128, 8960), (200, 4136), (321, 2728), (450, 2408)])
@pytest.mark.parametrize("row_major", [False, True])
def test_groups_chosen_for_the_rounds_match_the_oracle(smat, cuda, oracle, mb, N, row_major):
    import torch
    A = gen.random_bcsr(mb, 40, 0.3, seed=mb)
    M, K, nnzb = A["M"], A["K"], A["nnzb"]
    rows = smat.lib.smat_internal_sweep_even_rounds
    rows.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_size_t, ctypes.c_size_t, ctypes.c_int]
    g = rows(A["b_row_ptr"].ctypes.data, A["b_col_idx"].ctypes.data, M, K, N, int(row_major))
    assert g < 64
    B = gen.dense_b(K, N, seed=N)
    vals, rp, ci = (to_dev(torch, x, cuda) for x in (A["b_val"], A["b_row_ptr"].astype(np.int32), A["b_col_idx"].astype(np.int32)))
    Bd = to_dev(torch, np.ascontiguousarray(B.reshape(N, K).T) if row_major else B, cuda)
    plan = smat.Plan(A["b_row_ptr"], M, K, nnzb, N, col_idx_host=A["b_col_idx"], b_row_major=row_major)
    assert plan.info()["kernel"] == smat.KERNEL_SWEEP
    C = torch.full((M, N), float("nan"), dtype=torch.float16, device=cuda)
    smat.spmm(vals, rp, ci, Bd, C, M, N, K, nnzb, plan=plan, b_row_major=row_major)
    torch.cuda.synchronize()
    want = oracle.spmm_bcsr(M, N, K, A["b_row_ptr"], A["b_col_idx"], A["b_val"], B, threads=4)
    assert oracle.compare(C.cpu().numpy().view(np.uint16), want)[0] <= 1e-3
