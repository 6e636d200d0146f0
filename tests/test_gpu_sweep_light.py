"""Light streams of the sweep kernel: products of few blocks a wavefront and chunk against the oracle, and against the other streams."""
import ctypes

import numpy as np
import pytest

from tests.test_gpu_compact_narrow import to_dev
from tests.test_sweep_plan import random_mask_matrix

pytestmark = pytest.mark.gpu


@pytest.fixture
def force(smat):
    smat.lib.smat_internal_sweep_force_light.argtypes = [ctypes.c_int]
    yield smat.lib.smat_internal_sweep_force_light
    smat.lib.smat_internal_sweep_force_light(0)


# one chunk of K, two, three (no boundary copies anything), five and many; empty rows and a row alone; full chunks, many ops a boundary
@pytest.mark.parametrize("mb,kb,density", [(1, 16, 0.5), (70, 32, 0.2), (64, 48, 0.1), (33, 65, 0.05), (16, 300, 0.02), (64, 100, 0.9)])
@pytest.mark.parametrize("N", [8, 72, 200])
@pytest.mark.parametrize("row_major,c_f32", [(False, False), (True, True), (False, True)])
def test_light_streams_match_the_oracle(smat, cuda, oracle, force, mb, kb, density, N, row_major, c_f32):
    import torch
    A = random_mask_matrix(mb, kb, density, seed=mb + kb)
    M, K = A["M"], A["K"]
    A["b_val"] = np.random.default_rng(1).integers(-2, 3, A["b_val"].size).astype(np.float16).view(np.uint16)
    b = np.random.default_rng(N).integers(-4, 5, (N, K)).astype(np.float16)
    want = oracle.spmm_bcsr(M, N, K, A["b_row_ptr"], A["b_col_idx"], A["b_val"], b.reshape(-1).view(np.uint16), threads=4)
    want = want if c_f32 else want.astype(np.float16)
    vals, rp, ci = (to_dev(torch, A[x], cuda) for x in ("b_val", "b_row_ptr", "b_col_idx"))
    Bd = to_dev(torch, (np.ascontiguousarray(b.T) if row_major else b).reshape(-1).view(np.uint16), cuda)
    nnzb = A["b_col_idx"].size
    for what in (1, -1):  # whole numbers: the sums are exact in fp32 in any order
        force(what)
        plan = smat.Plan(A["b_row_ptr"], M, K, nnzb, N, col_idx_host=A["b_col_idx"], kernel=smat.KERNEL_SWEEP, b_row_major=row_major)
        for _ in range(2):
            C = torch.full((M, N), float("nan"), dtype=torch.float32 if c_f32 else torch.float16, device=cuda)
            smat.spmm(vals, rp, ci, Bd, C, M, N, K, nnzb, plan=plan, c_f32=c_f32, kernel=smat.KERNEL_SWEEP, b_row_major=row_major)
            assert np.array_equal(C.cpu().numpy(), want)
        plan.close()
