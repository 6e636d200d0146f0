"""Paths that only a large B takes: entries staged in LDS beside row addresses of 64 bits, and a row-major B of half of the memory-side
cache and more on its way to the kernels that read column-major B."""
import numpy as np
import pytest

from smat_amd import generators as gen
from tests.test_gpu_compact_entries import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per_column", [1, 3])  # 64 or 128 entries asked for a step
@pytest.mark.parametrize("row_major,c_f32", [(False, False), (True, True)])
def test_staged_entries_with_wide_row_addresses(smat, cuda, oracle, per_column, row_major, c_f32):
    import torch
    K, N, mb = (1 << 24) + 160, 8, 5
    rng = np.random.default_rng(per_column)
    kb = K // 16
    # 1 to 600 blocks of four nonzero columns a block row, in the first and the last block columns and all between: 1 to 80 steps
    per_row = [np.unique(np.concatenate([rng.integers(0, kb, n), [0, kb - 1]])) for n in (1, 600, 0, 70, 250)]
    rp = np.concatenate([[0], np.cumsum([len(c) for c in per_row])]).astype(np.int32)
    ci = (np.concatenate(per_row) * 16).astype(np.int32)
    v = np.zeros((len(ci), 16, 16), np.float16)
    for p in range(len(ci)):
        for c in rng.choice(16, 4, replace=False):
            v[p, rng.choice(16, per_column, replace=False), c] = rng.normal(size=per_column)
    M, nnzb, val = mb * 16, len(ci), v.view(np.uint16).reshape(-1)
    B = torch.randn(K * N, generator=torch.Generator("cuda").manual_seed(3), device=cuda, dtype=torch.float16)
    used = np.unique(ci).astype(np.int64)
    rows = (torch.as_tensor(used)[:, None] + torch.arange(16)).reshape(-1).to(cuda)
    small = B.view(K, N)[rows].t() if row_major else B.view(N, K)[:, rows]  # the rows of B that are used, column-major
    small = np.ascontiguousarray(small.cpu().numpy().view(np.uint16)).reshape(-1)
    A = {"M": M, "b_row_ptr": rp, "b_col_idx": (np.searchsorted(used, ci) * 16).astype(np.int32), "b_val": val}
    want = oracle.spmm_bcsr(M, N, len(used) * 16, rp, A["b_col_idx"], val, small, threads=4)
    vals, rpd, cid = (to_dev(torch, x, cuda) for x in (val, rp, ci))
    out = []
    try:
        smat.lib.smat_internal_compact_list(2)
        plan = smat.Plan(rp, M, K, nnzb, N, col_idx_host=ci, kernel=smat.KERNEL_COMPACT, b_row_major=row_major)
        plan.attach_values(vals, rpd, cid)
        for staged in (1, 2):
            smat.lib.smat_internal_compact_staged(staged)
            C = torch.full((M, N), float("nan"), dtype=torch.float32 if c_f32 else torch.float16, device=cuda)
            smat.spmm(vals, rpd, cid, B, C, M, N, K, nnzb, plan=plan, kernel=smat.KERNEL_COMPACT, c_f32=c_f32, b_row_major=row_major)
            torch.cuda.synchronize()
            out.append(C.cpu().numpy())
    finally:
        smat.lib.smat_internal_compact_list(0)
        smat.lib.smat_internal_compact_staged(0)
    plan.close()
    assert np.array_equal(out[0], out[1])
    if c_f32:
        oracle.assert_fp32_close(out[0], want, N, len(used) * 16, A, small)
    else:
        assert oracle.compare(out[0].view(np.uint16), want)[0] <= 1e-3


# tiles of 64 x 64 cut off in K, in N, in both, in neither; N = 1024 is exactly 128 MiB
@pytest.mark.parametrize("K,N", [(65536, 1024), (65552, 1032), (65584, 1088), (65536, 1080)])
@pytest.mark.parametrize("kernel", ["ROWWISE_DIRECT", "ROWWISE_PACKED"])
def test_row_major_b_of_128_mib_through_the_row_wise_kernel(smat, cuda, oracle, K, N, kernel):
    import torch
    assert K * N * 2 >= 128 << 20
    rng = np.random.default_rng(N)
    lengths = [0, 1, 2, 40, 7, 129]
    cols = [np.sort(rng.choice(K // 16, n, replace=False)) for n in lengths]
    cols[3] = np.unique(np.concatenate([cols[3], [0, K // 16 - 1]]))
    rp = np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.int32)
    ci = (np.concatenate(cols) * 16).astype(np.int32)
    M, nnzb = 16 * len(lengths), len(ci)
    val = rng.normal(size=nnzb * 256).astype(np.float16).view(np.uint16)
    B = gen.dense_b(K, N, seed=N)
    want = oracle.spmm_bcsr(M, N, K, rp, ci, val, B, threads=4)
    vals, rpd, cid, Bd = (to_dev(torch, x, cuda) for x in (val, rp, ci, B))
    which = getattr(smat, "KERNEL_" + kernel)
    out = []
    for row_major in (True, False):
        plan = smat.Plan(rp, M, K, nnzb, N, col_idx_host=ci, kernel=which, b_row_major=row_major)
        b = Bd.view(N, K).t().contiguous() if row_major else Bd
        C = torch.full((M, N), float("nan"), dtype=torch.float16, device=cuda)
        smat.spmm(vals, rpd, cid, b, C, M, N, K, nnzb, plan=plan, kernel=which, b_row_major=row_major)
        torch.cuda.synchronize()
        out.append(C.cpu().numpy())
    assert np.array_equal(out[0], out[1])
    assert oracle.compare(out[0].view(np.uint16), want)[0] <= 1e-3
