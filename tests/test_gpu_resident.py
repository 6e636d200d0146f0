"""Products with whole columns of B in LDS: plans with values for matrices of few nonzeros a block."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def to_dev(torch, a, cuda):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int16) if a.dtype == np.uint16 else np.ascontiguousarray(a)).to(cuda)


@pytest.fixture
def force(smat):
    smat.lib.smat_internal_resident_force.argtypes = [ctypes.c_int, ctypes.c_int]
    smat.lib.smat_internal_window_force(-1, 0)
    yield smat.lib.smat_internal_resident_force
    smat.lib.smat_internal_resident_force(0, 0)
    smat.lib.smat_internal_window_force(0, 0)


def scattered(smat, lengths, K, seed):
    """Rows of so many nonzeros, small whole numbers (every order of the sums gives the same bits), the last column among them."""
    rng = np.random.default_rng(seed)
    rp, ci = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32), []
    for n in lengths:
        c = rng.choice(K, n, replace=False)
        if n and K - 1 not in c:
            c[0] = K - 1
        ci.append(np.sort(c))
    ci = np.concatenate(ci).astype(np.int32)
    v = rng.choice([-3, -2, -1, 1, 2, 3], len(ci)).astype(np.float16).view(np.uint16)
    return smat.csr_to_bcsr(len(lengths), K, rp, ci, v)


def plan_of(smat, A, d, N):
    plan = smat.Plan(A.row_ptr, A.M, A.K, len(A.col_idx), N, col_idx_host=A.col_idx)
    plan.attach_values(*d[:3])
    return plan


# rows of no, one, three, four and five nonzeros (a row's number and three to a lane's first load), fewer rows than a slice of 64 and not a
# whole number of them; K up to the most that LDS holds of 8, 4 and 2 columns
@pytest.mark.parametrize("M,K", [(16, 32), (48, 96), (208, 10224), (1040, 20464), (2064, 40944)])
@pytest.mark.parametrize("columns,shares,N", [(2, 1, 8), (2, 3, 24), (4, 1, 16), (4, 5, 136), (8, 1, 8), (8, 2, 264)])
def test_resident_columns_match_the_oracle(smat, cuda, oracle, force, M, K, columns, shares, N):
    import torch
    if (K + 1) * 2 * columns > 160 * 1024:
        pytest.skip("columns longer than LDS")
    lengths = np.random.default_rng(M).choice([0, 1, 3, 4, 5, 11] if K > 32 else [0, 1], M)
    lengths[0], lengths[-1] = 0, 7
    A = scattered(smat, lengths, K, seed=M)
    B = np.random.default_rng(N).integers(-4, 5, K * N).astype(np.float16).view(np.uint16)
    d = [to_dev(torch, x, cuda) for x in (A.val, A.row_ptr, A.col_idx, B)]
    want = oracle.spmm_bcsr(M, N, K, A.row_ptr, A.col_idx, A.val, B, threads=8)
    force(columns, shares)
    plan = plan_of(smat, A, d, N)
    assert plan.info()["kernel"] == smat.KERNEL_COMPACT
    assert smat.lib.smat_internal_plan_resident(plan.handle) == 1
    d[0].zero_()  # the values are the ones attached
    for n in {N, max(8, N * 3 // 4 // 8 * 8)}:
        for c_f32 in (False, True):
            for kernel in (smat.KERNEL_AUTO, smat.KERNEL_COMPACT):
                C = torch.full((M, n), float("nan"), dtype=torch.float32 if c_f32 else torch.float16, device=cuda)
                smat.spmm(d[0], d[1], d[2], d[3][:K * n], C, M, n, K, len(A.col_idx), plan=plan, c_f32=c_f32, kernel=kernel)
                assert np.array_equal(C.cpu().numpy().astype(np.float32), want[:, :n].astype(np.float32 if c_f32 else np.float16).astype(np.float32))
    plan.close()


@pytest.mark.parametrize("longest,taken", [(4096, 1), (4097, 0)])
def test_rows_longer_than_a_list_stay_with_the_compact_kernel(smat, cuda, force, longest, taken):
    import torch
    M, K, N = 1040, 32768, 1000
    lengths = np.full(M, 900)
    lengths[77] = longest
    A = scattered(smat, lengths, K, seed=longest)
    B = np.random.default_rng(N).integers(-1, 2, K * N).astype(np.float16)
    d = [to_dev(torch, x, cuda) for x in (A.val, A.row_ptr, A.col_idx, B.view(np.uint16))]
    force(2, 2)
    plan = plan_of(smat, A, d, N)
    assert plan.info()["kernel"] == smat.KERNEL_COMPACT
    assert smat.lib.smat_internal_plan_resident(plan.handle) == taken
    C = torch.empty((M, N), dtype=torch.float32, device=cuda)
    smat.spmm(d[0], d[1], d[2], d[3], C, M, N, K, len(A.col_idx), plan=plan, c_f32=True)
    full = np.zeros((M, K), np.float32)
    blocks = A.val.view(np.float16).reshape(-1, 16, 16)
    for i in range(M // 16):
        for q in range(A.row_ptr[i], A.row_ptr[i + 1]):
            full[16 * i:16 * i + 16, A.col_idx[q]:A.col_idx[q] + 16] = blocks[q]
    want = torch.from_numpy(full).to(cuda) @ torch.from_numpy(B.astype(np.float32).reshape(N, K)).to(cuda).T.contiguous()  # whole numbers: exact
    assert torch.equal(C, want)
    plan.close()


# rows shared by 2, 4, 8 and 64 lanes, at the borders between them, in block rows that the compact kernel's list splits and in ones that it leaves whole
@pytest.mark.parametrize("heavy", [[65], [64, 65, 128, 129, 255, 257], [2049, 4000, 66, 1024]])
@pytest.mark.parametrize("columns,shares,N", [(2, 1, 24), (4, 3, 40), (8, 1, 8)])
def test_long_rows_are_shared_by_lanes(smat, cuda, oracle, force, heavy, columns, shares, N):
    import torch
    M, K = 1616, 10224
    lengths = np.random.default_rng(len(heavy)).choice([0, 1, 3, 9], M)
    lengths[20:20 + 17 * len(heavy):17] = heavy  # one in a block row
    A = scattered(smat, lengths, K, seed=heavy[0])
    B = np.random.default_rng(N).integers(-2, 3, K * N).astype(np.float16).view(np.uint16)
    d = [to_dev(torch, x, cuda) for x in (A.val, A.row_ptr, A.col_idx, B)]
    want = oracle.spmm_bcsr(M, N, K, A.row_ptr, A.col_idx, A.val, B, threads=8)
    force(columns, shares)
    plan = plan_of(smat, A, d, N)
    assert plan.info()["kernel"] == smat.KERNEL_COMPACT and smat.lib.smat_internal_plan_resident(plan.handle) == 1
    for c_f32 in (False, True):
        C = torch.full((M, N), float("nan"), dtype=torch.float32 if c_f32 else torch.float16, device=cuda)
        smat.spmm(d[0], d[1], d[2], d[3], C, M, N, K, len(A.col_idx), plan=plan, c_f32=c_f32)
        assert np.array_equal(C.cpu().numpy().astype(np.float32), want.astype(np.float32 if c_f32 else np.float16).astype(np.float32))
    plan.close()


def test_sums_are_no_further_from_the_exact_ones(smat, cuda, force):
    """fp32 sums of 4 to 60 products against fp64: the root mean square error is that of the compact kernel or less."""
    import torch
    for n in (4, 17, 60):
        rng = np.random.default_rng(n)
        M, K, N = 2048, 4096, 64
        A = scattered(smat, np.full(M, n), K, seed=n)
        blocks = A.val.view(np.float16).reshape(-1, 16, 16)
        blocks[blocks != 0] = rng.standard_normal(np.count_nonzero(blocks)).astype(np.float16)
        B = rng.standard_normal((N, K)).astype(np.float16)
        d = [to_dev(torch, x, cuda) for x in (A.val, A.row_ptr, A.col_idx, B.reshape(-1).view(np.uint16))]
        full = np.zeros((M, K))
        for i in range(M // 16):
            for q in range(A.row_ptr[i], A.row_ptr[i + 1]):
                full[16 * i:16 * i + 16, A.col_idx[q]:A.col_idx[q] + 16] = blocks[q]
        want = full @ B.astype(np.float64).T
        rms = {}
        for columns in (-1, 4):
            force(columns, 0)
            plan = plan_of(smat, A, d, N)
            C = torch.empty((M, N), dtype=torch.float32, device=cuda)
            smat.spmm(d[0], d[1], d[2], d[3], C, M, N, K, len(A.col_idx), plan=plan, c_f32=True)
            rms[columns] = np.sqrt(np.mean((C.cpu().numpy() - want) ** 2))
            plan.close()
        assert rms[4] <= 1.02 * rms[-1], rms


def test_which_products_hold_columns(smat, cuda, force):
    import torch

    def takes(M, K, per_row, N):
        A = scattered(smat, np.full(M, per_row), K, seed=M)
        d = [to_dev(torch, x, cuda) for x in (A.val, A.row_ptr, A.col_idx)]
        plan = plan_of(smat, A, d, N)
        r = smat.lib.smat_internal_plan_resident(plan.handle)
        plan.close()
        return r

    assert takes(2048, 2048, 8, 64) == 1
    assert takes(4096, 16384, 16, 256) == 1
    assert takes(1024, 65536, 8, 64) == 0


def test_calls_of_the_plan_s_width_do_not_work_out_their_launch(smat, cuda):
    import torch
    smat.lib.smat_internal_resident_searches.restype = ctypes.c_int64
    M, K, N = 2048, 2048, 64
    A = scattered(smat, np.full(M, 8), K, seed=M)
    d = [to_dev(torch, x, cuda) for x in (A.val, A.row_ptr, A.col_idx, np.zeros(K * N, np.uint16))]
    plan = plan_of(smat, A, d, N)
    assert smat.lib.smat_internal_plan_resident(plan.handle) == 1
    C = torch.empty((M, N), dtype=torch.float32, device=cuda)
    searches = []
    for n in (N, 40):
        before = smat.lib.smat_internal_resident_searches()
        for c_f32 in (False, True):
            smat.spmm(*d, C, M, n, K, len(A.col_idx), plan=plan, c_f32=c_f32)
        searches.append(smat.lib.smat_internal_resident_searches() - before)
    assert searches == [0, 2]
    torch.cuda.synchronize()
    plan.close()


@pytest.mark.parametrize("windows", [False, True])
def test_captured_launches_replay(smat, cuda, oracle, force, windows):
    """Columns in LDS and windows of listed nonzeros in a graph, replayed between launches outside of it, B changing from replay to replay."""
    import torch
    force(4 if not windows else -1, 0)
    smat.lib.smat_internal_window_force(8 if windows else -1, 2 if windows else 0)
    M, K, N = 2048, 2048, 64
    rng = np.random.default_rng(3)
    if windows:  # every row two nonzeros near the diagonal
        rp = np.arange(M + 1, dtype=np.int32) * 2
        lo = np.clip(np.arange(M) - 20, 0, K - 41)
        ci = np.sort(lo[:, None] + np.stack([rng.integers(0, 20, M), rng.integers(20, 41, M)], 1), 1).astype(np.int32).reshape(-1)
        A = smat.csr_to_bcsr(M, K, rp, ci, np.ones(2 * M, np.float16).view(np.uint16))
    else:
        A = scattered(smat, np.full(M, 5), K, seed=8)
    Bs = [rng.integers(-4, 5, K * N).astype(np.float16).view(np.uint16) for _ in range(4)]
    d = [to_dev(torch, x, cuda) for x in (A.val, A.row_ptr, A.col_idx, Bs[0])]
    plan = plan_of(smat, A, d, N)
    assert plan.info()["kernel"] == smat.KERNEL_COMPACT
    assert smat.lib.smat_internal_plan_resident(plan.handle) == (not windows) and (smat.lib.smat_internal_plan_window_rows(plan.handle) == 8) == windows
    C = torch.zeros((M, N), dtype=torch.float16, device=cuda)
    other = torch.zeros_like(C)
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=stream):
        smat.spmm(d[0], d[1], d[2], d[3], C, M, N, K, len(A.col_idx), plan=plan, stream=torch.cuda.current_stream().cuda_stream)
    for B in Bs:
        d[3].copy_(to_dev(torch, B, cuda))
        C.fill_(float("nan"))
        graph.replay()
        smat.spmm(d[0], d[1], d[2], d[3], other, M, N, K, len(A.col_idx), plan=plan)
        torch.cuda.synchronize()
        want = oracle.spmm_bcsr(M, N, K, A.row_ptr, A.col_idx, A.val, B, threads=4).astype(np.float16)
        assert np.array_equal(C.cpu().numpy(), want) and torch.equal(C, other)
    plan.close()
