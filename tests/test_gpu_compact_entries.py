"""The compact kernel on lists of single nonzeros: steps with more entries than are asked for at once, items put together
into tasks, empty block rows between and around them."""
import numpy as np
import pytest

from smat_amd import generators as gen

pytestmark = pytest.mark.gpu


def to_dev(torch, a, cuda):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int16) if a.dtype == np.uint16 else np.ascontiguousarray(a)).to(cuda)


@pytest.fixture
def lists(smat):
    """lists(1): plans list whole columns; lists(2): nonzeros one by one (how many wavefronts and nonzeros decides otherwise)."""
    yield smat.lib.smat_internal_compact_list
    smat.lib.smat_internal_compact_list(0)


def matrix(fill, seed):
    """Block rows of 0 .. 70 blocks, fill nonzeros per nonzero column on average:
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
def test_lists_of_nonzeros_match_the_oracle(smat, cuda, oracle, lists, fill, N, c_f32, row_major):
    import torch
    lists(2)
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
        if c_f32:
            oracle.assert_fp32_close(C.cpu().numpy(), want, N, K, A, B)
        else:
            assert oracle.compare(C.cpu().numpy().view(np.uint16), want)[0] <= 1e-3


# block rows of up to 260 steps: around what one load of entry ranges covers (64 steps), and around two
STEPS = [1, 7, 60, 61, 62, 63, 64, 65, 66, 71, 126, 127, 128, 129, 130, 131, 191, 193, 260]


@pytest.mark.parametrize("fill", [1, 2])
@pytest.mark.parametrize("what,K", [(2, 8448), (1, 8448), (1, 4080)])
@pytest.mark.parametrize("N", [64, 200])
@pytest.mark.parametrize("n_hint", [0, 4096])
def test_long_even_block_rows(smat, cuda, oracle, lists, fill, what, K, N, n_hint):
    """Lists of nonzeros and of whole columns.  A plan for a wide product has wavefronts enough and leaves the
    rows whole, one for N columns splits them."""
    import torch
    lists(what)
    rng = np.random.default_rng(fill)
    lengths = [min(2 * s, K // 16) for s in STEPS]  # blocks with all their columns: two a step
    A = gen.random_bcsr(len(lengths), K // 16, 0.0, seed=fill, row_lengths=lengths)
    M, nnzb = A["M"], A["nnzb"]
    v = A["b_val"].reshape(-1, 16, 16).copy()
    keep = np.zeros((nnzb, 16, 16), bool)
    for _ in range(fill):
        keep[np.arange(nnzb)[:, None], rng.integers(0, 16, (nnzb, 16)), np.arange(16)[None, :]] = True
    v[~keep] = 0
    A["b_val"] = v.reshape(-1)
    B = gen.dense_b(K, N, seed=N)
    vals, rp, ci, Bd = (to_dev(torch, x, cuda) for x in (A["b_val"], A["b_row_ptr"].astype(np.int32), A["b_col_idx"].astype(np.int32), B))
    want = oracle.spmm_bcsr(M, N, K, A["b_row_ptr"], A["b_col_idx"], A["b_val"], B, threads=4)
    for tq in (1, 2):
        smat.lib.smat_internal_compact_panel(tq)
        try:
            C = torch.full((M, N), float("nan"), dtype=torch.float32, device=cuda)
            plan = smat.Plan(A["b_row_ptr"], M, K, nnzb, n_hint or N, col_idx_host=A["b_col_idx"], kernel=5)
            plan.attach_values(vals, rp, ci)
            split = smat.lib.smat_internal_compact_split_rows(plan.handle)
            assert split == 0 if n_hint else split == sum(min(s, K // 32) > 56 for s in STEPS)
            smat.spmm(vals, rp, ci, Bd, C, M, N, K, nnzb, plan=plan, kernel=5, c_f32=True)
            torch.cuda.synchronize()
        finally:
            smat.lib.smat_internal_compact_panel(0)
        oracle.assert_fp32_close(C.cpu().numpy(), want, N, K, A, B)


# copies of B of 4 GiB and more, K above 2^24: row addresses in 64 bits
@pytest.mark.parametrize("what", [1, 2])
@pytest.mark.parametrize("K,N,row_major", [((1 << 24) + 160, 136, True), ((1 << 24) + 160, 8, False), (1 << 20, 2056, True)])
@pytest.mark.parametrize("c_f32", [False, True])
def test_wide_row_addresses_match_the_oracle(smat, cuda, oracle, lists, what, K, N, row_major, c_f32):
    import torch
    lists(what)
    rng = np.random.default_rng(N)
    mb, kb = 6, K // 16
    # block columns all over K, the first and the last among them, and around 2^32 bytes of B
    edge = min(kb - 2, (1 << 32) // (N * 2) // 16)
    per_row = [np.unique(np.concatenate([rng.integers(0, kb, n), [0, edge - 1, edge, edge + 1, kb - 1]])) for n in (3, 20, 60, 0, 40, 9)]
    rp = np.concatenate([[0], np.cumsum([len(c) for c in per_row])]).astype(np.int32)
    ci = (np.concatenate(per_row) * 16).astype(np.int32)
    v = np.zeros((len(ci), 16, 16), np.float16)
    for p in range(len(ci)):
        for c in rng.choice(16, 3, replace=False):
            v[p, rng.choice(16, 2, replace=False), c] = rng.normal(size=2)
    M, nnzb, val = mb * 16, len(ci), v.view(np.uint16).reshape(-1)
    g = torch.Generator("cuda").manual_seed(3)
    B = torch.randn(K * N, generator=g, device=cuda, dtype=torch.float16) if K * N < 1 << 31 else \
        torch.cat([torch.randn(K // 2 * N, generator=g, device=cuda, dtype=torch.float16) for _ in range(2)])
    used = np.unique(ci).astype(np.int64)
    rows = (torch.as_tensor(used)[:, None] + torch.arange(16)).reshape(-1).to(cuda)
    small = B.view(K, N)[rows].t() if row_major else B.view(N, K)[:, rows]  # the rows of B that are used, column-major
    small = np.ascontiguousarray(small.cpu().numpy().view(np.uint16)).reshape(-1)
    A = {"M": M, "b_row_ptr": rp, "b_col_idx": (np.searchsorted(used, ci) * 16).astype(np.int32), "b_val": val}
    want = oracle.spmm_bcsr(M, N, len(used) * 16, rp, A["b_col_idx"], val, small, threads=4)
    vals, rpd, cid = (to_dev(torch, x, cuda) for x in (val, rp, ci))
    C = torch.full((M, N), float("nan"), dtype=torch.float32 if c_f32 else torch.float16, device=cuda)
    plan = smat.Plan(rp, M, K, nnzb, N, col_idx_host=ci, kernel=5, b_row_major=row_major)
    plan.attach_values(vals, rpd, cid)
    smat.spmm(vals, rpd, cid, B, C, M, N, K, nnzb, plan=plan, kernel=5, c_f32=c_f32, b_row_major=row_major)
    torch.cuda.synchronize()
    plan.close()
    if c_f32:
        oracle.assert_fp32_close(C.cpu().numpy(), want, N, len(used) * 16, A, small)
    else:
        assert oracle.compare(C.cpu().numpy().view(np.uint16), want)[0] <= 1e-3
