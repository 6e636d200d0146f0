"""Device memory of plans: a failing allocation inside attach_values, and what is given back afterwards."""
import ctypes as C

import numpy as np
import pytest

from smat_amd import generators as gen

pytestmark = pytest.mark.gpu


def to_dev(torch, a, cuda):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int16) if a.dtype == np.uint16 else np.ascontiguousarray(a)).to(cuda)


def held(smat):
    """Device blocks that the library has handed out and not taken back."""
    out = (C.c_int64 * 2)()
    smat.lib.smat_internal_alloc_counts(out)
    return out[0] - out[1]


def split_in_steps(seed):
    """Columns with up to 16 nonzeros: in lists of nonzeros, groups of 32 columns that take several steps."""
    rng = np.random.default_rng(seed)
    A = gen.random_bcsr(24, 300, 0.1, seed=seed)
    v = A["b_val"].reshape(-1, 16, 16).copy()
    for p in range(v.shape[0]):
        keep = np.zeros((16, 16), bool)
        for c in rng.choice(16, 3, replace=False):
            keep[rng.choice(16, 16 if p % 9 == 0 else 2, replace=False), c] = True
        v[p][~keep] = 0
    A["b_val"] = v.reshape(-1)
    return A


def test_attach_values_survives_every_failing_allocation(smat, cuda, oracle):
    import torch
    lib = smat.lib
    lib.smat_internal_fail_alloc.argtypes = [C.c_int64]
    lib.smat_internal_compact_list(2)  # the lists with the most allocations
    A = split_in_steps(3)
    M, K, nnzb, N = A["M"], A["K"], A["nnzb"], 72
    B = gen.dense_b(K, N, seed=1)
    vals, rp, ci, Bd = (to_dev(torch, x, cuda) for x in (A["b_val"], A["b_row_ptr"].astype(np.int32), A["b_col_idx"].astype(np.int32), B))
    want = oracle.spmm_bcsr(M, N, K, A["b_row_ptr"], A["b_col_idx"], A["b_val"], B, threads=4)
    plan = smat.Plan(A["b_row_ptr"], M, K, nnzb, N, col_idx_host=A["b_col_idx"])
    before = held(smat)
    failures = 0
    for n in range(200):
        lib.smat_internal_fail_alloc(n)
        try:
            plan.attach_values(vals, rp, ci)
            failed = False
        except smat.SmatError:
            failed = True
        finally:
            lib.smat_internal_fail_alloc(-1)
        C_out = torch.full((M, N), float("nan"), dtype=torch.float16, device=cuda)
        smat.spmm(vals, rp, ci, Bd, C_out, M, N, K, nnzb, plan=plan)
        torch.cuda.synchronize()
        assert oracle.compare(C_out.cpu().numpy().view(np.uint16), want)[0] <= 1e-3, f"after failing allocation {n}"
        if not failed:
            break
        failures += 1
        assert plan.info()["kernel"] == smat.KERNEL_ROWWISE
        assert held(smat) <= before + 1, f"device blocks lost by failing allocation {n}"  # the copy of B may stay for the next attempt
    lib.smat_internal_compact_list(0)
    assert failures >= 15 and plan.info()["kernel"] == smat.KERNEL_COMPACT
    plan.close()


def test_clearing_the_plan_cache_gives_kept_memory_back(smat, cuda):
    import torch
    torch.cuda.synchronize()
    smat.lib.smat_plan_cache_clear()
    free = torch.cuda.mem_get_info()[0]
    big = 256 << 20
    slack = 16 << 20  # the runtime holds chunks of 2 MiB of its own that an allocation may come out of in part
    p = C.c_void_p()
    assert smat.lib.smat_malloc(C.byref(p), big) == 0
    assert torch.cuda.mem_get_info()[0] <= free - big + slack
    assert smat.lib.smat_free(p) == 0
    assert torch.cuda.mem_get_info()[0] <= free - big + slack  # kept
    assert smat.lib.smat_plan_cache_clear() == 0
    assert torch.cuda.mem_get_info()[0] >= free - slack
