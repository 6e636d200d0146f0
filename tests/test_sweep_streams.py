"""Streams of the sweep kernel as it runs them (checked on the CPU): the plan's entries with the A operands asked for seven
positions ahead.  What every wait of the kernel allows to be under way is compared with the order in which the vector
memory operations are issued: nothing that a position needs may be among the operations that its wait leaves."""
import ctypes as C

import numpy as np
import pytest

from smat_amd import generators as gen
from smat_amd._lib import lib
from tests.test_sweep_plan import BLOCK_BYTES, COPIES, END_OFF, N_BLOCKS, PAD, TRAMP_BASE, TRAMP_BYTES, WAVES, ZERO_OFF, random_mask_matrix, sweep_plan

AHEAD, HEAD, DEV_MIN_OPS, MARKS, TOUCHES = 7, 2, 2, 6, 2


def encode(plan, row_major):
    fn = lib.smat_internal_sweep_encode
    fn.restype = C.c_int
    fn.argtypes = [C.c_void_p, C.c_int64, C.c_void_p, C.c_void_p, C.c_int, C.c_void_p]
    n_rg = plan["rg_chunk_ptr"].size - 1
    out = np.zeros((plan["n_entries"] + HEAD * WAVES * n_rg + PAD, 4), np.uint32)
    assert fn(plan["rg_chunk_ptr"].ctypes.data, n_rg, plan["op_ptr"].ctypes.data, plan["ops"].ctypes.data, row_major, out.ctypes.data) == 0
    return out


def lds_offset(off, row_major):
    """of a block in a stage of [8-slab group][column][slot] -> in one of [slab][k][column]; the region of zeros stays"""
    return np.where(off == ZERO_OFF, off, (off // 16384 * 8 + off % 16384 // 32) * 2048) if row_major else off


def check(plan, row_major):
    dev = encode(plan, row_major)
    block_bytes = 192 if row_major else BLOCK_BYTES
    tramp_base = N_BLOCKS * block_bytes
    mark_off = tramp_base + MARKS * N_BLOCKS * TRAMP_BYTES
    end_off = mark_off + 512
    seen = set()
    for s in range(plan["op_ptr"].size - 1):
        a, b = plan["op_ptr"][s], plan["op_ptr"][s + 1]
        ops = plan["ops"][a:b].astype(np.int64)
        head = dev[a + HEAD * s:a + HEAD * (s + 1)].astype(np.int64).reshape(-1)
        out = dev[a + HEAD * (s + 1):b + HEAD * (s + 1)].astype(np.int64)
        if a == b:
            continue
        assert ops[-1, 3] == END_OFF
        # what is left of the plan's entries: all but fillers that do not open a chunk, two of a chunk at least
        opens = ops[:-1, 3] >= TRAMP_BASE
        chunk = np.cumsum(opens)
        first = opens | (np.arange(opens.size) == 0)
        filler = (ops[:-1, 1] == ZERO_OFF) & (ops[:-1, 2] == 0)
        keep = first | ~filler
        for c in range(chunk[-1] + 1):
            spare = np.flatnonzero((chunk == c) & ~keep)
            keep[spare[:max(0, DEV_MIN_OPS - int(keep[chunk == c].sum()))]] = True
        assert np.all(np.bincount(chunk[keep]) >= DEV_MIN_OPS)
        seen.add(("dropped", bool((~keep).any())))
        ops = ops[:-1][keep]
        n = ops.shape[0]
        assert np.all(out[n:] == (0, ZERO_OFF, 0, end_off))
        a_of = np.concatenate([ops[:, 0], np.zeros(AHEAD, np.int64)])
        assert np.array_equal(head[:AHEAD], a_of[:AHEAD]) and not head[AHEAD:].any()
        assert np.array_equal(out[:n, 0], a_of[AHEAD - 1:AHEAD - 1 + n])
        delta = ops[:, 2].astype(np.uint32).view(np.int32), out[:n, 2].astype(np.uint32).view(np.int32)
        assert np.array_equal(out[:n, 1], lds_offset(ops[:, 1], row_major))
        assert np.array_equal(out[:n, 1] + delta[1], lds_offset(ops[:, 1] + delta[0], row_major))
        n_chunks = int(plan["rg_chunk_ptr"][s // WAVES + 1] - plan["rg_chunk_ptr"][s // WAVES])
        # issue order: copies of chunks 0..2, the first A operands, the touches, then per position [copies of a boundary], A
        issued = [("copy", c) for c in range(min(3, n_chunks)) for _ in range(COPIES)]
        issued += [("a", k) for k in range(AHEAD)] + [("touch", 0)] * TOUCHES
        cur = 0

        def landed(what, allowed):
            return what not in issued[len(issued) - allowed:]
        for i in range(n):
            w3, plan_w3 = int(out[i, 3]), int(ops[i, 3])
            if plan_w3 >= TRAMP_BASE:
                m, k = divmod((w3 - tramp_base) // TRAMP_BYTES, N_BLOCKS)
                assert tramp_base <= w3 < mark_off and (w3 - tramp_base) % TRAMP_BYTES == 0
                plan_k = (plan_w3 - TRAMP_BASE) // TRAMP_BYTES
                assert landed(("copy", cur + 2), DEV_MIN_OPS + m) or cur + 2 >= n_chunks
                cur += 1
                if cur + 2 < n_chunks:
                    issued += [("copy", cur + 2)] * COPIES
                seen.add(("mark", m))
            else:
                assert w3 < tramp_base and w3 % block_bytes == 0
                k, plan_k = w3 // block_bytes, plan_w3 // BLOCK_BYTES
            assert k // 16 == i % 8 and k // 2 % 8 == plan_k // 2 % 8  # stream position and block row
            issued.append(("a", i + AHEAD))
            assert landed(("a", i), AHEAD + COPIES * (k % 2))
            seen.add(("op", k % 2))
        assert cur == n_chunks - 1
    tail = dev[dev.shape[0] - PAD:]
    assert np.all(tail == np.array([0, ZERO_OFF, 0, end_off], np.uint32))
    return seen


@pytest.mark.parametrize("row_major", [0, 1])
@pytest.mark.parametrize("mb,kb,density,seed,group_rows", [(64, 64, 0.10, 1, 64), (70, 40, 0.30, 2, 64), (16, 300, 0.03, 3, 16), (50, 20, 0.02, 4, 32),
                                                           (64, 16, 0.5, 5, 64), (3, 2, 1.0, 6, 16), (130, 33, 0.0005, 7, 64)])
def test_waits_of_the_device_streams(mb, kb, density, seed, group_rows, row_major):
    A = random_mask_matrix(mb, kb, density, seed)
    check(sweep_plan(A["b_row_ptr"], A["b_col_idx"], A["M"], A["K"], group_rows=group_rows), row_major)


def test_device_streams_use_every_wait():
    A = gen.block_pruned(4096, 0.10, 0.02)
    plan = sweep_plan(A["b_row_ptr"], A["b_col_idx"], A["M"], A["K"])
    seen = check(plan, 0)
    A = random_mask_matrix(64, 200, 0.03, 1)
    seen |= check(sweep_plan(A["b_row_ptr"], A["b_col_idx"], A["M"], A["K"], group_rows=32), 0)
    assert seen == {("op", 0), ("op", 1), ("dropped", False), ("dropped", True)} | {("mark", m) for m in range(MARKS)}
