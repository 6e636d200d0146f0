"""Light streams of the sweep kernel, checked on the CPU: they are replayed like all streams, an op uses no block of a chunk after the one
being swept, and every wait of a chunk boundary leaves none of the copies of the chunk that is entered under way."""
import ctypes as C

import numpy as np
import pytest

from smat_amd._lib import lib
from tests import test_sweep_plan as plans
from tests.test_sweep_plan import BLOCK_BYTES, COPIES, END_OFF, N_BLOCKS, PAD, TRAMP_BASE, TRAMP_BYTES, WAVES, ZERO_OFF, random_mask_matrix, replay, slot_of
from tests.test_sweep_streams import AHEAD, DEV_MIN_OPS, HEAD, MARKS, TOUCHES

LIGHT_MARKS = 4


@pytest.fixture
def light_plan(monkeypatch):
    class Light:  # the plan builder's hook for smaller row groups, with light streams
        smat_internal_sweep_plan = lib.smat_internal_sweep_plan
        smat_internal_sweep_plan_groups = lib.smat_internal_sweep_plan_light
        smat_host_free = lib.smat_host_free
    monkeypatch.setattr(plans, "lib", Light)
    return plans.sweep_plan


def encode(plan, row_major):
    fn = lib.smat_internal_sweep_encode
    fn.restype = C.c_int
    fn.argtypes = [C.c_void_p, C.c_int64, C.c_void_p, C.c_void_p, C.c_int, C.c_void_p]
    n_rg = plan["rg_chunk_ptr"].size - 1
    out = np.zeros((plan["n_entries"] + HEAD * WAVES * n_rg + PAD, 4), np.uint32)
    assert fn(plan["rg_chunk_ptr"].ctypes.data, n_rg, plan["op_ptr"].ctypes.data, plan["ops"].ctypes.data, row_major + 2, out.ctypes.data) == 0
    return out


def check_chunks(plan):
    for s in range(plan["op_ptr"].size - 1):
        cur = 0
        for w0, w1, w2, w3 in plan["ops"][plan["op_ptr"][s]:plan["op_ptr"][s + 1]].astype(np.int64):
            if w3 == END_OFF:
                continue
            opens = w3 >= TRAMP_BASE
            cur += opens
            for off in (int(w1), int(w1 + np.int32(np.uint32(w2)))):
                if off != ZERO_OFF:  # chunks cur - 1 and cur; the first op of a chunk reads before its barrier: cur - 1
                    assert slot_of(off)[0] in ({(cur - 1) % 4} if opens else {cur % 4, (cur - 1) % 4})


def check_waits(plan, row_major):
    dev = encode(plan, row_major)
    block_bytes = 192 if row_major else BLOCK_BYTES
    tramp_base = N_BLOCKS * block_bytes
    mark_off = tramp_base + MARKS * N_BLOCKS * TRAMP_BYTES
    light_base = mark_off + 512 + 64
    seen = set()
    for s in range(plan["op_ptr"].size - 1):
        a, b = plan["op_ptr"][s], plan["op_ptr"][s + 1]
        if a == b:
            continue
        out = dev[a + HEAD * (s + 1):b + HEAD * (s + 1), 3].astype(np.int64)
        n_chunks = int(plan["rg_chunk_ptr"][s // WAVES + 1] - plan["rg_chunk_ptr"][s // WAVES])
        issued = [("copy", c) for c in range(min(3, n_chunks)) for _ in range(COPIES)]
        issued += [("a", k) for k in range(AHEAD)] + [("touch", 0)] * TOUCHES
        cur = 0
        for i, w3 in enumerate(int(x) for x in out):
            if w3 == mark_off + 512:
                break
            k = w3 // block_bytes
            if w3 >= tramp_base:
                light = w3 >= light_base
                m, k = divmod((w3 - (light_base if light else tramp_base)) // TRAMP_BYTES, N_BLOCKS)
                assert m < (LIGHT_MARKS if light else MARKS)
                allowed = COPIES + 2 * DEV_MIN_OPS + m if light else DEV_MIN_OPS + m
                cur += 1
                assert ("copy", cur) not in issued[len(issued) - allowed:]
                if cur + 2 < n_chunks:
                    issued += [("copy", cur + 2)] * COPIES
                seen.add((light, m))
            assert k // 16 == i % 8
            issued.append(("a", i + AHEAD))
            assert ("a", i) not in issued[len(issued) - AHEAD - COPIES * (k % 2):]
        assert cur == n_chunks - 1
    return seen


CASES = [(64, 64, 0.10, 1, 16), (70, 40, 0.30, 2, 32), (16, 300, 0.03, 3, 16), (50, 20, 0.02, 4, 48), (64, 16, 0.5, 5, 63), (3, 2, 1.0, 6, 16), (5, 33, 0.2, 8, 16), (130, 33, 0.0005, 7, 32), (40, 120, 0.3, 9, 40)]


@pytest.mark.parametrize("mb,kb,density,seed,group_rows", CASES)
def test_light_streams_give_a_times_b(light_plan, mb, kb, density, seed, group_rows):
    A = random_mask_matrix(mb, kb, density, seed)
    plan = light_plan(A["b_row_ptr"], A["b_col_idx"], A["M"], A["K"], group_rows=group_rows)
    B = np.random.default_rng(seed).standard_normal((A["K"], 3))
    blocks = A["b_val"].view(np.float16).astype(np.float64).reshape(-1, 16, 16)
    want = np.zeros((A["M"], 3))
    for i in range(A["M"] // 16):
        for q in range(A["b_row_ptr"][i], A["b_row_ptr"][i + 1]):
            want[16 * i:16 * i + 16] += blocks[q] @ B[A["b_col_idx"][q]:A["b_col_idx"][q] + 16]
    assert np.allclose(replay(plan, A, B, group_rows=group_rows), want, rtol=1e-9, atol=1e-9)  # fp64 sums of a few thousand products
    check_chunks(plan)
    for row_major in (0, 1):
        check_waits(plan, row_major)


def test_light_streams_use_every_wait(light_plan):
    seen = set()
    for mb, kb, density, seed, group_rows in CASES:
        A = random_mask_matrix(mb, kb, density, seed)
        seen |= check_waits(light_plan(A["b_row_ptr"], A["b_col_idx"], A["M"], A["K"], group_rows=group_rows), 0)
    assert {(True, m) for m in range(LIGHT_MARKS)} <= seen and {m for light, m in seen if not light} >= {0, 2}
