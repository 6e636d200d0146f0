"""The work that a user of this framework has it do, as cases that can be timed.

The framework multiplies sparse fp16 matrices in 16x16 blocks with dense fp16 ones.  A program that uses it reorders a
matrix (offline, if at all), blocks it, makes a plan and then multiplies with the plan again and again; or it calls the
drop-in entry point, which plans by itself.  Most cases are therefore one product each; one is the way from a new
matrix to its first product and one the reorder.  The matrices are those of the benchmark and of the tests (band,
Erdos-Renyi, R-MAT, 27-point stencil, block-pruned weights, weights with stray nonzeros), drawn on the GPU.

  listed()             the cases
  draw(rng)            one more of the same ranges
  prepare(case, seed)  what the program has before the call
  run(state)           one pass
  work(case)           bytes and operations that a pass cannot do without
  tolerance(case)      how far another correct result may be off

Fields of a case:
  task      "spmm" (one product), "setup" (CSR on the device -> blocks -> plan -> first product) or "reorder"
  matrix    "band" (m, bandwidth), "er" (m, k, per_row), "rmat" (scale, degree), "stencil" (nx, ny, nz),
            "pruned" (m, k, keep), "mixed" (m, k, keep, per_row)
  n         columns of B and C
  entry     "plan" (plan with attached values) or "drop_in" (the positional call without a plan)
  c_f32     C in fp32 instead of fp16
  row_major B[k*N + n] instead of the drop-in layout B[n*K + k]
"""
import functools
import math

import numpy as np
import torch

import smat_amd

BS = 16


def listed():
    return [
        # the smallest product, through the call that replaces the reference's launcher: what one call costs
        _spmm("drop_in_band_1024", "band", 136, entry="drop_in", m=1024, bandwidth=40),
        # a banded system (benchmark configuration 1): short block rows, few wavefronts
        _spmm("band_4096", "band", 128, m=4096, bandwidth=64),
        # a pruned layer fed with a few vectors at a time: reading the weight is the work
        _spmm("pruned_8192_thin", "pruned", 16, m=8192, k=8192, keep=0.10),
        # a pruned layer of odd sizes in fp32 output, too small for one tile per compute unit
        _spmm("pruned_3088_ragged_f32", "pruned", 1000, m=3088, k=4112, keep=0.15, c_f32=True),
        # uniform random sparsity (configuration 2): about one nonzero per block
        _spmm("er_16384", "er", 256, m=16384, k=16384, per_row=16.4),
        # a discretised operator (configuration 5), with a plan and as the drop-in call sees it
        _spmm("stencil_64", "stencil", 64, nx=64, ny=64, nz=64),
        _spmm("drop_in_stencil_64", "stencil", 64, entry="drop_in", nx=64, ny=64, nz=64),
        # the headline configuration 4: a block-pruned layer on a large batch
        _spmm("pruned_8192", "pruned", 4096, m=8192, k=8192, keep=0.10),
        # a pruned layer with stray nonzeros between its blocks, activations row-major as array programs hold them
        _spmm("mixed_8192_row_major", "mixed", 4096, m=8192, k=8192, keep=0.10, per_row=8.2, row_major=True),
        # a power-law graph (configuration 3), the largest
        _spmm("rmat_20", "rmat", 128, scale=20, degree=16),
        # a new matrix: blocked on the device, planned, its values looked at, first product
        {"name": "setup_er_16384", "task": "setup", "matrix": "er", "m": 16384, "k": 16384, "per_row": 16.4, "n": 256,
         "entry": "plan", "c_f32": False, "row_major": False},
        # the offline row and column clustering (host)
        {"name": "reorder_er_4096", "task": "reorder", "matrix": "er", "m": 4096, "k": 4096, "per_row": 16.4},
    ]


def _spmm(name, matrix, n, entry="plan", c_f32=False, row_major=False, **sizes):
    return {"name": name, "task": "spmm", "matrix": matrix, "n": n, "entry": entry, "c_f32": c_f32, "row_major": row_major, **sizes}


def draw(rng):
    while True:
        task = rng.choice(["spmm"] * 10 + ["setup", "reorder"])
        if task == "reorder":
            case = {"task": task, **_draw_matrix(rng, rng.choice(["er", "rmat"]), small=True)}
            return case
        matrix = rng.choice(["band", "er", "rmat", "stencil", "pruned", "pruned", "mixed"] if task == "spmm" else ["er", "stencil", "rmat"])
        case = {"task": task, **_draw_matrix(rng, matrix)}
        widest = {"band": 1024, "er": 1024, "rmat": 256, "stencil": 256, "pruned": 4096, "mixed": 4096}[matrix]
        case["n"] = _log(rng, 64 if matrix == "mixed" else 8, widest, 8)
        case["entry"] = rng.choice(["plan", "plan", "plan", "drop_in"]) if task == "spmm" else "plan"
        case["c_f32"] = case["entry"] == "plan" and rng.random() < 0.25
        case["row_major"] = case["entry"] == "plan" and rng.random() < 0.25
        if _cost(case) <= _largest(task):
            return case


def _draw_matrix(rng, matrix, small=False):
    if matrix == "band":
        return {"matrix": matrix, "m": _log(rng, 512, 65536, 16), "bandwidth": _log(rng, 8, 256, 1)}
    if matrix == "er":
        top = 4096 if small else 65536
        return {"matrix": matrix, "m": _log(rng, 1024, top, 16), "k": _log(rng, 1024, top, 16), "per_row": round(4 * 16 ** rng.random() if not small else 16.0, 2)}
    if matrix == "rmat":
        return {"matrix": matrix, "scale": rng.randint(10, 12) if small else rng.randint(12, 19), "degree": 16 if small else rng.randint(8, 24)}
    if matrix == "stencil":
        return {"matrix": matrix, "nx": _log(rng, 12, 80, 1), "ny": _log(rng, 12, 80, 1), "nz": _log(rng, 12, 80, 1)}
    if matrix == "pruned":
        return {"matrix": matrix, "m": _log(rng, 768, 16384, 16), "k": _log(rng, 768, 16384, 16), "keep": round(0.03 * 12 ** rng.random(), 4)}
    return {"matrix": matrix, "m": _log(rng, 2048, 8192, 16), "k": _log(rng, 2048, 8192, 16), "keep": round(0.05 * 4 ** rng.random(), 4), "per_row": round(2 * 8 ** rng.random(), 2)}


def _log(rng, lo, hi, step):
    """A multiple of `step` between lo and hi, spread over the logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random() / step)) * step))


def _cost(case):
    """Rough bytes that a product touches, block by block: bounds what is drawn."""
    s = _size(case)
    return s["nnzb"] * (512 + 32 * case["n"]) + 2 * s["k"] * case["n"] + 4 * s["m"] * case["n"]


@functools.lru_cache(None)
def _largest(task):
    return max(_cost(c) for c in listed() if c["task"] == task) * (4 if task == "setup" else 1)


# ---- sizes ----


def _size(case):
    return _size_of(*[case.get(f) for f in ("matrix", "m", "k", "keep", "per_row", "bandwidth", "scale", "degree", "nx", "ny", "nz")])


@functools.lru_cache(None)
def _size_of(matrix, m, k, keep, per_row, bandwidth, scale, degree, nx, ny, nz):
    """m, k and the (expected) numbers of nonzeros and of nonzero blocks."""
    if matrix == "band":
        i = np.arange(m)
        nnz = int((np.minimum(m, i + bandwidth + 1) - np.maximum(0, i - bandwidth)).sum())
        b = np.arange(m // BS) * BS
        nnzb = int((np.minimum(m - 1, b + BS - 1 + bandwidth) // BS - np.maximum(0, b - bandwidth) // BS + 1).sum())
        return {"m": m, "k": m, "nnz": nnz, "nnzb": nnzb}
    if matrix == "er":
        return {"m": m, "k": k, "nnz": _distinct(m * per_row, m * k), "nnzb": _distinct(m * per_row, m * k / 256)}
    if matrix == "rmat":
        edges = degree << scale
        return {"m": 1 << scale, "k": 1 << scale, "nnz": _rmat_distinct(edges, scale), "nnzb": _rmat_distinct(edges, scale - 4)}
    if matrix == "stencil":
        m = -(-nx * ny * nz // BS) * BS
        nnz = math.prod(3 * d - 2 for d in (nx, ny, nz))
        first = np.arange(0, nx * ny * nz, BS)
        x, y, z = first % nx, first // nx % ny, first // (nx * ny)
        keys = []
        for dz in (-1, 0, 1):
            for dy in (-1, 0, 1):
                for end, there in ((-1, x > 0), (7, x >= 0), (BS, (x + BS - 1) % nx != nx - 1)):
                    ok = there & (y + dy >= 0) & (y + dy < ny) & (z + dz >= 0) & (z + dz < nz)
                    c = first[ok] + nx * dy + nx * ny * dz
                    keys.append(first[ok] // BS * m + np.clip(c + end, 0, m - 1) // BS)
        return {"m": m, "k": m, "nnz": nnz, "nnzb": int(np.unique(np.concatenate(keys)).size)}
    kept = round(keep * (m // BS) * (k // BS))
    if matrix == "pruned":
        return {"m": m, "k": k, "nnz": kept * 256, "nnzb": kept}
    stray = _distinct(m * per_row, m * k) * (1 - keep)
    return {"m": m, "k": k, "nnz": kept * 256 + stray, "nnzb": kept + _distinct(m * per_row, m * k / 256) * (1 - keep)}


def _distinct(draws, cells):
    return cells * -math.expm1(-draws / cells)


PROBS = (0.57, 0.19, 0.19, 0.05)


def _rmat_distinct(edges, levels):
    total = 0.0
    for i in range(levels + 1):
        for j in range(levels + 1 - i):
            l = levels - i - j
            cells = math.comb(levels, i) * math.comb(levels - i, j) * 2 ** j
            total += cells * -math.expm1(-edges * PROBS[0] ** i * PROBS[1] ** j * PROBS[3] ** l)
    return total


# ---- matrices ----


class DeviceArray:
    """One of the arrays that blocking on the device returned, for the calls that take .data_ptr() and for torch."""

    def __init__(self, owner, address, count, typestr):
        self.owner, self.address = owner, address
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": typestr, "data": (address, False), "version": 2}

    def data_ptr(self):
        return self.address


class Blocked:
    """A blocked matrix on the device and, for the plan, its block pattern on the host."""

    def __init__(self, m, k, nnzb, row_ptr, col_idx, vals):
        self.m, self.k, self.nnzb, self.row_ptr, self.col_idx, self.vals = m, k, nnzb, row_ptr, col_idx, vals

    def plan(self, n, row_major):
        p = smat_amd.Plan(_host(self.row_ptr), self.m, self.k, self.nnzb, n, col_idx_host=_host(self.col_idx), b_row_major=row_major)
        p.attach_values(self.vals, self.row_ptr, self.col_idx)
        return p


def _host(a):
    return (a if isinstance(a, torch.Tensor) else torch.as_tensor(a, device="cuda")).cpu().numpy()


def _block(m, k, row_ptr, col_idx, val):
    d = smat_amd.csr_to_bcsr_device(m, k, row_ptr, col_idx, val, val.numel())
    return Blocked(m, k, d.nnzb, DeviceArray(d, d.row_ptr, m // BS + 1, "<i4"), DeviceArray(d, d.col_idx, d.nnzb, "<i4"),
                   DeviceArray(d, d.val, d.nnzb * 256, "<i2"))


def _row_ptr(rows, m):
    return torch.cat([torch.zeros(1, dtype=torch.int64, device=rows.device), torch.bincount(rows, minlength=m).cumsum(0)]).int()


def _csr(case, gen):
    """(m, k, row_ptr, col_idx, val) on the device."""
    dev = gen.device
    s = _size(case)
    m, k = s["m"], s["k"]
    if case["matrix"] == "band":
        bw = case["bandwidth"]
        i, d = torch.arange(m, device=dev)[:, None], torch.arange(-bw, bw + 1, device=dev)[None, :]
        ok = (i + d >= 0) & (i + d < m)
        rows, cols = (i + 0 * d)[ok], (i + d)[ok]
        val = torch.rand(rows.numel(), generator=gen, device=dev) * 2 - 1
    elif case["matrix"] == "stencil":
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        p = torch.arange(nx * ny * nz, device=dev)[:, None]
        o = torch.tensor([(x, y, z) for z in (-1, 0, 1) for y in (-1, 0, 1) for x in (-1, 0, 1)], device=dev)
        x, y, z = p % nx + o[:, 0], p // nx % ny + o[:, 1], p // (nx * ny) + o[:, 2]
        ok = (x >= 0) & (x < nx) & (y >= 0) & (y < ny) & (z >= 0) & (z < nz)
        cols = (x + nx * y + nx * ny * z)[ok]
        rows = p.expand(-1, 27)[ok]
        val = torch.where(rows == cols, 26.0, -1.0)
    else:
        if case["matrix"] == "rmat":
            a, b, c, _ = PROBS
            edges = case["degree"] << case["scale"]
            rows, cols = torch.zeros(edges, dtype=torch.int64, device=dev), torch.zeros(edges, dtype=torch.int64, device=dev)
            for _ in range(case["scale"]):
                u = torch.rand(edges, generator=gen, device=dev)
                rows = rows * 2 + (u >= a + b)
                cols = cols * 2 + (((u >= a) & (u < a + b)) | (u >= a + b + c))
        else:
            draws = round(m * case["per_row"])
            rows = torch.randint(m, (draws,), generator=gen, device=dev)
            cols = torch.randint(k, (draws,), generator=gen, device=dev)
        keys = torch.unique(rows * k + cols)
        rows, cols = keys // k, keys % k
        val = torch.randn(rows.numel(), generator=gen, device=dev)
    return m, k, _row_ptr(rows, m), cols.int(), val.half()


def _weight(case, gen):
    """A block-pruned weight, for "mixed" with stray nonzeros in other blocks."""
    dev = gen.device
    m, k = case["m"], case["k"]
    mb, kb = m // BS, k // BS
    keys = torch.randperm(mb * kb, generator=gen, device=dev)[:round(case["keep"] * mb * kb)].sort().values
    if case["matrix"] == "mixed":
        draws = round(m * case["per_row"])
        r = torch.randint(m, (draws,), generator=gen, device=dev)
        c = torch.randint(k, (draws,), generator=gen, device=dev)
        stray = (r // BS) * kb + c // BS
        out = ~torch.isin(stray, keys)
        # of draws that meet in one element the first stays
        elem = torch.unique(stray[out] * 256 + r[out] % BS * BS + c[out] % BS)
        full = keys
        keys = torch.unique(torch.cat([full, elem // 256]))
        val = torch.zeros(keys.numel() * 256, dtype=torch.float16, device=dev)
        at = torch.searchsorted(keys, full)[:, None] * 256 + torch.arange(256, device=dev)
        val[at.reshape(-1)] = (torch.randn(at.numel(), generator=gen, device=dev) * 0.02).half()
        val[torch.searchsorted(keys, elem // 256) * 256 + elem % 256] = (torch.randn(elem.numel(), generator=gen, device=dev) * 0.02).half()
    else:
        val = (torch.randn(keys.numel() * 256, generator=gen, device=dev) * 0.02).half()
    return Blocked(m, k, keys.numel(), _row_ptr(keys // kb, mb), (keys % kb * BS).int(), val)


# ---- passes ----


def prepare(case, seed):
    if case["task"] == "reorder":
        m, k, row_ptr, col_idx, _ = _csr(case, torch.Generator("cpu").manual_seed(seed))
        return {"case": case, "m": m, "k": k, "row_ptr": row_ptr.numpy(), "col_idx": col_idx.numpy()}
    gen = torch.Generator("cuda").manual_seed(seed)
    s = {"case": case}
    if case["task"] == "setup":
        s["csr"] = _csr(case, gen)
        m, k = s["csr"][:2]
    else:
        s["a"] = a = _weight(case, gen) if case["matrix"] in ("pruned", "mixed") else _block(*_csr(case, gen))
        m, k = a.m, a.k
        if case["entry"] == "plan":
            s["plan"] = a.plan(case["n"], case["row_major"])
        else:
            smat_amd.lib.smat_plan_cache_clear()  # what a program calls when it has written another pattern
    s["b"] = torch.randn(k * case["n"], generator=gen, device="cuda").half()
    s["c"] = torch.empty((m, case["n"]), dtype=torch.float32 if case["c_f32"] else torch.float16, device="cuda")
    return s


def run(state):
    case = state["case"]
    if case["task"] == "reorder":
        rows, cols, row_stats, col_stats = smat_amd.reorder_csr(state["m"], state["k"], state["row_ptr"], state["col_idx"])
        return {"perm_rows": rows, "perm_cols": cols, "stats_rows": row_stats, "stats_cols": col_stats}
    if case["task"] == "setup":
        a = _block(*state["csr"])
        _multiply(a, a.plan(case["n"], case["row_major"]), state, case)
        return {"row_ptr": torch.as_tensor(a.row_ptr, device="cuda"), "c": state["c"]}
    _multiply(state["a"], state.get("plan"), state, case)
    return state["c"]


def _multiply(a, plan, state, case):
    smat_amd.spmm(a.vals, a.row_ptr, a.col_idx, state["b"], state["c"], a.m, case["n"], a.k, a.nnzb, plan=plan,
                  c_f32=case["c_f32"], drop_in=plan is None, b_row_major=case["row_major"])


def work(case):
    s = _size(case)
    if case["task"] == "reorder":
        return {"bytes": 4 * s["nnz"] + 4 * s["m"] + 8 * (s["m"] + s["k"]), "flops": 0}
    dense = 2 * s["k"] * case["n"] + (4 if case["c_f32"] else 2) * s["m"] * case["n"]
    blocks = 516 * s["nnzb"] + s["m"] / 4
    entries = 6 * s["nnz"] + 4 * s["m"]
    if case["task"] == "setup":
        sparse = entries + blocks  # the CSR in, the blocks out
    elif case["entry"] == "plan":
        sparse = min(blocks, entries)  # the plan has seen where the nonzeros are
    else:
        sparse = blocks
    return {"bytes": sparse + dense, "flops": 2 * s["nnz"] * case["n"]}


def tolerance(case):
    if case["task"] == "reorder":
        return "exact"
    # fp32 sums of fp16 products in another order; results in fp16 may round the other way
    return {"rel": 1e-5, "max": 1e-4} if case["c_f32"] else {"rel": 1e-3, "max": 4e-3}
