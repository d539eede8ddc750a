"""The workloads that this library's speed is measured on.

Each case is one call (for the merge and the Galerkin batch, one call on many
matrices) of a public entry point of ``combblas_amd``, as a program that uses
the library makes it: operands resident in HBM, library-default tunables, the
result left in HBM (SpMSpV, whose Python form takes and returns host arrays,
excepted).  The kinds:

  spgemm    C = A*A on one block (``spgemm``): R-MAT graphs, from blocks of a
            few hundred columns to a million, every semiring and value type,
            exact two-phase or learned sizing
  mcl       one MCL expansion (``mcl_expand``): column-stochastic power-law A
            in FP32, A*A pruned at 1e-4 and to the top 1000 of a column
  galerkin  batched triple products T^T A T (``galerkin_batched``): 27-point
            stencils with varying coefficients and 2x2x2 aggregation, FP64
  merge     the merge of SUMMA's stage products (``merge``)
  spmv      y += A*x with a dense x (``spmv_dense_device``)
  spmspv    y = A (x) x with a sparse x (``spmspv``): one BFS level's product
  bfs       a whole BFS from one root on a plan (``BfsPlan.run``)
  build     an edge list to DCSC (``from_coo_device``)

Inputs are drawn on the GPU with torch.  A case's graph (its entries up to a
relabelling) belongs to the case, so that results of every seed have the same
sizes; the seed shifts the vertex labels cyclically and draws the values, the
vectors and the roots.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import combblas_amd as cb
from combblas_amd import predictor

DEV = "cuda"
TORCH_DTYPE = {"int64": torch.int64, "float64": torch.float64, "float32": torch.float32, "bool": torch.uint8}
TYPESTR = {"int64": "<i8", "float64": "<f8", "float32": "<f4", "bool": "|u1"}
RMAT_A, RMAT_B, RMAT_C = 0.57, 0.19, 0.19  # quadrant probabilities of the Graph500 generator
MCL_THR, MCL_SELECT = 1e-4, 1000
# Products that exact() expands (as 64-bit keys and values, sorted) in one piece, and at most.
EXACT_PIECE, EXACT_MOST = 400_000_000, 13_000_000_000


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # A small block's product: a coarse multigrid level, a small SUMMA stage.  Launches and host work count.
        {"name": "spgemm_s9_int64", "kind": "spgemm", "n": 512, "ef": 8, "dtype": "int64",
         "semiring": "plus_times", "mode": "two_phase"},
        # The plain local product of a 2^14-vertex graph.
        {"name": "spgemm_s14_int64", "kind": "spgemm", "n": 1 << 14, "ef": 8, "dtype": "int64",
         "semiring": "plus_times", "mode": "two_phase"},
        # Two-hop shortest paths on an odd-sized graph.
        {"name": "spgemm_minplus_f64", "kind": "spgemm", "n": 70_001, "ef": 12, "dtype": "float64",
         "semiring": "min_plus", "mode": "two_phase"},
        # The headline product's shape, at the size whose output fits the card beside the previous one.
        {"name": "spgemm_s19_int64", "kind": "spgemm", "n": 1 << 19, "ef": 16, "dtype": "int64",
         "semiring": "plus_times", "mode": "two_phase"},
        # The learned single pass, on a size that its network was trained for.
        {"name": "spgemm_learned_s17", "kind": "spgemm", "n": 1 << 17, "ef": 16, "dtype": "int64",
         "semiring": "plus_times", "mode": "learned"},
        # Markov clustering: one expansion with its pruning.
        {"name": "mcl_n500k_f32", "kind": "mcl", "n": 500_000, "mean": 32},
        # Multigrid setup on a batch of blocks of uneven size.
        {"name": "galerkin_16_f64", "kind": "galerkin", "count": 16, "lo": 16, "hi": 96},
        # SUMMA's end of a multiplication: four stage products into one.
        {"name": "merge_4_s16_int64", "kind": "merge", "n": 1 << 16, "ef": 16, "parts": 4, "dtype": "int64"},
        # One step of a power iteration (PageRank, an eigensolver) on a large graph.
        {"name": "spmv_s20_f64", "kind": "spmv", "n": 1 << 20, "ef": 16, "dtype": "float64"},
        # One sparse frontier's product, vectors on the host.
        {"name": "spmspv_s18", "kind": "spmspv", "n": 1 << 18, "ef": 16, "share": 0.02},
        # Graph500's kernel 2.
        {"name": "bfs_s20", "kind": "bfs", "n": 1 << 20, "ef": 16, "direction": "optimizing"},
        # Graph500's kernel 1.
        {"name": "build_s20_int64", "kind": "build", "n": 1 << 20, "ef": 16, "dtype": "int64"},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["spgemm", "spgemm", "spgemm", "mcl", "galerkin", "merge", "spmv", "spmspv", "bfs", "build"])
    if kind == "spgemm":
        semiring, dtype = rng.choice([("plus_times", "int64"), ("plus_times", "int64"), ("plus_times", "float64"),
                                      ("plus_times", "float32"), ("plus_times", "bool"), ("min_plus", "float64"),
                                      ("min_plus", "int64"), ("select_max", "int64")])
        n, ef = _log_uniform(rng, 500, 400_000), rng.randint(4, 16)
        mode = "learned" if n >= 1 << 14 and rng.random() < 0.2 else "two_phase"
        return {"kind": kind, "n": n, "ef": ef, "dtype": dtype, "semiring": semiring, "mode": mode}
    if kind == "mcl":
        return {"kind": kind, "n": _log_uniform(rng, 300_000, 700_000), "mean": rng.randint(12, 28)}
    if kind == "galerkin":
        lo = rng.randint(4, 32)
        return {"kind": kind, "count": rng.randint(4, 16), "lo": lo, "hi": lo + rng.randint(4, 60)}
    if kind == "merge":
        return {"kind": kind, "n": _log_uniform(rng, 3000, 1 << 16), "ef": rng.randint(4, 15), "parts": rng.randint(2, 6),
                "dtype": rng.choice(["int64", "float64"])}
    if kind == "spmv":
        return {"kind": kind, "n": _log_uniform(rng, 2000, 1 << 20), "ef": rng.randint(4, 15),
                "dtype": rng.choice(["int64", "float64", "float32"])}
    if kind == "spmspv":
        return {"kind": kind, "n": _log_uniform(rng, 2000, 1 << 20), "ef": rng.randint(4, 16),
                "share": round(math.exp(rng.uniform(math.log(1e-4), math.log(0.1))), 6)}
    if kind == "bfs":
        return {"kind": kind, "n": _log_uniform(rng, 4000, 1 << 20), "ef": rng.randint(4, 15),
                "direction": rng.choice(["optimizing", "optimizing", "top_down"])}
    return {"kind": kind, "n": _log_uniform(rng, 2000, 1 << 20), "ef": rng.randint(4, 15),
            "dtype": rng.choice(["int64", "int64", "bool"])}


# ----------------------------------------------------------------- the inputs
def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _shift(n, seed):
    """The seed's cyclic relabelling of n vertices, in [0, n)."""
    return int(np.random.default_rng([int(seed), 11]).integers(n))


def _rmat_edges(n, ef):
    """(rows, cols) of n * ef R-MAT edges, duplicates and loops among them, labels unshifted."""
    g = _generator(n * 64 + ef)
    scale = max(1, (n - 1).bit_length())
    e = n * ef
    rows = torch.zeros(e, dtype=torch.int64, device=DEV)
    cols = torch.zeros(e, dtype=torch.int64, device=DEV)
    for _ in range(scale):
        u = torch.rand(e, generator=g, device=DEV)
        down = u >= RMAT_A + RMAT_B
        right = ((u >= RMAT_A) & ~down) | (u >= RMAT_A + RMAT_B + RMAT_C)
        rows = rows * 2 + down
        cols = cols * 2 + right
    if n != 1 << scale:
        rows, cols = (rows * n) >> scale, (cols * n) >> scale
    return rows, cols


def _values(count, dtype, g):
    if dtype == "bool":
        return torch.ones(count, dtype=torch.uint8, device=DEV)
    if dtype == "int64":
        return torch.randint(1, 10, (count,), generator=g, device=DEV)
    return (torch.rand(count, generator=g, device=DEV, dtype=torch.float64) * 8 + 1).to(TORCH_DTYPE[dtype])


def _rmat(n, ef, dtype, seed, symmetric=False):
    """(rows, cols, values) of an R-MAT matrix without duplicate entries."""
    rows, cols = _rmat_edges(n, ef)
    if symmetric:
        keep = rows != cols
        rows, cols = rows[keep], cols[keep]
        rows, cols = torch.cat([rows, cols]), torch.cat([cols, rows])
    key = torch.unique(cols * n + rows)
    s = _shift(n, seed)
    return (key % n + s) % n, (key // n + s) % n, _values(key.numel(), dtype, _generator(seed))


def _powerlaw(n, mean, seed):
    """(rows, cols, values) of a column-stochastic matrix: configuration model of a power-law degree sequence
    (exponent 2.1, cut off at sqrt(n * mean)), log-normal weights normalised per column and rounded to 12 bits, the
    precision at which sums of products are exact in FP32 in any order, so that two runs prune alike.  Only the labels
    come from the seed: other weights would keep another number of entries."""
    g = _generator(n * 64 + mean)
    cut = math.sqrt(n * mean)
    u = torch.rand(n, generator=g, device=DEV, dtype=torch.float64).clamp_min(1e-12)
    tail = u.pow(-1.0 / 1.1)
    lo, hi = 1.0, float(mean)
    for _ in range(40):  # the smallest degree at which the mean comes out
        mid = (lo + hi) / 2
        lo, hi = (mid, hi) if float((tail * mid).clamp_max(cut).floor().mean()) < mean else (lo, mid)
    deg = (tail * hi).clamp_max(cut).floor().to(torch.int64)
    cols = torch.repeat_interleave(torch.arange(n, device=DEV), deg)
    rows = cols[torch.randperm(cols.numel(), generator=g, device=DEV)]
    key = torch.unique(cols * n + rows)
    rows, cols = key % n, key // n
    w = torch.exp(torch.randn(key.numel(), generator=g, device=DEV, dtype=torch.float64))
    total = torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, cols, w)
    v = (w / total[cols] * 4096).round().clamp_min(1) / 4096
    s = _shift(n, seed)
    rows, cols = (rows + s) % n, (cols + s) % n
    order = torch.argsort(cols * n + rows)
    return rows[order], cols[order], v[order].to(torch.float32)


def _grids(case):
    r = np.random.default_rng([case["count"], case["lo"], case["hi"]])
    return [case["hi"]] + [int(x) for x in r.integers(case["lo"], case["hi"] + 1, case["count"] - 1)]


def _stencil(grid, g):
    """(rows, cols, values) of a 27-point operator on a grid^3 mesh with varying coefficients."""
    i = torch.arange(grid, device=DEV)
    d = torch.arange(-1, 2, device=DEV)
    cell = torch.cartesian_prod(i, i, i)
    off = torch.cartesian_prod(d, d, d)
    to = cell[:, None, :] + off[None, :, :]
    ok = ((to >= 0) & (to < grid)).all(-1)
    place = torch.tensor([grid * grid, grid, 1], device=DEV)
    cols = (cell * place).sum(-1)[:, None].expand(ok.shape)
    rows = (to * place).sum(-1)
    rows, cols = rows[ok], cols[ok]
    v = -(torch.rand(rows.numel(), generator=g, device=DEV, dtype=torch.float64) + 0.5)
    return rows, cols, torch.where(rows == cols, 26.0 - v, v)


def _aggregates(grid):
    """The coarse cell of every fine cell, and the coarse grid's edge."""
    half = (grid + 1) // 2
    i = torch.arange(grid, device=DEV) // 2
    c = torch.cartesian_prod(i, i, i)
    return (c * torch.tensor([half * half, half, 1], device=DEV)).sum(-1), half


def _device_array(t):
    t = t.contiguous()
    dtype = {torch.int64: np.int64, torch.float64: np.float64, torch.float32: np.float32, torch.uint8: np.uint8}[t.dtype]
    d = cb.DeviceArray(t.numel(), dtype)
    if t.numel():
        status = cb.lib().cbx_memcpy(d.ptr, t.data_ptr(), t.numel() * t.element_size(), 2)
        if status:
            raise RuntimeError(f"copy to a library array failed ({status})")
    return d


def _matrix(m, n, coo, dtype):
    rows, cols, vals = coo
    r, c, v = (_device_array(x) for x in (rows, cols, vals))
    torch.cuda.synchronize()
    M = cb.from_coo_device(m, n, r, c, v, dtype=dtype)
    cb.synchronize()
    return M


def _vector(n, dtype, g):
    if dtype == "int64":
        return torch.randint(-9, 10, (n,), generator=g, device=DEV)
    return (torch.rand(n, generator=g, device=DEV, dtype=torch.float64) * 2 - 1).to(TORCH_DTYPE[dtype])


def _spmv_inputs(case, seed):
    g = _generator(seed + 1)
    coo = _rmat(case["n"], case["ef"], case["dtype"], seed)
    return coo, _vector(case["n"], case["dtype"], g), _vector(case["n"], case["dtype"], g)


def _galerkin_inputs(case, seed):
    g = _generator(seed)
    out = []
    for grid in _grids(case):
        agg, half = _aggregates(grid)
        out.append((grid, half, _stencil(grid, g), agg))
    return out


# ------------------------------------------------------- the library's results
class _Span:
    """Device memory of the library, seen by torch without a copy; keeps its owner alive."""

    def __init__(self, ptr, count, dtype, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": TYPESTR[dtype], "data": (ptr or 0, False),
                                         "version": 2, "strides": None}


def _tensor(ptr, count, dtype, owner):
    if count == 0:
        return torch.empty(0, dtype=TORCH_DTYPE[dtype], device=DEV)
    return torch.as_tensor(_Span(ptr, count, dtype, owner), device=DEV)


_NAMES = {v: k for k, v in cb.DTYPES.items()}


def _arrays(M):
    """A device matrix as its four arrays."""
    s = M.s
    return {"cp": _tensor(s.cp, s.nzc + 1, "int64", M), "jc": _tensor(s.jc, s.nzc, "int64", M),
            "ir": _tensor(s.ir, s.nnz, "int64", M), "val": _tensor(s.val, s.nnz, _NAMES[s.dtype], M)}


def _bytes(M):
    return 16 * M.nzc + 8 + (8 + {"int64": 8, "float64": 8, "float32": 4, "bool": 1}[_NAMES[M.s.dtype]]) * M.nnz


# ------------------------------------------------------------ prepare and run
def prepare(case, seed):
    kind, state = case["kind"], dict(case)
    if kind == "spgemm":
        state["A"] = _matrix(case["n"], case["n"], _rmat(case["n"], case["ef"], case["dtype"], seed), case["dtype"])
        if case["mode"] == "learned":
            cb.set_predictor(predictor.load())
    elif kind == "mcl":
        state["A"] = _matrix(case["n"], case["n"], _powerlaw(case["n"], case["mean"], seed), "float32")
    elif kind == "galerkin":
        state["A"], state["T"] = [], []
        for grid, half, coo, agg in _galerkin_inputs(case, seed):
            fine = torch.arange(agg.numel(), device=DEV)
            state["A"].append(_matrix(grid ** 3, grid ** 3, coo, "float64"))
            state["T"].append(_matrix(grid ** 3, half ** 3, (fine, agg, torch.ones(agg.numel(), dtype=torch.float64, device=DEV)), "float64"))
    elif kind == "merge":
        n = case["n"]
        rows, cols, vals = _rmat(n, case["ef"], case["dtype"], seed)
        row0, col0 = ((x + n - _shift(n, seed)) % n for x in (rows, cols))  # labels that every seed shares
        state["parts"] = []
        for s in range(case["parts"]):
            lo, hi = s * n // case["parts"], (s + 1) * n // case["parts"]
            of_a, of_b = (col0 >= lo) & (col0 < hi), (row0 >= lo) & (row0 < hi)
            A = _matrix(n, n, (rows[of_a], cols[of_a], vals[of_a]), case["dtype"])
            B = _matrix(n, n, (rows[of_b], cols[of_b], vals[of_b]), case["dtype"])
            state["parts"].append(cb.spgemm(A, B)[0])
    elif kind == "spmv":
        coo, x, y = _spmv_inputs(case, seed)
        state["A"], state["x"], state["y"] = _matrix(case["n"], case["n"], coo, case["dtype"]), _device_array(x), _device_array(y)
    elif kind == "spmspv":
        n = case["n"]
        state["A"] = _matrix(n, n, _rmat(n, case["ef"], "bool", seed, symmetric=True), "bool")
        count = max(1, int(n * case["share"]))
        at = torch.randperm(n, generator=_generator(n), device=DEV)[:count]
        at = torch.sort((at + _shift(n, seed)) % n).values.cpu().numpy()
        state["xind"], state["xval"] = at.astype(np.int32), at.astype(np.int64)
    elif kind == "bfs":
        g = _generator(seed)
        coo = _rmat(case["n"], case["ef"], "bool", seed, symmetric=True)
        state["A"] = _matrix(case["n"], case["n"], coo, "bool")
        state["root"] = int(coo[1][int(torch.randint(0, coo[1].numel(), (1,), generator=g, device=DEV))])
        state["plan"] = cb.BfsPlan(state["A"], case["direction"])
    elif kind == "build":
        n, s = case["n"], _shift(case["n"], seed)
        rows, cols = ((x + s) % n for x in _rmat_edges(n, case["ef"]))
        state["rows"], state["cols"] = _device_array(rows), _device_array(cols)
        state["vals"] = None if case["dtype"] == "bool" else _device_array(_values(rows.numel(), case["dtype"], _generator(seed)))
    return state


def _call(state):
    """(outputs, bytes of the inputs and outputs, operations) of one pass."""
    kind = state["kind"]
    if kind == "spgemm":
        C, st = cb.spgemm(state["A"], state["A"], state["semiring"], state["mode"])
        return _arrays(C), 2 * _bytes(state["A"]) + _bytes(C), 2 * st["flops"]
    if kind == "mcl":
        C, st = cb.mcl_expand(state["A"], None, MCL_THR, MCL_SELECT)
        return _arrays(C), 2 * _bytes(state["A"]) + _bytes(C), 2 * st["flops"]
    if kind == "galerkin":
        S, st = cb.galerkin_batched(state["A"], state["T"])
        moved = sum(_bytes(X) for X in state["A"] + state["T"] + S)
        return [_arrays(X) for X in S], moved, 2 * st["flops"]
    if kind == "merge":
        C = cb.merge(state["parts"])
        return _arrays(C), sum(_bytes(P) for P in state["parts"]) + _bytes(C), sum(P.nnz for P in state["parts"])
    if kind == "spmv":
        A, x, y = state["A"], state["x"], state["y"]
        cb.spmv_dense_device(A, x, y)
        moved = _bytes(A) + x.dtype.itemsize * (A.nzc + 2 * A.m)
        return _tensor(y.ptr, y.n, state["dtype"], y), moved, 2 * A.nnz
    if kind == "spmspv":
        yi, yv = cb.spmspv(state["A"], state["xind"], state["xval"])
        return {"index": yi, "value": yv}, 12 * (len(state["xind"]) + len(yi)) + 9 * int(state["A"].nnz * state["share"]), 0
    if kind == "bfs":
        plan = state["plan"]
        _, st = plan.run(state["root"], copy=False)
        parents = _tensor(plan.parents.ptr, plan.n, "int64", plan)
        return {"parents": parents, "reached": st["reached"]}, 4 * state["A"].nnz + 16 * plan.n, 0
    C = cb.from_coo_device(state["n"], state["n"], state["rows"], state["cols"], state["vals"], dtype=state["dtype"],
                           remove_loops=True)
    edges = state["rows"].n * (16 if state["vals"] is None else 24)
    return _arrays(C), edges + _bytes(C), 0


def run(state):
    return _call(state)[0]


def work(case):
    outputs, moved, operations = _call(prepare(case, 0))
    del outputs
    return {"bytes": moved, "flops": operations}


# ------------------------------------------------------ the results in 64 bits
def _compress(keys, vals, n, keep=None):
    """The four arrays of a matrix whose sorted distinct entries have the keys col * n + row."""
    if keep is not None:
        keys, vals = keys[keep], vals[keep]
    jc, counts = torch.unique_consecutive(keys // n, return_counts=True)
    cp = torch.cat([torch.zeros(1, dtype=torch.int64, device=DEV), torch.cumsum(counts, 0)])
    return {"cp": cp, "jc": jc, "ir": keys % n, "val": vals}


def _reduce(keys, vals, semiring):
    keys, at = torch.sort(keys)
    vals = vals[at]
    keys, counts = torch.unique_consecutive(keys, return_counts=True)
    to = torch.repeat_interleave(torch.arange(keys.numel(), device=DEV), counts)
    if semiring == "plus_times":
        return keys, torch.zeros(keys.numel(), dtype=torch.float64, device=DEV).index_add_(0, to, vals)
    start = torch.full((keys.numel(),), math.inf, dtype=torch.float64, device=DEV)
    return keys, start.scatter_reduce_(0, to, vals, "amin")


def _square(n, coo, semiring):
    """Pieces (sorted keys, values) of A*A, whole columns in each, from the products of all entry pairs."""
    order = torch.argsort(coo[1] * n + coo[0])
    rows, cols, vals = (x[order] for x in coo)
    vals = vals.double()
    length = torch.bincount(cols, minlength=n)
    first = torch.cumsum(length, 0) - length
    products = length[rows]
    so_far = torch.cumsum(products, 0)
    total = int(so_far[-1])
    if total > EXACT_MOST:
        return None
    ends = torch.cumsum(length, 0)  # entries up to the end of each column
    upto = torch.where(ends > 0, so_far[(ends - 1).clamp_min(0)], torch.zeros_like(ends))
    pieces, lo = [], 0
    while lo < n:
        base = int(upto[lo - 1]) if lo else 0
        hi = max(lo + 1, int(torch.searchsorted(upto, base + EXACT_PIECE, right=True)))
        pieces.append((int(ends[lo - 1]) if lo else 0, int(ends[min(hi, n) - 1])))
        lo = hi

    def expand():
        for e0, e1 in pieces:
            count = products[e0:e1]
            which = torch.repeat_interleave(torch.arange(e0, e1, device=DEV), count)
            start = torch.cumsum(count, 0) - count
            a = first[rows[which]] + torch.arange(which.numel(), device=DEV) - start[which - e0]
            v = vals[a] * vals[which] if semiring == "plus_times" else vals[a] + vals[which]
            yield _reduce(cols[which] * n + rows[a], v, semiring)

    return expand()


def exact(case, seed):
    kind, n = case["kind"], case.get("n")
    if kind == "spgemm" and case["dtype"].startswith("float"):
        pieces = _square(n, _rmat(n, case["ef"], case["dtype"], seed), case["semiring"])
        if pieces is None:
            return None
        keys, vals = zip(*pieces)
        return _compress(torch.cat(keys), torch.cat(vals), n)
    if kind == "mcl":
        pieces = _square(n, _powerlaw(n, case["mean"], seed), "plus_times")
        if pieces is None:
            return None
        kept = []
        for keys, vals in pieces:
            big = vals >= MCL_THR
            keys, vals = keys[big], vals[big]
            # the largest MCL_SELECT entries of a column, with all that equal the last of them
            by = torch.argsort(vals, descending=True, stable=True)
            by = by[torch.argsort(keys[by] // n, stable=True)]
            col, counts = torch.unique_consecutive(keys[by] // n, return_counts=True)
            start = torch.cumsum(counts, 0) - counts
            last = start + counts.clamp_max(MCL_SELECT) - 1
            cut = torch.zeros(n, dtype=torch.float64, device=DEV)
            cut[col] = vals[by][last]
            keep = vals >= cut[keys // n]
            kept.append((keys[keep], vals[keep]))
        keys, vals = zip(*kept)
        return _compress(torch.cat(keys), torch.cat(vals), n)
    if kind == "galerkin":
        out = []
        for _, half, (rows, cols, vals), agg in _galerkin_inputs(case, seed):
            nc = half ** 3
            out.append(_compress(*_reduce(agg[cols] * nc + agg[rows], vals, "plus_times"), nc))
        return out
    if kind == "spmv" and case["dtype"].startswith("float"):
        (rows, cols, vals), x, y = _spmv_inputs(case, seed)
        return y.double().index_add_(0, rows, vals.double() * x.double()[cols])
    return None
