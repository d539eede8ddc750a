"""Infinite and NaN products under min-plus and select-max.  A row of one
product has that product; infinities take part like numbers.  Of several
products, the semiring's add keeps a NaN that comes first and passes over
later ones (the columns of few products, merges and the dense SpMV do so);
columns of many products and the product with a sparse vector have NaN only
where every product is."""
from __future__ import annotations

import numpy as np
import pytest

import combblas_amd as cb
import oracle
from combblas_amd import predictor

pytestmark = pytest.mark.gpu
KINDS = [(sr, dt) for sr in ("min_plus", "select_max") for dt in ("float64", "float32")]


def _special(rng, size, dtype):
    v = rng.integers(-9, 10, size).astype(dtype)
    u = rng.random(size)
    v[u < 0.2] = np.inf
    v[(u >= 0.2) & (u < 0.3)] = -np.inf
    v[(u >= 0.3) & (u < 0.5)] = np.nan
    return v


def _fold(values, semiring):
    """The semiring's add from left to right."""
    acc = values[0]
    for v in values[1:]:
        acc = (v if v < acc else acc) if semiring == "min_plus" else (v if acc < v else acc)
    return acc


def _many(values, semiring):
    return (np.fmin if semiring == "min_plus" else np.fmax).reduce(values)


def _by_row(rows, values, semiring, how):
    order = np.argsort(rows, kind="stable")
    rows, values = rows[order], values[order]
    starts = np.flatnonzero(np.append(True, rows[1:] != rows[:-1]))
    return rows[starts], np.array([how(v, semiring) for v in np.split(values, starts[1:])])


def _one_column(rng, m, products, dtype):
    """(A, B): B's column takes `products` products from 6 columns of A."""
    k, length = 6, products // 6
    rows = np.concatenate([np.sort(rng.choice(m, length, replace=False)) for _ in range(k)])
    cols = np.repeat(np.arange(k), length)
    A = cb.Dcsc.from_coo(m, k, rows, cols, _special(rng, rows.size, dtype), dtype)
    B = cb.Dcsc.from_coo(k, 1, np.arange(k), np.zeros(k, np.int64), np.ones(k), dtype)
    return A, B


# rows and products: tiny (twice), the three sizes of the sort tier, small, list and large units
@pytest.mark.parametrize("m,products", [(30, 60), (100, 252), (500, 900), (900, 1800), (2000, 4000), (6000, 9000),
                                        (2_000_000, 9000), (200_000, 300_000)])
@pytest.mark.parametrize("semiring,dtype", KINDS)
def test_products(m, products, semiring, dtype):
    A, B = _one_column(np.random.default_rng(m), m, products, dtype)
    terms = A.val + 1 if semiring == "min_plus" else A.val
    rows, want = _by_row(A.ir, terms, semiring, _fold if products <= 256 else _many)
    C, _ = cb.spgemm(A.to_device(), B.to_device(), semiring)
    C = C.to_host()
    assert np.array_equal(C.ir, rows) and np.array_equal(C.val, want, equal_nan=True)


@pytest.mark.parametrize("semiring,dtype", KINDS)
def test_learned_product(semiring, dtype):
    A, B = _one_column(np.random.default_rng(4), 8000, 12_000, dtype)
    rows, want = _by_row(A.ir, A.val + 1 if semiring == "min_plus" else A.val, semiring, _many)
    cb.set_predictor(predictor.load())
    try:
        C, _ = cb.spgemm(A.to_device(), B.to_device(), semiring, "learned")
    finally:
        cb.set_predictor(None)
    C = C.to_host()
    assert np.array_equal(C.ir, rows) and np.array_equal(C.val, want, equal_nan=True)


@pytest.mark.parametrize("semiring,dtype", KINDS)
def test_merge(semiring, dtype):
    rng = np.random.default_rng(7)
    parts = []
    for _ in range(3):
        key = np.unique(rng.integers(0, 40 * 60, 1500))
        parts.append(cb.Dcsc.from_coo(40, 60, key % 40, key // 40, _special(rng, key.size, dtype), dtype))
    key = np.concatenate([p.col_ids() * 40 + p.ir for p in parts])
    at, want = _by_row(key, np.concatenate([p.val for p in parts]), semiring, _fold)
    got = cb.merge([p.to_device() for p in parts], semiring).to_host()
    assert np.array_equal(got.col_ids() * 40 + got.ir, at) and np.array_equal(got.val, want, equal_nan=True)


@pytest.mark.parametrize("nnz", [5000, 120_000])  # direct, tiled
@pytest.mark.parametrize("semiring,dtype", KINDS)
def test_dense_spmv(nnz, semiring, dtype):
    rng = np.random.default_rng(nnz)
    m, n = 3000, 4000
    key = np.unique(rng.integers(0, m * n, nnz))
    A = cb.Dcsc.from_coo(m, n, key % m, key // m, _special(rng, key.size, dtype), dtype)
    x, y = rng.integers(1, 4, n).astype(dtype), _special(rng, m, dtype)
    got = cb.spmv_dense(A.to_device(), x, y, semiring)
    assert np.array_equal(got, oracle.spmv_dense(A, x, y, semiring), equal_nan=True)


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("semiring,dtype", KINDS)
def test_sparse_vector(noalloc, semiring, dtype):
    rng = np.random.default_rng(8)
    lengths = np.append(rng.integers(1, 40, 60), [300, 700])  # and two columns that are set aside
    rows = np.concatenate([np.sort(rng.choice(2000, d, replace=False)) for d in lengths])
    A = cb.Dcsc.from_coo(2000, lengths.size, rows, np.repeat(np.arange(lengths.size), lengths),
                         _special(rng, rows.size, dtype), dtype)
    x = np.arange(lengths.size, dtype=np.int32)
    xv = rng.integers(1, 4, x.size).astype(dtype)
    per = np.repeat(xv, lengths)
    at, want = _by_row(A.ir, A.val + per if semiring == "min_plus" else A.val * per, semiring, _many)
    gi, gv = cb.spmspv(A.to_device(), x, xv, semiring, noalloc=noalloc)
    assert np.array_equal(gi, at) and np.array_equal(gv, want, equal_nan=True)


@pytest.mark.parametrize("count,spread", [(3, 1), (64, 1), (700, 5), (20_000, 1), (20_000, 300), (200_000, 2)])
@pytest.mark.parametrize("semiring,dtype", KINDS)
def test_edge_list(count, spread, semiring, dtype):
    """Equal entries are folded in input order, in runs within a wave and over many strips."""
    rng = np.random.default_rng(count + spread)
    rows, cols = rng.integers(0, spread, count), rng.integers(0, 2, count)
    vals = _special(rng, count, dtype)
    at, want = _by_row(cols * spread + rows, vals, semiring, _fold)
    dr, dc, dv = (cb.DeviceArray.from_host(a) for a in (rows, cols, vals))
    got = cb.from_coo_device(spread, 2, dr, dc, dv, dtype=dtype, semiring=semiring).to_host()
    assert np.array_equal(got.col_ids() * spread + got.ir, at) and np.array_equal(got.val, want, equal_nan=True)
