"""The merge in column ranges (cbx_dcsc_merge_in_ranges): with bounds from
one column's entries up, and by itself beyond 2^31 entries."""
from __future__ import annotations

import numpy as np
import pytest

import combblas_amd as cb
import oracle
from tests.helpers import bit_exact

pytestmark = pytest.mark.gpu


def _parts(rng, m, n, counts, dtype):
    out = []
    for k in counts:
        key = np.unique(rng.integers(0, n, k) * m + rng.integers(0, m, k))
        vals = np.ones(key.size, np.uint8) if dtype == "bool" else rng.integers(-9, 10, key.size)
        out.append(cb.Dcsc.from_coo(m, n, key % m, key // m, vals, dtype))
    return out


# m x n, entries drawn per part, and the smallest bound that a column's two partial sums surely fit
SHAPES = [(400, 90, [3000, 0, 2500, 10], 400 * 2), (50, 1, [40, 45, 30, 50, 50], 100), (30, 3000, [100, 4000], 60),
          (70_000, 3, [50_000, 60_000, 9000], 140_000)]


@pytest.mark.parametrize("shape", range(len(SHAPES)))
@pytest.mark.parametrize("semiring,dtype", [("plus_times", "int64"), ("min_plus", "float64"), ("plus_times", "bool"),
                                            ("select_max", "float32")])
def test_ranges_give_the_same_merge(shape, semiring, dtype):
    m, n, counts, least = SHAPES[shape]
    rng = np.random.default_rng(shape)
    parts = _parts(rng, m, n, counts, dtype)
    want = oracle.merge(parts, semiring)
    dparts = [p.to_device() for p in parts]
    total = sum(p.nnz for p in parts)
    for most in sorted({least, least + 1, (least + total) // 2, max(least, total - 1), total, 2**31 - 1}):
        bit_exact(cb.merge(dparts, semiring, max_entries=most).to_host(), want)


def test_bounds_that_do_not_fit():
    rng = np.random.default_rng(5)
    parts = [p.to_device() for p in _parts(rng, 100, 4, [300, 300], "int64")]
    for most, status in ((0, cb.ERR_INVALID), (2**31, cb.ERR_INVALID), (1, cb.ERR_LIMIT)):
        with pytest.raises(cb.CbxError) as ei:
            cb.merge(parts, max_entries=most)
        assert ei.value.status == status


@pytest.mark.parametrize("fault", ["column_at_n", "negative_column", "column_order", "cp_short", "cp_start", "cp_order",
                                   "cp_far", "row", "row_order"])
def test_malformed_parts_are_refused_in_ranges(fault):
    rng = np.random.default_rng(6)
    parts = _parts(rng, 300, 60, [2000, 2500, 1800], "int64")
    X = parts[1]
    if fault == "column_at_n":
        X.jc[-1] = X.n
    elif fault == "negative_column":
        X.jc[0] = -1
    elif fault == "column_order":
        X.jc[[20, 40]] = X.jc[[40, 20]]
    elif fault == "cp_short":
        X.cp[-1] -= 1
    elif fault == "cp_start":
        X.cp[0] = 1
    elif fault == "cp_order":
        X.cp[[20, 40]] = X.cp[[40, 20]]
    elif fault == "cp_far":
        X.cp[30] = 1 << 40
    elif fault == "row":
        X.ir[1000] = X.m
    else:
        X.ir[X.cp[30]:X.cp[30] + 2] = X.ir[X.cp[30]:X.cp[30] + 2][::-1]
    for most in (700, 2000, 2**31 - 1):
        with pytest.raises(cb.CbxError) as ei:
            cb.merge([P.to_device() for P in parts], max_entries=most)
        assert ei.value.status == cb.ERR_INVALID


def _dense(m, n):
    """A full m x n matrix with values 1..9 in a pattern, and its arrays."""
    i = np.arange(m, dtype=np.int64)
    ir = np.tile(i, n)
    return cb.Dcsc(m, n, np.arange(n + 1, dtype=np.int64) * m, np.arange(n, dtype=np.int64), ir, ir % 9 + 1, "int64")


def _sums(X):
    return X.column_checksums(3)


@pytest.mark.parametrize("beyond", [-1, 20_000])
def test_entries_around_two_to_the_31(beyond):
    """16 times one matrix (the parts share its arrays) and a last part that brings the entries to 2^31 + beyond."""
    m = 20_000
    n = 2**31 // (16 * m)
    A = _dense(m, n)
    rest = 2**31 + beyond - 16 * A.nnz  # in whole columns and a shorter one
    full, tail = divmod(rest, m)
    assert 0 < full < n
    keep = full * m + tail
    last = cb.Dcsc(m, n, np.append(A.cp[:full + 1], keep) if tail else A.cp[:full + 1],
                   A.jc[:full + (tail > 0)], A.ir[:keep], A.val[:keep], "int64")
    dA, dlast = A.to_device(), last.to_device()
    parts = [dA] * 16 + [dlast]
    assert sum(P.nnz for P in parts) == 2**31 + beyond
    got = cb.merge(parts)
    assert got.nnz == A.nnz and got.nzc == n
    want = _sums(dA) * np.uint64(16)  # column checksums are linear in the values
    want[:last.nzc] += _sums(dlast)
    assert np.array_equal(_sums(got), want)
    got.check()

