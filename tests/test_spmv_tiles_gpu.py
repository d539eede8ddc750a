"""The tiled dense SpMV at the edges of its tiles, row blocks and chunks."""
import numpy as np
import pytest

import combblas_amd as cb
import oracle

pytestmark = pytest.mark.gpu

TILE = 4096


def _matrix(shape, rng):
    if shape == "whole_tiles":  # 16 full tiles, column starts at tile starts
        m, n = 5000, 32
        cols = np.repeat(np.arange(n), TILE // 2)
        rows = np.concatenate([np.sort(rng.choice(m, TILE // 2, replace=False)) for _ in range(n)])
    elif shape == "one_more":  # a last tile of one entry, columns of one entry
        k = 16 * TILE + 1
        m, n = 1 << 20, k + 7
        cols, rows = np.arange(k) + 3, rng.integers(0, m, k)
    elif shape == "hub_columns":  # columns over several tiles, empty row blocks between
        m, n = (1 << 20) + 1, 5  # the first size with 16384-row blocks
        cols = np.repeat(np.arange(n), 30_000)
        rows = np.concatenate([np.sort(rng.choice(m // 3, 30_000, replace=False)) + (m - m // 3) * (j % 2)
                               for j in range(n)])
    elif shape == "hot_row_block":  # one block with several chunks, the others with one or none
        m, n = 40_000, 200_000
        cols = np.repeat(np.arange(n), 2)
        rows = np.sort(rng.integers(0, 2000, (n, 2)) * 2 + np.arange(2), axis=1).ravel()
        rows[::5000] = m - 1 - np.arange(rows[::5000].size) % 30_000
        keep = np.unique(cols * m + rows)
        cols, rows = keep // m, keep % m
    else:  # banded: a tile's products fall in one or two blocks
        m = n = 30_000
        cols = np.repeat(np.arange(n), 5)
        rows = (cols.reshape(n, 5) + np.arange(-2, 3)).ravel()
        keep = (rows >= 0) & (rows < m)
        cols, rows = cols[keep], rows[keep]
    return m, n, rows.astype(np.int64), cols.astype(np.int64)


@pytest.mark.parametrize("shape", ["whole_tiles", "one_more", "hub_columns", "hot_row_block", "banded"])
def test_tiled_spmv_at_its_edges(shape):
    rng = np.random.default_rng(5)
    m, n, rows, cols = _matrix(shape, rng)
    A = cb.Dcsc.from_coo(m, n, rows, cols, rng.integers(-9, 10, rows.size), "int64")
    assert A.nnz >= 1 << 16  # the tiled form's smallest product
    x, y = rng.integers(-20, 20, n), rng.integers(-50, 50, m)
    for sr in ("plus_times", "min_plus"):
        assert np.array_equal(cb.spmv_dense(A.to_device(), x, y, sr), oracle.spmv_dense(A, x, y, sr))
    # FP32: products of positive numbers are rounded once, their sums in double;
    # a row's rounded parts (one per chunk of its block and y) are at most a few dozen
    Af = A.astype("float32")
    Af.val = rng.uniform(0.5, 2.0, A.nnz).astype(np.float32)
    xf, yf = rng.uniform(0.5, 2.0, n).astype(np.float32), rng.uniform(0.5, 2.0, m).astype(np.float32)
    want = oracle.spmv_dense(Af.astype("float64"), xf.astype(np.float64), yf.astype(np.float64), "plus_times")
    got = cb.spmv_dense(Af.to_device(), xf, yf, "plus_times")
    assert np.allclose(got, want, rtol=64 * 2.0**-24, atol=0)
    # a boolean matrix contributes x itself
    Ab = A.astype("bool")
    assert np.array_equal(cb.spmv_dense(Ab.to_device(), x, y, "select_max"), oracle.spmv_dense(Ab, x, y, "select_max"))
