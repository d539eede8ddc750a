"""Edge lists to DCSC at the edges of the strips that combine equal entries:
lengths around 64, 512 and 2048, runs over many strips, dropped loops, and
shapes whose last key is an entry."""
import numpy as np
import pytest

import combblas_amd as cb

pytestmark = pytest.mark.gpu


def _build(m, n, rows, cols, vals, dtype, semiring="plus_times", loops=False):
    r, c = cb.DeviceArray.from_host(rows.astype(np.int64)), cb.DeviceArray.from_host(cols.astype(np.int64))
    v = None if vals is None else cb.DeviceArray.from_host(vals)
    try:
        return cb.from_coo_device(m, n, r, c, v, dtype=dtype, semiring=semiring, remove_loops=loops).to_host()
    finally:
        for a in (r, c, v):
            if a is not None:
                a.release()


def _check(m, n, rows, cols, vals, semiring="plus_times", loops=False):
    """Against sorting on the host; integer values, so exact."""
    got = _build(m, n, rows, cols, vals, "int64", semiring, loops)
    keep = rows != cols if loops else np.ones(rows.size, bool)
    v = np.ones(rows.size, np.int64) if vals is None else vals
    key, inv = np.unique(cols[keep] * m + rows[keep], return_inverse=True)
    want = {"plus_times": np.zeros(key.size, np.int64), "min_plus": np.full(key.size, np.iinfo(np.int64).max),
            "select_max": np.full(key.size, np.iinfo(np.int64).min)}[semiring]
    {"plus_times": np.add, "min_plus": np.minimum, "select_max": np.maximum}[semiring].at(want, inv, v[keep])
    jc, first = np.unique(key // m, return_index=True)
    assert got.nnz == key.size and np.array_equal(got.jc, jc)
    assert np.array_equal(got.cp, np.append(first, key.size))
    assert np.array_equal(got.ir, key % m) and np.array_equal(got.val, want)


@pytest.mark.parametrize("count", [1, 63, 64, 65, 511, 512, 513, 2047, 2048, 2049, 20_000])
def test_lengths_and_runs(count):
    rng = np.random.default_rng(count)
    for spread in (1, 3, max(2, count // 40), count * 4):  # one entry, runs over strips, runs within, hardly any
        rows, cols = rng.integers(0, spread, count), rng.integers(0, min(spread, 50), count)
        vals = rng.integers(-9, 10, count)
        for sr in ("plus_times", "min_plus", "select_max"):
            _check(spread, 50, rows, cols, vals, sr)
        _check(spread, 50, rows, cols, None)


def test_run_over_more_strips_than_lanes():
    count = 200_000  # 390 strips, a few entries on either side
    rows, cols = np.full(count, 7), np.full(count, 5)
    rows[:3], rows[-3:] = 6, 8
    _check(20, 20, rows, cols, np.arange(count))
    ones = _build(20, 20, rows, cols, None, "bool")
    assert ones.nnz == 3 and np.array_equal(ones.val, [1, 1, 1])


@pytest.mark.parametrize("shape", [(64, 64), (64, 32), (63, 64), (1, 1), (1, 8)])
def test_dropped_loops_and_last_key(shape):
    m, n = shape
    rng = np.random.default_rng(m + n)
    rows, cols = rng.integers(0, m, 3000), rng.integers(0, n, 3000)
    rows[:5], cols[:5] = m - 1, n - 1
    _check(m, n, rows, cols, rng.integers(-9, 10, 3000), loops=True)
    _check(m, n, rows, cols, rng.integers(-9, 10, 3000), loops=False)


def test_infinities_and_floats():
    rng = np.random.default_rng(1)
    rows, cols = rng.integers(0, 40, 5000), rng.integers(0, 40, 5000)
    vals = np.where(rng.random(5000) < 0.9, np.inf, rng.random(5000))
    got = _build(40, 40, rows, cols, vals, "float64", "min_plus")
    key, inv = np.unique(cols * 40 + rows, return_inverse=True)
    want = np.full(key.size, np.inf)
    np.minimum.at(want, inv, vals)
    assert np.array_equal(got.val, want)
    pos = rng.random(5000)  # sums of at most 20 positive numbers: 20 roundings of 2^-53
    got = _build(40, 40, rows, cols, pos, "float64")
    want = np.zeros(key.size)
    np.add.at(want, inv, pos)
    assert np.allclose(got.val, want, rtol=40 * 2.0**-53, atol=0)
