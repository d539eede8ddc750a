"""SpMSpV where its kernels can go wrong: columns around the length that is set
aside, more of them than their list holds, row counts around bitmap words and
blocks, x at the first and last columns, malformed operands."""
import numpy as np
import pytest

import combblas_amd as cb
import oracle

pytestmark = pytest.mark.gpu


def _check(A, x, xv, semiring):
    dA = A.to_device()
    want = oracle.spmspv(A, x, xv, semiring)
    calls = [False]
    if 4 * A.n + 8 * A.m + A.m // 4 + 4096 <= 16 << 20:
        calls.append(True)
    for noalloc in calls:
        gi, gv = cb.spmspv(dA, x, xv, semiring, noalloc=noalloc)
        assert np.array_equal(gi, want[0]) and np.array_equal(gv, want[1]), noalloc


def _columns(m, lengths, rng):
    rows = np.concatenate([np.sort(rng.choice(m, d, replace=False)) for d in lengths])
    cols = np.repeat(np.arange(len(lengths)), lengths)
    return cb.Dcsc.from_coo(m, len(lengths), rows, cols, rng.integers(-9, 10, rows.size), "int64")


@pytest.mark.parametrize("m", [1, 31, 32, 33, 2047, 2048, 2049, 70_000])
def test_row_counts(m):
    rng = np.random.default_rng(m)
    lengths = [int(d) for d in rng.integers(1, min(m, 40) + 1, 50)]
    A = _columns(m, lengths, rng)
    x = np.array([0, 1, 7, 48, 49], np.int32)
    for sr in ("plus_times", "min_plus", "select_max"):
        _check(A, x, rng.integers(-50, 50, x.size), sr)


def test_long_columns_and_full_list():
    rng = np.random.default_rng(3)
    m = 2100  # 67 bitmap words: the list of long columns holds 134 less the blocks' sums
    A = _columns(m, [1023, 1024, 1025, 2048, 2049, 1, 15, 16, 17, 64, 65] + [1100] * 200, rng)
    x = np.arange(A.n, dtype=np.int32)
    for sr in ("plus_times", "min_plus"):
        _check(A, x, rng.integers(-50, 50, x.size), sr)


def test_blocks_of_many_words():
    rng = np.random.default_rng(4)
    m, k = 9_000_000, 30_000  # more than 4096 blocks of 64 words
    rows, cols = rng.integers(0, m, k), rng.integers(0, 100, k)
    key = np.unique(cols * m + rows)
    A = cb.Dcsc.from_coo(m, 100, key % m, key // m, rng.integers(-9, 10, key.size), "int64")
    x = np.arange(0, 100, 3, dtype=np.int32)
    _check(A, x, rng.integers(-50, 50, x.size), "plus_times")


@pytest.mark.parametrize("fault", ["row", "order", "column", "cp", "x_range", "x_order", "x_twice"])
def test_malformed_operands_are_refused(fault):
    rng = np.random.default_rng(5)
    A = _columns(3000, [20] * 500 + [1500], rng)
    x, xv = np.array([2, 5, 500], np.int32), np.array([1, 2, 3], np.int64)
    if fault == "row":
        A.ir[A.cp[5]] = -1
    elif fault == "order":
        A.ir[[0, 1]] = A.ir[[1, 0]]
    elif fault == "column":
        A.jc[-1] = A.n
    elif fault == "cp":
        A.cp[3] = A.cp[4]
    elif fault == "x_range":
        x[2] = A.n
    elif fault == "x_order":
        x[:2] = x[1::-1]
    else:
        x[1] = x[0]
    dA = A.to_device()
    for noalloc in (False, True):
        with pytest.raises(cb.CbxError) as ei:
            cb.spmspv(dA, x, xv, "plus_times", noalloc=noalloc)
        assert ei.value.status == cb.ERR_INVALID
