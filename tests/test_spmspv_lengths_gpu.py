"""SpMSpV with columns around the length from which they are set aside (256
entries) and around the pieces that they are taken in (512), for matrices with
values and boolean ones."""
import numpy as np
import pytest

import combblas_amd as cb
import oracle

pytestmark = pytest.mark.gpu
LENGTHS = [255, 256, 257, 511, 512, 513, 767, 768, 1023, 1024, 1025, 1, 64]


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("dtype,semiring", [("int64", "plus_times"), ("int64", "min_plus"), ("float64", "plus_times"),
                                            ("bool", "select_max"), ("bool", "plus_times")])
@pytest.mark.parametrize("m", [1100, 70_000])
def test_lengths(m, dtype, semiring, noalloc):
    rng = np.random.default_rng(m)
    rows = np.concatenate([np.sort(rng.choice(m, d, replace=False)) for d in LENGTHS])
    cols = np.repeat(np.arange(len(LENGTHS)), LENGTHS)
    vals = np.ones(rows.size, np.uint8) if dtype == "bool" else rng.integers(-9, 10, rows.size)
    dA = (A := cb.Dcsc.from_coo(m, len(LENGTHS), rows, cols, vals, dtype)).to_device()
    xdt = np.int64 if dtype == "bool" else vals.dtype if dtype == "int64" else np.float64
    for x in [np.arange(len(LENGTHS))] + [np.array([i]) for i in range(len(LENGTHS))]:
        x = x.astype(np.int32)
        xv = rng.integers(-50, 50, x.size).astype(xdt)  # small integers: exact in any order
        want = oracle.spmspv(A, x, xv, semiring)
        got = cb.spmspv(dA, x, xv, semiring, noalloc=noalloc)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), x
