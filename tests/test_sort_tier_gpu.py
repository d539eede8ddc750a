"""The mid tier's product sort (columns of a few hundred to 4096 products) at
the edges of its workgroup sizes, digit widths and gather chunks, against the
oracle."""
import numpy as np
import pytest

import combblas_amd as cb
import oracle
from tests.helpers import bit_exact, same_pattern

pytestmark = pytest.mark.gpu

FLOPS = [257, 1023, 1024, 1025, 2047, 2048, 2049, 4095, 4096]


def column_of_flops(rng, m, flops, one_row, empties):
    """(A, B): B's column j takes flops[j] products from A columns of 1..40 rows (all the row m - 1 when one_row),
    with `empties` entries between them that meet no column of A."""
    n = 30_000
    rows, cols, brow, bcol = [], [], [], []
    at = 0
    for j, f in enumerate(flops):
        left = f
        while left:
            length = 1 if one_row else int(min(left, rng.integers(1, 41), m))
            some = np.unique(rng.integers(0, m, 4 * length + 8))
            rows.append(np.full(1, m - 1) if one_row else rng.permutation(some)[:length])
            cols.append(np.full(length, at))
            brow.append(at)
            bcol.append(j)
            at += 1
            left -= length
        brow.extend(range(at, at + empties))
        bcol.extend([j] * empties)
        at += empties
    assert at <= n
    A = cb.Dcsc.from_coo(m, n, np.concatenate(rows), np.concatenate(cols),
                         rng.integers(-9, 10, sum(map(len, rows))), "int64")
    B = cb.Dcsc.from_coo(n, len(flops), np.array(brow), np.array(bcol), rng.integers(-9, 10, len(brow)), "int64")
    return A, B


@pytest.mark.parametrize("semiring,dtype", [("plus_times", "int64"), ("min_plus", "int64"), ("select_max", "float64"),
                                            ("plus_times", "float32"), ("plus_times", "bool")])
@pytest.mark.parametrize("m,one_row,empties", [(300, False, 0), (100_003, False, 0), (1 << 30, False, 900),
                                               (1 << 20, True, 0)])
def test_sort_tier_edges(semiring, dtype, m, one_row, empties):
    rng = np.random.default_rng(m + len(semiring))
    flops = FLOPS[:4] if one_row else FLOPS
    A, B = column_of_flops(rng, m, flops, one_row, empties)
    A, B = A.astype(dtype), B.astype(dtype)
    C, st = cb.spgemm(A.to_device(), B.to_device(), semiring)
    want, flop = oracle.spgemm(A, B, semiring, "hybrid")
    assert st["flops"] == flop == sum(flops)
    got = C.to_host()
    if dtype.startswith("float"):  # small integers: exact in any order, but which of 0.0 and -0.0 max keeps is not
        same_pattern(got, want)
        assert np.array_equal(got.val, want.val)
    else:
        bit_exact(got, want)
