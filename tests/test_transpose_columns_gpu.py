"""Transposes of matrices with columns around the lengths where lanes share
them, among short, middling and long ones."""
import numpy as np
import pytest

import combblas_amd as cb
import oracle
from tests.helpers import bit_exact

pytestmark = pytest.mark.gpu
EDGES = [1, 3, 4, 5, 15, 16, 17, 63, 64, 65, 127, 128, 129, 319, 320, 321, 575, 576, 577, 5000]


@pytest.mark.parametrize("others", [0, 2, 9, 20, 80])  # the other columns' length, and so the lanes per column
@pytest.mark.parametrize("dtype", ["int64", "float32", "bool"])
def test_column_lengths(others, dtype):
    rng = np.random.default_rng(others)
    m = 6000
    lengths = np.array(EDGES if not others else [x for e in EDGES for x in [e] + [others] * 40 * max(1, e // others // 10)])
    rows = np.concatenate([np.sort(rng.choice(m, d, replace=False)) for d in lengths])
    cols = np.repeat(np.sort(rng.choice(3 * lengths.size, lengths.size, replace=False)), lengths)
    vals = np.ones(rows.size, np.uint8) if dtype == "bool" else rng.integers(-9, 10, rows.size)
    A = cb.Dcsc.from_coo(m, 3 * lengths.size, rows, cols, vals, dtype)
    bit_exact(cb.transpose(A.to_device()).to_host(), oracle.transpose(A))
