"""SpGEMM kernels at their edges: value windows and direct blocks of the unit
tier, chunks of more products than a tile of the flattening and more segments
than a workgroup, the tiny tier's distinct-row counts, and column counts around
the tiles of the setup, against the oracle."""
import numpy as np
import pytest

import combblas_amd as cb
import oracle
from tests.helpers import bit_exact

pytestmark = pytest.mark.gpu


def _operands(m, columns, rng):
    """(A, B): column j of B takes the A columns whose rows columns[j] lists (None: a stored entry of B that meets an
    empty column of A)."""
    rows, cols, brow, bcol = [], [], [], []
    at = 0
    for j, parts in enumerate(columns):
        for r in parts:
            if r is not None:
                rows.append(np.asarray(r))
                cols.append(np.full(len(r), at))
            brow.append(at)
            bcol.append(j)
            at += 1
    A = cb.Dcsc.from_coo(m, at, np.concatenate(rows), np.concatenate(cols),
                         rng.integers(1, 10, sum(map(len, rows))), "int64")
    B = cb.Dcsc.from_coo(at, len(columns), np.array(brow), np.array(bcol), rng.integers(1, 10, len(brow)), "int64")
    return A, B


def _check(A, B, kinds):
    flops = None
    for semiring, dtype in kinds:
        a, b = A.astype(dtype), B.astype(dtype)
        C, st = cb.spgemm(a.to_device(), b.to_device(), semiring)
        want, flop = oracle.spgemm(a, b, semiring, "hybrid")
        assert st["flops"] == flop
        bit_exact(C.to_host(), want)  # small positive integers: sums exact in any order, also in FP32
        flops = flop
    return flops


KINDS = [("plus_times", "int64"), ("plus_times", "float32"), ("min_plus", "float64"), ("select_max", "int64")]


def test_unit_windows_and_direct_blocks():
    rng = np.random.default_rng(1)
    m = 70_000  # 18 blocks of 4096 rows: a unit has at most 16
    columns = []
    for count in (3263, 3264, 3265, 6529):  # outputs spread over many blocks
        r = np.sort(rng.choice(m, count, replace=False))
        columns.append([r, r, r[::7], r[::11]])
    for lo, count in ((0, 4096), (0, 4097), (4095, 2), (65_536, m - 65_536), (8192, 4095)):  # dense blocks
        r = np.arange(lo, lo + count)
        columns.append([r] * max(2, 4200 // count + 1))
    columns.append([np.arange(0, m, 16)] * 3)
    A, B = _operands(m, columns, rng)
    _check(A, B, KINDS)


def test_unit_chunks_and_tiles():
    rng = np.random.default_rng(2)
    m = 9000
    short = [np.sort(rng.choice(m, 8, replace=False)) for _ in range(1200)]  # 3 chunks of 512 segments, 9600 products
    long = [np.arange(i % 5, m, 5) for i in range(30)]  # one chunk of 54,000 products: seven tiles
    holes = [x for i in range(700) for x in (None, short[i])]  # segments between entries that meet nothing
    one = [np.arange(17, 17 + 64)] * 100  # 6400 products on 64 rows
    A, B = _operands(m, [short, long, holes, one, [np.arange(m)]], rng)
    _check(A, B, KINDS)


def test_large_units():
    rng = np.random.default_rng(3)
    m = 300_000
    wide = np.sort(rng.choice(m, 140_000, replace=False))  # beyond the split to large units
    A, B = _operands(m, [[wide, wide[::3]], [np.arange(100_000, 240_000)], [np.arange(20)]], rng)
    _check(A, B, KINDS)


@pytest.mark.parametrize("m", [40, 300, 1 << 20])
def test_tiny_columns(m):
    rng = np.random.default_rng(m)
    columns = []
    for distinct in (1, 2, 63, 64, 65, 127, 128, 129, 255, 256):
        d = min(distinct, m)
        r = np.sort(rng.choice(m, d, replace=False))
        columns.append([r])
        columns.append([r[i:i + 1] for i in range(d)])  # one product per entry of B
        columns.append([r] * max(1, 256 // d))  # up to 256 products on d rows
        columns.append([x for k in range(0, d, 3) for x in (r[k:k + 3], None, None)] + [None] * 300)
    columns.append([None] * 5)
    A, B = _operands(m, columns, rng)
    _check(A, B, KINDS + [("plus_times", "bool")])


@pytest.mark.parametrize("ncols", [1, 255, 256, 257, 1023, 1024, 1025, 2049, 70_000])
def test_column_counts(ncols):
    rng = np.random.default_rng(ncols)
    n = 500
    key = np.unique(rng.integers(0, n // 2, 4000) * 2 * n + rng.integers(0, n, 4000))
    A = cb.Dcsc.from_coo(n, n, key % n, key // n, rng.integers(1, 10, key.size), "int64")
    cols = np.repeat(np.arange(ncols), 3)
    key = np.unique(cols * n + rng.integers(0, n, cols.size))
    B = cb.Dcsc.from_coo(n, ncols, key % n, key // n, rng.integers(1, 10, key.size), "int64")
    _check(A, B, KINDS[:1])


@pytest.mark.parametrize("fault", ["row", "order", "column", "cp"])
def test_square_with_a_malformed_operand(fault):
    """A*A looks at its operand once."""
    A = cb.gen_rmat(8, 8, seed=5)
    if fault == "row":
        A.ir[-1] = A.m
    elif fault == "order":
        A.ir[[0, 1]] = A.ir[[1, 0]]
    elif fault == "column":
        A.jc[-1] = A.n
    else:
        A.cp[-1] -= 1
    dA = A.to_device()
    with pytest.raises(cb.CbxError) as ei:
        cb.spgemm(dA, dA, "plus_times")
    assert ei.value.status == cb.ERR_INVALID


@pytest.mark.parametrize("count", [1, 5, 300])
def test_batch_members_around_tiles(count):
    """Members of one and of several packing tiles, empty ones between, against single products and transposes."""
    rng = np.random.default_rng(count)
    As, Bs = [], []
    for i in range(count):
        m, n = int(rng.integers(1, 90)), int(rng.integers(1, 90))
        k = 0 if i % 7 == 3 else 6000 if i % 5 == 0 and i < 50 else int(rng.integers(1, 60))
        for out, p, q in ((As, m, n), (Bs, n, m)):
            key = np.unique(rng.integers(0, p * q, k))
            out.append(cb.Dcsc.from_coo(p, q, key % p, key // p, rng.integers(1, 9, key.size), "int64"))
    Cs, _ = cb.spgemm_batched([A.to_device() for A in As], [B.to_device() for B in Bs], "plus_times")
    for A, B, C in zip(As, Bs, Cs):
        bit_exact(C.to_host(), oracle.spgemm(A, B, "plus_times", "hybrid")[0])
    bit_exact(cb.transpose(As[0].to_device()).to_host(), oracle.transpose(As[0]))
    if count > 5:  # one bad member among good ones
        bad = As[4]
        bad.ir[0] = bad.m
        with pytest.raises(cb.CbxError) as ei:
            cb.spgemm_batched([A.to_device() for A in As], [B.to_device() for B in Bs], "plus_times")
        assert ei.value.status == cb.ERR_INVALID
