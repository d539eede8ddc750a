"""BFS levels at the edges of their kernels: vertices of the degrees where a
scan changes its form, vertex counts around a bitmap word, and frontiers that
change between list and bitmap."""
import numpy as np
import pytest

import combblas_amd as cb
import oracle

pytestmark = pytest.mark.gpu


def _hubs(n, degrees):
    """Hub i (vertex 7 i) has degrees[i] neighbours, counted up from different ends; a path joins the hubs."""
    rows, cols = [], []
    for i, d in enumerate(degrees):
        v = 7 * i
        others = np.array([u for u in range(n) if u % 7 or u >= 7 * len(degrees)])
        pick = others[:d - 2] if i % 2 else others[len(others) - (d - 2):]
        pick = np.concatenate([pick, [7 * (i - 1)] if i else [], [7 * (i + 1)] if i + 1 < len(degrees) else []])
        rows.append(np.full(pick.size, v))
        cols.append(pick.astype(np.int64))
    r, c = np.concatenate(rows), np.concatenate(cols)
    key = np.unique(np.concatenate([r * n + c, c * n + r]))
    return cb.Dcsc.from_coo(n, n, key % n, key // n, np.ones(key.size, np.uint8), "bool")


@pytest.mark.parametrize("n", [1280, 1281, 1343])
def test_bfs_scan_forms_and_word_edges(n):
    A = _hubs(n, [3, 8, 9, 32, 33, 40, 128, 129, 512, 513, 514, 1024, 1026])
    deg = np.diff(A.cp)
    assert deg.min() <= 8 and {32, 33}.issubset(set(deg)) and deg.max() > 1024
    dA = A.to_device()
    plans = {d: cb.BfsPlan(dA, d) for d in ("top_down", "bottom_up", "optimizing")}
    for root in (0, 7 * 12, 7 * 5, n - 1, 1):
        want, levels = oracle.bfs(A, root)
        for d, plan in plans.items():
            got, st = plan.run(root)
            assert st["levels"] == levels and st["reached"] == int((want >= 0).sum()), d
            assert np.array_equal(got, want), d
    for plan in plans.values():
        plan.release()


def test_bfs_long_path_changes_direction_back():
    """A dense core with a long tail: the core's levels go bottom-up, the tail's back to top-down."""
    core, tail = 600, 300
    n = core + tail
    rng = np.random.default_rng(2)
    r, c = rng.integers(0, core, 40_000), rng.integers(0, core, 40_000)
    r = np.concatenate([r, np.arange(core - 1, n - 1)])
    c = np.concatenate([c, np.arange(core, n)])
    keep = r != c
    r, c = r[keep], c[keep]
    key = np.unique(np.concatenate([r * n + c, c * n + r]))
    A = cb.Dcsc.from_coo(n, n, key % n, key // n, np.ones(key.size, np.uint8), "bool")
    plan = cb.BfsPlan(A.to_device())
    for root in (0, n - 1):
        want, levels = oracle.bfs(A, root)
        got, st = plan.run(root)
        assert st["levels"] == levels and np.array_equal(got, want)
        assert st["bottom_up_levels"] > 0
    plan.release()
