"""The cut of a graph into regions, on the host, against a plain restatement of
its rule: consecutive ids where few of their edges cross, else regions grown
breadth-first and continued in pockets; up to 1024 vertices each, by falling
degree.  Graphs around the region size, shuffled and in order, with isolated
vertices, small components, parallel edges and self-loops, and vertices of up to
64 edges (one more, or a mean past 8: not cut)."""
import ctypes
import os
from collections import deque

import numpy as np
import pytest

from graphs_util import grid_csr, random_csr

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "libregionplan.so")
FULL = 1024


@pytest.fixture(scope="module")
def plan():
    if not os.path.exists(LIB):
        raise RuntimeError(f"{LIB} missing: build() compiles it")
    lib = ctypes.CDLL(LIB)

    def run(row, col):
        n = len(row) - 1
        row, col = (np.ascontiguousarray(x, dtype=np.uint32) for x in (row, col))
        order, first = np.empty(n, np.uint32), np.empty(n + 1, np.uint32)
        k = lib.region_plan_check(ctypes.c_uint32(n), *(ctypes.c_void_p(x.ctypes.data)
                                                        for x in (row, col, order, first)))
        assert k >= -1
        return None if k < 0 else [order[first[i]:first[i + 1]].tolist() for i in range(k)]
    return run


def expected(row, col):
    n, m = len(row) - 1, len(col)
    deg = np.diff(row)
    if m > 8 * n or deg.max() > 64:
        return None
    src = np.repeat(np.arange(n), deg)
    if (src // FULL != col // FULL).sum() <= 0.06 * m:
        regions = [list(range(a, min(n, a + FULL))) for a in range(0, n, FULL)]
    else:
        regions, region, rim, taken, nxt = [], [], deque(), np.zeros(n, bool), 0
        while taken.sum() < n:
            seed = None
            while rim and seed is None:
                v = rim.popleft()
                seed = None if taken[v] else v
            if seed is None:
                while taken[nxt]:
                    nxt += 1
                seed = nxt
            if len(region) > FULL * 3 // 4:
                regions.append(region)
                region = []
            head = len(region)
            taken[seed] = True
            region.append(seed)
            while head < len(region):
                for v in col[row[region[head]]:row[region[head] + 1]]:
                    if taken[v]:
                        continue
                    if len(region) < FULL:
                        taken[v] = True
                        region.append(int(v))
                    else:
                        rim.append(int(v))
                head += 1
        regions.append(region)
    return [sorted(r, key=lambda v: -deg[v]) for r in regions]   # (stable)


def shuffled(row, col, seed):
    n = len(row) - 1
    p = np.random.default_rng(seed).permutation(n)
    src, dst = p[np.repeat(np.arange(n), np.diff(row))], p[col]
    order = np.lexsort((dst, src))
    return np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]), dst[order]


def chain(n):
    a = np.arange(n - 1)
    src = np.concatenate([a, a + 1])
    dst = np.concatenate([a + 1, a])
    order = np.lexsort((dst, src))
    return np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]), dst[order]


@pytest.mark.parametrize("n", [1, 2, 767, 768, 769, 1023, 1024, 1025, 2048, 5000])
@pytest.mark.parametrize("mix", [False, True])
def test_chains(plan, n, mix):
    g = chain(n)
    g = shuffled(*g, n) if mix else g
    assert plan(*g) == expected(*g)


@pytest.mark.parametrize("rows,cols", [(32, 32), (33, 32), (60, 70), (10, 900)])
@pytest.mark.parametrize("mix", [False, True])
def test_grids(plan, rows, cols, mix):
    row, col, _ = grid_csr(rows, cols, 1)
    g = shuffled(row, col, 2) if mix else (row, col)
    assert plan(*g) == expected(*g)


@pytest.mark.parametrize("n,m,seed", [(3000, 0, 1), (3000, 900, 2), (3000, 3000, 3), (3000, 12000, 4), (900, 7200, 5)])
def test_random_multigraphs(plan, n, m, seed):
    """From isolated vertices and small components to one dense whole."""
    row, col, _ = random_csr(n, m, seed)
    assert plan(row, col) == expected(row, col)


@pytest.mark.parametrize("degree,mean,cut", [(64, 2, True), (65, 2, False), (9, 8, True), (9, 9, False)])
def test_degrees(plan, degree, mean, cut):
    n = 2500
    rng = np.random.default_rng(degree)
    src = np.concatenate([np.full(degree, 700), np.repeat(np.setdiff1d(np.arange(n), [700]), mean)])
    if mean >= 8:   # exactly 8 n edges, or one more
        src = src[:8 * n + (0 if cut else 1)]
    dst = (src + rng.integers(1, 30, len(src))) % n
    order = np.lexsort((dst, src))
    row = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))])
    got = plan(row, dst[order])
    assert got == expected(row, dst[order]) and (got is not None) == cut
