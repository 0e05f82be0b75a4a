"""The region solver (graphs cut into LDS-sized regions of up to 1024 vertices)
against the oracle, bit for bit, at the sizes where it can go wrong: region
sizes around 1024, more than eight edges per vertex, weights at the packed
limit, one-way and zero-weight edges, separate components, and batches with
more regions than the device serves at once (regions are left and adopted
again).  The timing tells which solver ran: the region solver reports six or ten
waves per workgroup.  Tolerance: none, distances are whole numbers."""
import sys

import numpy as np
import pytest

from mlmq_tpds_withl3_amd import HostGraph, Solver
from oracle import oracle as O

pytestmark = pytest.mark.gpu
TIMEOUT = 20.0


def say(msg):
    print(f"[gpu-regions] {msg}", flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def solver():
    s = Solver(0)
    yield s
    s.close()


def csr(n, src, dst, w):
    order = np.lexsort((dst, src))
    src, dst, w = np.asarray(src)[order], np.asarray(dst)[order], np.asarray(w)[order]
    row = np.zeros(n + 1, dtype=np.int64)
    np.add.at(row, src + 1, 1)
    return np.cumsum(row), dst.astype(np.int32), w.astype(np.int32)


def strip(n, reach, seed, wmax=1000, one_way=0.0, zero=0.0):
    """A long strip: edges from each vertex to a few of the next `reach` ones."""
    rng = np.random.default_rng(seed)
    src, dst, w = [], [], []
    for u in range(n):
        for v in {u + 1, u + int(rng.integers(1, reach + 1))}:
            if v >= n:
                continue
            x = 0 if rng.random() < zero else int(rng.integers(1, wmax + 1))
            src.append(u), dst.append(v), w.append(x)
            if rng.random() >= one_way:
                src.append(v), dst.append(u), w.append(x)
    return csr(n, np.array(src, dtype=np.int64), np.array(dst, dtype=np.int64), np.array(w, dtype=np.int64))


def check(solver, graph, sources, regions, **params):
    row, col, w = graph
    solver.load_csr(row, col, w)
    for src in sources:
        t = solver.solve(int(src), timeout_s=TIMEOUT, **params)
        ref, work, _ = O.dijkstra(row, col, w, int(src))
        bad = np.flatnonzero(solver.dist() != ref)
        assert bad.size == 0, f"source {src}: {bad.size} mismatches, first v={bad[0]}"
        assert (t["waves"] in (6 * t["work_blocks"], 10 * t["work_blocks"])) == regions
        assert t["relaxations"] >= work
        q = solver.queue_counts()
        assert q["writes"] == q["reads"] and sum(q["writes"]) == q["completed"] == t["l2_pushes"]


@pytest.mark.parametrize("n", [2, 63, 257, 1023, 1024, 1025, 2049, 5000])
def test_region_sizes(solver, n):
    say(f"strip of {n}")
    check(solver, strip(n, 6, n), {0, n - 1, n // 2}, True)


@pytest.mark.parametrize("kw", [dict(one_way=0.5), dict(zero=0.4), dict(one_way=1.0, zero=0.2)])
def test_one_way_and_zero_weights(solver, kw):
    say(f"strip {kw}")
    check(solver, strip(6000, 8, 3, **kw), (0, 17, 3000, 5999), True)


def test_renumbered_and_separate_components(solver):
    say("shuffled ids, components")
    parts = [strip(1500, 5, s) for s in (1, 2, 3)]
    row = np.concatenate([[0]] + [p[0][1:] + k for p, k in zip(parts, np.cumsum([0] + [len(p[1]) for p in parts]))])
    col = np.concatenate([p[1] + 1500 * i for i, p in enumerate(parts)])
    w = np.concatenate([p[2] for p in parts])
    n = len(row) - 1
    perm = np.random.default_rng(5).permutation(n)
    src = np.repeat(np.arange(n), np.diff(row))
    check(solver, csr(n, perm[src], perm[col], w), (0, 1, 4000), True)


def test_many_edges_per_vertex(solver):
    """Vertices of up to 24 edges: all but eight go through the region's own
    inbox; a vertex beyond 64 edges, or a mean beyond 8, is not cut."""
    say("degrees past eight")
    rng = np.random.default_rng(8)
    n = 3000
    src, dst = [np.arange(n - 1)], [np.arange(1, n)]
    for u in range(0, n - 40, 50):
        k = int(rng.integers(8, 24))
        src.append(np.full(k, u))
        dst.append(u + rng.integers(1, 40, size=k))
    a, b = np.concatenate(src), np.concatenate(dst)
    w = rng.integers(1, 500, size=len(a))
    g = csr(n, np.concatenate([a, b]), np.concatenate([b, a]), np.concatenate([w, w]))
    assert np.diff(g[0]).max() > 8
    check(solver, g, (0, 1234, 2999), True)
    hub = csr(n, np.concatenate([a, np.zeros(100, int)]), np.concatenate([b, np.arange(100, 200)]),
              np.concatenate([w, np.ones(100, int)]))
    check(solver, hub, (0, 5), False)


@pytest.mark.parametrize("top,regions", [((1 << 20) - 2, True), (1 << 20, False), ((1 << 31) - 1, False)])
def test_weight_limit(solver, top, regions):
    say(f"largest weight {top}")
    row, col, w = strip(2500, 6, 4)
    w = w.copy()
    w[len(w) // 2] = w[7] = top
    check(solver, (row, col, w), (0, 2499), regions)


def test_distances_near_the_end_of_range(solver):
    """A chain whose distances pass INT_MAX: those vertices stay unreached."""
    say("distances past the range")
    n = 2600
    g = csr(n, np.arange(n - 1), np.arange(1, n), np.full(n - 1, (1 << 20) - 2))
    row, col, w = g
    solver.load_csr(row, col, w)
    t = solver.solve(0, timeout_s=TIMEOUT)
    d = np.arange(n, dtype=np.int64) * ((1 << 20) - 2)
    assert t["waves"] == 10 * t["work_blocks"]
    assert np.array_equal(solver.dist(), np.where(d < 0x7FFFFFFF, d, 0x7FFFFFFF).astype(np.int32))


@pytest.mark.parametrize("n,nq", [(1000, 1), (5000, 7), (40_000, 64), (2500, 1500)])
def test_batches(solver, n, nq):
    """40 regions x 64 queries: more than the device serves at once."""
    say(f"batch of {nq} over {n} vertices")
    g = HostGraph.knn(n, 3, seed=n, weight_scale=1e5)
    row, col, w = (x.copy() for x in g.arrays())
    solver.load_csr(row, col, w)
    src = np.random.default_rng(nq).integers(0, n, size=nq)
    for rep in range(2):
        t = solver.solve_batch(src, timeout_s=TIMEOUT)
        assert t["queries"] == nq and t["relaxations"] > 0 and t["query_ms_max"] > 0
        for i in range(0, nq, max(1, nq // 40)):
            assert np.array_equal(solver.batch_dist(i), O.dijkstra(row, col, w, int(src[i]))[0]), f"query {i}"
    solver.solve(int(src[0]), timeout_s=TIMEOUT)
    assert np.array_equal(solver.dist(), O.dijkstra(row, col, w, int(src[0]))[0])


def test_stopped_solve_leaves_a_clean_solver(solver):
    """A solve stopped by the watchdog (every workgroup sees its deadline
    passed and returns), then the same query without one."""
    say("watchdog, then a good solve")
    row, col, w = strip(9000, 6, 9)
    solver.load_csr(row, col, w)
    for _ in range(2):
        with pytest.raises(Exception) as e:
            solver.solve(3, timeout_s=1e-7)
        assert e.value.code == -7
        solver.solve(3, timeout_s=TIMEOUT)
        assert np.array_equal(solver.dist(), O.dijkstra(row, col, w, 3)[0])


@pytest.mark.parametrize("nq", [199, 200])
def test_large_batches(solver, nq):
    """Around the size from which a batch on a large graph goes to the vertex
    queue (200 queries, 384 regions)."""
    say(f"{nq} queries on 400k vertices")
    g = HostGraph.knn(400_000, 3, seed=3, weight_scale=1e5, morton=True)
    row, col, w = (x.copy() for x in g.arrays())
    g.close()
    solver.load_csr(row, col, w)
    src = np.random.default_rng(nq).integers(0, 400_000, nq).astype(np.int32)
    solver.solve_batch(src, timeout_s=TIMEOUT)
    for i in (0, nq // 2, nq - 1):
        assert np.array_equal(solver.batch_dist(i), O.dijkstra(row, col, w, int(src[i]))[0]), i
