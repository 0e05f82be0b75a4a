"""The push-pull solver (undirected graphs of strongly varying degree) against
the oracle, bit for bit: degrees around the hop block's seven edges and the
wave's and workgroup's widths, zero, equal and very large weights, separate
parts, a tail of more rounds than the solver launches blindly, a tail longer
than it is meant for (the vertex queue answers), and directed graphs (never
taken).  It reports eight waves per workgroup.  Tolerance: none, distances are
whole numbers."""
import sys

import numpy as np
import pytest

from mlmq_tpds_withl3_amd import HostGraph, Solver
from oracle import oracle as O

pytestmark = pytest.mark.gpu
TIMEOUT = 20.0


def say(msg):
    print(f"[gpu-pushpull] {msg}", flush=True)
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


def both_ways(n, a, b, w):
    return csr(n, np.concatenate([a, b]), np.concatenate([b, a]), np.concatenate([w, w]))


def hubs(n, degrees, per_vertex, seed, weights):
    """Random edges plus hubs of the given degrees, each edge both ways."""
    rng = np.random.default_rng(seed)
    a = [rng.integers(0, n, size=per_vertex * n)]
    for h, d in enumerate(degrees):
        a.append(np.full(d, h))
    a = np.concatenate(a)
    b = rng.integers(0, n, size=len(a))
    return both_ways(n, a, b, weights(rng, len(a)))


def check(solver, graph, sources, taken, **params):
    row, col, w = graph
    solver.load_csr(row, col, w)
    for src in sources:
        t = solver.solve(int(src), timeout_s=TIMEOUT, **params)
        ref, _, _ = O.dijkstra(row, col, w, int(src))
        bad = np.flatnonzero(solver.dist() != ref)
        assert bad.size == 0, f"source {src}: {bad.size} mismatches, first v={bad[0]}"
        assert (t["waves"] == 8 * t["work_blocks"]) == taken
        q = solver.queue_counts()
        assert q["writes"] == q["reads"] and sum(q["writes"]) == q["completed"] == t["l2_pushes"]


DEGREES = [5000, 4096, 2049, 1025, 1024, 1023, 513, 257, 256, 255, 129, 65, 64, 63, 8, 7]
WEIGHTS = {
    "uniform": lambda rng, k: rng.integers(1, 1001, size=k),
    "zeros": lambda rng, k: rng.integers(0, 3, size=k),
    "equal": lambda rng, k: np.full(k, 7),
    "huge": lambda rng, k: rng.integers(1 << 27, 1 << 30, size=k),   # hop blocks without back edges
}


@pytest.mark.parametrize("weights", list(WEIGHTS))
def test_degrees_and_weights(solver, weights):
    say(f"hubs, {weights} weights")
    check(solver, hubs(6000, DEGREES * 2, 2, 5, WEIGHTS[weights]), (0, 3, 15, 31, 5999), True)


@pytest.mark.parametrize("scale,factor", [(8, 2), (10, 4), (13, 16), (15, 9)])
@pytest.mark.parametrize("settings", [{}, dict(light_split=1, delta=50, buckets=64, bucket_window=2, l1_pop=64)])
def test_power_law(solver, scale, factor, settings):
    say(f"rmat {scale} {factor} {settings}")
    g = HostGraph.rmat(scale, factor, seed=scale)
    row, col, w = (x.copy() for x in g.arrays())
    if g.m >= 4 * g.n:
        hub = g.max_degree_vertex()
        leaf = int(np.flatnonzero(np.diff(row) == np.diff(row)[np.diff(row) > 0].min())[0])
        alone = np.flatnonzero(np.diff(row) == 0)
        check(solver, (row, col, w), [hub, leaf, *alone[:1]], True, **settings)
    else:
        check(solver, (row, col, w), [g.max_degree_vertex()], False, **settings)


@pytest.mark.parametrize("tail,taken", [(40, True), (600, True), (3000, False)])
def test_long_tails(solver, tail, taken):
    """A chain hangs off the graph: more rounds than are launched at once, then
    more than the solver goes on for."""
    say(f"tail of {tail}")
    row, col, w = hubs(6000, DEGREES * 2, 2, 6, WEIGHTS["uniform"])
    a = np.repeat(np.arange(6000), np.diff(row))
    keep = a < col
    chain = np.arange(6000 + tail - 1)[5999:]
    g = both_ways(6000 + tail, np.concatenate([a[keep], chain]), np.concatenate([col[keep], chain + 1]),
                  np.concatenate([w[keep], np.full(len(chain), 900)]))
    check(solver, g, (0, 6000 + tail - 1), taken)


def test_directed_graphs_are_not_taken(solver):
    say("one edge without its reverse")
    row, col, w = hubs(6000, DEGREES * 2, 2, 7, WEIGHTS["uniform"])
    a = np.repeat(np.arange(6000), np.diff(row))
    check(solver, (row, col, w), (0,), True)
    one = csr(6000, np.append(a, 4000), np.append(col, 17), np.append(w, 3))
    check(solver, one, (0, 4000, 17), False)
    other = w.copy()
    other[row[5000]] += 1   # the same edges, one weight differs between the directions
    check(solver, (row, col, other), (0, 5000), False)


def test_stopped_solve_leaves_a_clean_solver(solver):
    say("watchdog, then a good solve")
    row, col, w = hubs(6000, DEGREES * 2, 2, 8, WEIGHTS["uniform"])
    solver.load_csr(row, col, w)
    with pytest.raises(Exception) as e:
        solver.solve(0, timeout_s=1e-7)
    assert e.value.code == -7
    with pytest.raises(Exception):
        solver.dist()
    solver.solve(0, timeout_s=TIMEOUT)
    assert np.array_equal(solver.dist(), O.dijkstra(row, col, w, 0)[0])
