"""Which solver answers a single query, and on how many workgroups: a chosen
number of workgroups below the number of CUs (256) bounds the region and the
push-pull solver too, from there on they take what they need; with fewer
workgroups than a 32nd of a graph's regions the vertex queue answers.  The
timing tells the solver by the waves of a workgroup: one (vertex queue), six or
ten (regions), eight (push-pull).  Also the limits of a region (384 exits and
384 inbox slots), the largest packed weight, and what a solver counts.  Every row is compared with the oracle, bit
for bit."""
import sys

import numpy as np
import pytest

from mlmq_tpds_withl3_amd import HostGraph, Solver
from oracle import oracle as O
from test_region_plan import expected

pytestmark = pytest.mark.gpu
TIMEOUT = 20.0
CUS = 256


def say(msg):
    print(f"[gpu-solver-choice] {msg}", flush=True)
    sys.stdout.flush()


def arrays(g):
    out = tuple(x.copy() for x in g.arrays())
    g.close()
    return out


@pytest.fixture(scope="module")
def loaded():
    """A road-like graph of 70 regions and a power-law graph, resident."""
    graphs = {"road": arrays(HostGraph.knn(70_001, 3, seed=4, weight_scale=1e5)),
              "power": arrays(HostGraph.rmat(13, 16, seed=9, wmin=1, wmax=1000))}
    out = {}
    for name, g in graphs.items():
        s = Solver(0)
        s.load_csr(*g)
        out[name] = (s, g)
    yield out
    for s, _ in out.values():
        s.close()


def solve(loaded, name, src, **params):
    s, g = loaded[name]
    t = s.solve(src, timeout_s=TIMEOUT, **params)
    assert np.array_equal(s.dist(), O.dijkstra(*g, src)[0])
    return t["work_blocks"], t["waves"] // t["work_blocks"]


@pytest.mark.parametrize("blocks", [2, 3, 64, CUS - 1])
def test_chosen_workgroups_bound_the_regions(loaded, blocks):
    say(f"regions on {blocks} workgroups")
    free, _ = solve(loaded, "road", 11)
    used, waves = solve(loaded, "road", 11, work_blocks=blocks)
    assert waves in (6, 10) and used == min(blocks, free)


def test_few_workgroups_for_many_regions(loaded):
    say("one workgroup for 70 regions: the vertex queue")
    assert solve(loaded, "road", 11, work_blocks=1) == (1, 1)


@pytest.mark.parametrize("blocks", [1, 7, 64, CUS - 1])
def test_chosen_workgroups_bound_the_push_pull_rounds(loaded, blocks):
    say(f"push-pull on {blocks} workgroups")
    free, _ = solve(loaded, "power", 5)
    assert solve(loaded, "power", 5, work_blocks=blocks) == (min(blocks, free), 8)


@pytest.mark.parametrize("name", ["road", "power"])
def test_one_workgroup_per_cu_is_no_bound(loaded, name):
    say(f"{name}: one workgroup per CU or more")
    free = solve(loaded, name, 3)
    assert solve(loaded, name, 3, work_blocks=CUS) == free
    assert solve(loaded, name, 3, work_blocks=2 * CUS) == free


@pytest.mark.parametrize("top,waves", [((1 << 20) - 2, 10), ((1 << 20) - 1, 1)])
def test_weight_of_the_absent_edge(top, waves):
    """The region solver's packed edges keep one weight for edges that are not
    there: a graph with that weight is not cut, and every examined edge counts."""
    say(f"weights of {top}")
    n = 1500
    a = np.arange(n - 1)
    src, dst = np.concatenate([a, a + 1]), np.concatenate([a + 1, a])
    order = np.lexsort((dst, src))
    row = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]).astype(np.int64)
    g = (row, dst[order].astype(np.int32), np.full(len(order), top, dtype=np.int32))
    with Solver(0) as s:
        s.load_csr(*g)
        t = s.solve(700, timeout_s=TIMEOUT)
        dist, work, _ = O.dijkstra(*g, 700)
        assert np.array_equal(s.dist(), dist)
        assert t["waves"] == waves * t["work_blocks"] and t["relaxations"] >= work


@pytest.mark.parametrize("nq", [3, 64])
def test_batch_reports_its_queries_in_flight(loaded, nq):
    """A batch on the region solver admits a few queries at a time (70 regions
    each: about a thirtieth of its at most 1024 or, for few queries, 512
    workgroups, all of them where these are more than the queries)."""
    say(f"batch of {nq}: queries in flight")
    s, g = loaded["road"]
    src = np.random.default_rng(nq).integers(0, 70_001, nq).astype(np.int32)
    t = s.solve_batch(src, timeout_s=TIMEOUT)
    for i in (0, nq // 2, nq - 1):
        assert np.array_equal(s.batch_dist(i), O.dijkstra(*g, int(src[i]))[0])
    assert t["graph_replay"] == 0
    in_flight = int(1024 * 0.27 / 70 ** 0.5) if nq == 64 else 3
    assert t["work_blocks"] == in_flight
    # 1024 workgroups of six waves, or three times 70 of ten
    waves = 6 * 1024 if nq == 64 else 10 * 210
    assert t["waves_per_query"] == waves // in_flight


def block_with_exits(exits, entries):
    """Consecutive blocks of 1024 vertices, each a chain, of which the first has
    exactly so many edges out of it and into it."""
    n = 40 * 1024
    a = np.arange(n - 1)
    a = a[(a + 1) % 1024 != 0]
    far = np.arange(2048, n, 61)
    src = np.concatenate([a, a + 1, a, np.arange(exits) % 1024, far[:entries]])
    dst = np.concatenate([a + 1, a, a + 1, far[:exits], np.arange(entries) % 1024])
    w = np.random.default_rng(exits + entries).integers(1, 1000, len(src))
    order = np.lexsort((dst, src))
    row = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]).astype(np.int64)
    return row, dst[order].astype(np.int32), w[order].astype(np.int32)


@pytest.mark.parametrize("exits,entries,waves", [(384, 384, 10), (385, 10, 1), (10, 385, 1)])
def test_limits_of_a_region(exits, entries, waves):
    say(f"a region of {exits} exits and {entries} inbox slots")
    g = block_with_exits(exits, entries)
    with Solver(0) as s:
        s.load_csr(*g)
        for src in (0, 700, 5000):
            t = s.solve(src, timeout_s=TIMEOUT)
            assert np.array_equal(s.dist(), O.dijkstra(*g, src)[0])
            assert t["waves"] == waves * t["work_blocks"]


def test_push_pull_counts(loaded):
    """Every reached vertex but the source is lowered and queued at least once,
    each over an edge that is examined."""
    say("push-pull counts")
    s, g = loaded["power"]
    for src in (0, 5, 77):
        t = s.solve(src, timeout_s=TIMEOUT)
        dist = s.dist()
        reached = int((dist < 0x7FFFFFFF).sum())
        assert reached > 1000 and t["waves"] == 8 * t["work_blocks"]
        assert t["improvements"] >= reached - 1 and t["relaxations"] >= t["improvements"]
        assert t["l2_pushes"] >= reached


@pytest.mark.parametrize("far,waves", [(100, 10), (120, 1)])
def test_share_of_crossing_edges(far, waves):
    """One-way chains of 1024 with edges to anywhere: 10.3 and 12.2 % of the edges
    cross between the grown regions, which have up to 211 exits and slots."""
    say(f"{far} far edges per chain")
    n = 12 * 1024
    rng = np.random.default_rng(1)
    a = np.arange(n - 1)
    a = a[(a + 1) % 1024 != 0]
    tail = np.repeat(np.arange(12), far) * 1024 + rng.integers(0, 1024, 12 * far)
    src = np.concatenate([a, tail])
    dst = np.concatenate([a + 1, rng.integers(0, n, 12 * far)])
    order = np.lexsort((dst, src))
    row = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]).astype(np.int64)
    col = dst[order].astype(np.int32)
    region = np.empty(n, dtype=int)
    for i, r in enumerate(expected(row, col)):
        region[r] = i
    share = (region[np.repeat(np.arange(n), np.diff(row))] != region[col]).mean()
    assert (share <= 0.12) == (waves == 10)
    w = rng.integers(1, 1000, len(col)).astype(np.int32)
    with Solver(0) as s:
        s.load_csr(row, col, w)
        for x in (0, 5000, n - 1):
            t = s.solve(x, timeout_s=TIMEOUT)
            assert np.array_equal(s.dist(), O.dijkstra(row, col, w, x)[0])
            assert t["waves"] == waves * t["work_blocks"]
