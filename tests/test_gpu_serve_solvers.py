"""Requests of the launch lanes through the region and the push-pull solver:
every row against the oracle, bit for bit, alone and mixed in one launch with
requests of the vertex queue; the slots change hands between the solvers; a
power-law graph with a tail of more rounds than a lane runs goes to the vertex
queue as a rerun.  Tolerance: none, distances are whole numbers."""
import sys

import numpy as np
import pytest

from graphs_util import random_csr
from mlmq_tpds_withl3_amd import HostGraph
from mlmq_tpds_withl3_amd.serve import Server
from oracle import oracle as O

pytestmark = pytest.mark.gpu
TIMEOUT = 20.0


def say(msg):
    print(f"[gpu-serve-solvers] {msg}", flush=True)
    sys.stdout.flush()


def arrays(g):
    out = tuple(x.copy() for x in g.arrays())
    g.close()
    return out


def with_tail(graph, length):
    """The graph with a path of `length` new vertices hung on vertex 0."""
    row, col, w = graph
    n = len(row) - 1
    src = np.repeat(np.arange(n), np.diff(row))
    path = np.concatenate([[0], n + np.arange(length)])
    a = np.concatenate([src, path[:-1], path[1:]])
    b = np.concatenate([col, path[1:], path[:-1]])
    x = np.concatenate([w, np.full(2 * length, 5)])
    order = np.lexsort((b, a))
    r = np.zeros(n + length + 1, dtype=np.int64)
    np.add.at(r, a + 1, 1)
    return np.cumsum(r), b[order].astype(np.int32), x[order].astype(np.int32)


@pytest.fixture(scope="module")
def graphs():
    rmat = arrays(HostGraph.rmat(12, 16, seed=9, wmin=1, wmax=1000))
    return {"road": arrays(HostGraph.knn(50_021, 3, seed=1, weight_scale=1e5)),
            "town": arrays(HostGraph.knn(2_052, 3, seed=2, weight_scale=1e5)),
            "power": rmat, "tail": with_tail(rmat, 100),
            "random": random_csr(3000, 24000, seed=11, wmax=1000)}


def serve(graphs, requests, arrival=None, retries=0, settings=None, **cfg):
    names = sorted({name for name, _ in requests})
    with_rows = [np.empty(len(graphs[name][0]) - 1, dtype=np.int32) for name, _ in requests]
    s = Server(0, hbm_budget=1 << 30, timeout_s=TIMEOUT, **cfg)
    for name in names:
        s.add_graph(graphs[name], **(settings or {}).get(name, {}))
    which = np.array([names.index(name) for name, _ in requests], dtype=np.int32)
    src = np.array([x for _, x in requests], dtype=np.int32)
    expect = [O.dijkstra(*graphs[name], int(x))[0] for name, x in requests]
    for g, x, row in zip(which, src, expect):
        s.set_expected(int(g), int(x), row)
    at = np.zeros(len(requests)) if arrival is None else arrival
    for turn in range(3):   # the second and third on used slots
        for row in with_rows:
            row[:] = -1
        res, st = s.run(at, which, src, dist_out=with_rows)
        assert (res["status"] == 0).all(), res["status"]
        assert (res["mismatches"] == 0).all()
        assert res["retries"].sum() == retries
        assert (res["device_ms"] > 0).all()
        for i, row in enumerate(expect):
            assert np.array_equal(with_rows[i], row), (turn, requests[i])
    s.close()


@pytest.mark.parametrize("name", ["road", "town", "power"])
@pytest.mark.parametrize("count", [1, 2, 33])
def test_one_graph(graphs, name, count):
    say(f"{count} x {name}")
    n = len(graphs[name][0]) - 1
    serve(graphs, [(name, int(x)) for x in np.linspace(0, n - 1, count).astype(int)])


@pytest.mark.parametrize("streams,batch,spacing", [(1, 64, 0.0), (4, 3, 0.0), (3, 8, 0.0002)])
def test_mixed(graphs, streams, batch, spacing):
    say(f"mixed, {streams} lanes of {batch}")
    rng = np.random.default_rng(4)
    requests = [(name, int(rng.integers(0, 2000))) for name in ["road", "power", "random", "town"] * 6]
    serve(graphs, requests, arrival=np.arange(len(requests)) * spacing, streams=streams, max_batch=batch)


def test_light_split(graphs):
    say("light/heavy split: push-pull solver and vertex queue")
    split = dict(light_split=1, delta=100, buckets=32)
    serve(graphs, [("power", 1), ("road", 2), ("power", 3)], settings={"power": split, "road": split})


def test_long_tail(graphs):
    say("a tail beyond the lane's rounds")
    serve(graphs, [("tail", 5), ("power", 5), ("road", 5)], retries=1)
