"""Which solver answers a request of a launch lane, as its result says, at the
edges of the rules: settings and slots that only the vertex queue fits, requests
of other lanes in flight (32 or more: the queue), the buffer that push-pull
states too large for their slots share (a 64th of the slot arena), and reruns.
Every row is compared with the oracle, bit for bit."""
import sys

import numpy as np
import pytest

from graphs_util import random_csr
from mlmq_tpds_withl3_amd import HostGraph
from mlmq_tpds_withl3_amd._lib import SERVE_SOLVERS
from mlmq_tpds_withl3_amd.serve import Server
from oracle import oracle as O
from test_gpu_serve_solvers import with_tail

pytestmark = pytest.mark.gpu
TIMEOUT = 20.0


def say(msg):
    print(f"[gpu-serve-choice] {msg}", flush=True)
    sys.stdout.flush()


def arrays(g):
    out = tuple(x.copy() for x in g.arrays())
    g.close()
    return out


@pytest.fixture(scope="module")
def graphs():
    return {"road": arrays(HostGraph.knn(20_011, 3, seed=1, weight_scale=1e5)),
            "dense": arrays(HostGraph.knn(150_001, 4, seed=3, weight_scale=1e5)),
            "power": arrays(HostGraph.rmat(14, 16, seed=9, wmin=1, wmax=1000)),
            "random": random_csr(3000, 24000, seed=11, wmax=1000)}


def serve(graphs, requests, settings=None, **cfg):
    """Solvers and reruns of the requests (graph, source), in their order."""
    s = Server(0, timeout_s=TIMEOUT, **cfg)
    names = list(dict.fromkeys(name for name, _ in requests))
    for name in names:
        s.add_graph(graphs[name], **(settings or {}))
    rows = [np.empty(len(graphs[name][0]) - 1, dtype=np.int32) for name, _ in requests]
    res, _ = s.run(np.zeros(len(requests)), [names.index(name) for name, _ in requests],
                   [x for _, x in requests], dist_out=rows)
    s.close()
    assert (res["status"] == 0).all()
    expect = {}
    for r, row in zip(requests, rows):
        if r not in expect:
            expect[r] = O.dijkstra(*graphs[r[0]], r[1])[0]
        assert np.array_equal(row, expect[r]), r
    return [SERVE_SOLVERS[k] for k in res["solver"]], res["retries"].tolist()


@pytest.mark.parametrize("settings,road,power", [
    ({}, "regions", "push-pull"), (dict(light_split=1, delta=100, buckets=32), "queue", "push-pull"),
    (dict(hub_split=1), "queue", "queue"), (dict(bucket_capacity=1 << 16), "queue", "queue")])
def test_settings(graphs, settings, road, power):
    say(f"settings {settings}")
    requests = [("road", 1), ("power", 2), ("random", 3), ("road", 400)]
    got, _ = serve(graphs, requests, settings, hbm_budget=1 << 30)
    assert got == [road, power, "queue", road]


@pytest.mark.parametrize("buckets,solver", [(16, "regions"), (1, "queue")])
def test_inboxes_that_do_not_fit_the_slot(graphs, buckets, solver):
    """About 30,000 inbox slots of 4 bytes; a bucket has 8192 ring slots of 8."""
    say(f"{buckets} buckets")
    got, _ = serve(graphs, [("dense", 7), ("dense", 100_000)], dict(buckets=buckets, bucket_window=1),
                   hbm_budget=1 << 30)
    assert got == [solver, solver]


@pytest.mark.parametrize("batch,second", [(31, "regions"), (32, "queue")])
def test_crowded_lanes(graphs, batch, second):
    """A burst of two launches: the second starts with the first in flight."""
    say(f"two lanes of {batch}")
    requests = [("road", 11 * (i % 9)) for i in range(2 * batch)]
    got, _ = serve(graphs, requests, streams=2, max_batch=batch, hbm_budget=1 << 30)
    assert got == ["regions"] * batch + [second] * batch


def test_push_pull_states_beside_their_slots(graphs):
    """16,384 vertices: 12 bytes each and 4 KiB of counters, 200,712 bytes, in a
    slot with one ring of 64 KiB.  A 64th of 64 MiB holds five."""
    say("push-pull states in the lane's buffer")
    requests = [("power", 5 + i) for i in range(8)]
    got, _ = serve(graphs, requests, dict(buckets=1, bucket_window=1), streams=1, hbm_budget=64 << 20)
    assert got == ["push-pull"] * 5 + ["queue"] * 3


def test_reruns(graphs):
    say("a tail beyond the lane's rounds")
    mix = dict(graphs, tail=with_tail(graphs["power"], 100))
    got, retries = serve(mix, [("tail", 5), ("power", 5), ("road", 5)], hbm_budget=1 << 30)
    assert got == ["queue", "push-pull", "regions"] and retries == [1, 0, 0]
