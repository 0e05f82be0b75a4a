"""The watchdog of a launch lane's region solve, forced from the host by a limit
that short queries keep and a long one does not: requests that were over before
it are answered, exactly, only the others report the timeout, and the next
launches run on a clean ring.  Tolerance: none, distances are whole numbers."""
import sys

import numpy as np
import pytest

from mlmq_tpds_withl3_amd import HostGraph
from mlmq_tpds_withl3_amd.serve import Server
from oracle import oracle as O

pytestmark = pytest.mark.gpu
TIMED_OUT = -7


def say(msg):
    print(f"[gpu-serve-watchdog] {msg}", flush=True)
    sys.stdout.flush()


def test_finished_requests_outlive_the_watchdog():
    """A town takes about 0.1 ms, 3 million vertices from a corner 1.5 ms."""
    say("three towns beside a country, limit 0.5 ms")
    town = HostGraph.knn(2052, 3, seed=2, weight_scale=1e5)
    country = HostGraph.knn(3_000_000, 3, seed=3, weight_scale=-50_000.0, morton=True)
    arrays = [x.copy() for x in town.arrays()]
    s = Server(0, hbm_budget=4 << 30, timeout_s=0.5e-3, streams=1)
    s.add_graph(town)
    s.add_graph(country)
    src = np.array([5, 0, 1700, 900], dtype=np.int32)
    which = np.array([0, 1, 0, 0], dtype=np.int32)
    rows = [np.empty(town.n if g == 0 else country.n, dtype=np.int32) for g in which]
    expect = [O.dijkstra(*arrays, int(x))[0] for x in src[which == 0]]
    for turn in range(3):
        for r in rows:
            r[:] = -1
        res, _ = s.run(np.zeros(4), which, src, dist_out=rows)
        say(f"turn {turn}: status {res['status'].tolist()}")
        assert res["status"][1] == TIMED_OUT
        assert (res["status"][which == 0] == 0).all()
        for i, row in zip(np.flatnonzero(which == 0), expect):
            assert np.array_equal(rows[i], row), (turn, i)
        res, _ = s.run(np.zeros(3), np.zeros(3, dtype=np.int32), src[which == 0],
                       dist_out=[rows[i] for i in np.flatnonzero(which == 0)])
        assert (res["status"] == 0).all()
        for i, row in zip(np.flatnonzero(which == 0), expect):
            assert np.array_equal(rows[i], row), (turn, i)
    s.close()
