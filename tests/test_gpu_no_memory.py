"""Memory that runs out in the region or the push-pull solver: every allocation
of a load, a single query and a batch fails once, one after another.  Where the
vertex queue can do without it, it answers, exactly, with no memory of the other
solver still held, and the next call has that solver again.

Run in a process of its own: libhipallocfail.so has to be there before
libmlmq.so."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SHIM = os.path.join(HERE, "native", "libhipallocfail.so")


@pytest.mark.gpu
@pytest.mark.parametrize("name,what", [("road", "load"), ("power", "load"), ("road", "single"),
                                       ("power", "single"), ("road", "batch")])
def test_allocations_fail(name, what):
    print(f"[gpu-no-memory] {what} {name}", flush=True)
    if not os.path.exists(SHIM):
        raise RuntimeError(f"{SHIM} missing: build() compiles it")
    env = dict(os.environ, PYTHONPATH=os.pathsep.join([os.path.dirname(HERE), HERE]))
    done = subprocess.run([sys.executable, os.path.abspath(__file__), name, what], env=env, timeout=100,
                          capture_output=True, text=True)
    assert done.returncode == 0, done.stdout[-2000:] + done.stderr[-2000:]


def main(name, what):
    shim = ctypes.CDLL(SHIM, mode=ctypes.RTLD_GLOBAL)
    shim.alloc_live.restype = ctypes.c_size_t
    from mlmq_tpds_withl3_amd import HostGraph, MLMQError, Solver
    from oracle import oracle as O

    if name == "road":
        g = HostGraph.knn(5000, 3, seed=2, weight_scale=1e5)
    else:
        g = HostGraph.rmat(13, 16, seed=9, wmin=1, wmax=1000)
    row, col, w = (x.copy() for x in g.arrays())
    g.close()
    sources = [7, 900, 33]
    rows = [O.dijkstra(row, col, w, x)[0] for x in sources]

    def loaded():
        s = Solver(0)
        s.load_csr(row, col, w)
        return s

    def solver_of(t):   # waves of a workgroup: 1 is the vertex queue
        return t["waves"] // t["work_blocks"]

    def single(s, **params):
        t = s.solve(sources[0], timeout_s=20.0, **params)
        assert np.array_equal(s.dist(), rows[0])
        return solver_of(t)

    def batch(s, **params):
        t = s.solve_batch(sources, timeout_s=20.0, **params)
        for i, r in enumerate(rows):
            assert np.array_equal(s.batch_dist(i), r), i
        return t["graph_replay"]   # only the vertex queue's launch is a graph

    call = {"single": single, "batch": batch}.get(what)
    s = loaded()
    usual = single(s)
    assert usual in (6, 8, 10)
    usual = {"load": usual, "single": usual, "batch": batch(s)}[what]
    s.close()
    if call:
        # the queue's own memory: a call that its settings give to the queue
        # with the rings it takes by itself
        s = loaded()
        assert call(s, bucket_capacity=8192) == 1
        queue_bytes = shim.alloc_live()
        s.close()

    refused, answered = [], []
    for k in range(64):
        s = loaded() if call else Solver(0)
        print(f"{what} {name}: allocation {k} fails", flush=True)
        shim.alloc_fail_after(k)
        try:
            if call:
                by = call(s)
            else:
                s.load_csr(row, col, w)
            if shim.alloc_failures() == 0:
                shim.alloc_fail_after(-1)
                s.close()
                break
            answered.append(k)
            if call:
                assert by == 1, by
                assert shim.alloc_live() == queue_bytes, (shim.alloc_live(), queue_bytes)
                assert call(s) == usual
            else:
                assert single(s) in (1, usual)
        except MLMQError as e:
            assert shim.alloc_failures() == 1 and e.code == -4, e
            refused.append(k)
        s.close()
    else:
        raise AssertionError("no end to the allocations")
    print(f"{what} {name}: refused {refused}, answered {answered}", flush=True)
    # refused: what every solver needs (the graph, its hop blocks and the table
    # of its hubs; the row; the rows, sources, status, times and counter of a
    # batch)
    hubs = int((np.diff(row) > 2048).any())
    needed = {"load": 4 + hubs, "single": 1, "batch": 5}[what]
    assert refused == list(range(needed))
    assert answered


if __name__ == "__main__":
    main(*sys.argv[1:3])
