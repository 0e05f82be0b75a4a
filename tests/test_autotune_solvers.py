"""Host logic of the parameter search (no GPU) on graphs that the region or the
push-pull solver answers: settings that mean nothing to them are not searched,
and a serving tuner scores what the vertex queue gets."""
import numpy as np

from mlmq_tpds_withl3_amd import autotune as A


class FakeSolver:
    """Another solver answers, unless light_split is set; its time depends on
    work_blocks alone, the queue's also on delta."""

    def __init__(self, batch_by_regions=True):
        self.seen = []
        self.batch_by_regions = batch_by_regions

    def solve(self, src, p):
        self.seen.append((p.work_blocks, p.light_split, p.delta))
        blocks = max(1, p.work_blocks)
        if p.light_split:
            return {"device_ms": 1.0 + p.delta / 100, "waves": blocks, "work_blocks": blocks}
        return {"device_ms": 2.0 - blocks / 1024, "waves": 10 * blocks, "work_blocks": blocks}

    def solve_batch(self, sources, p):
        self.seen.append(p.delta)
        return {"graph_replay": 0 if self.batch_by_regions else 1}


def test_tune_single_leaves_out_what_means_nothing():
    s = FakeSolver()
    r = A.tune_single(s, 0, (100, 200, 400), repeats=1, confirm=1)
    # four grid sizes of the default grid, once each, and the four confirmed
    assert [x[0] for x in s.seen[:4]] == [192, 256, 384, 512] and len(s.seen) == 8
    assert r["params"]["work_blocks"] == 512


def test_tune_single_searches_what_the_queue_answers():
    s = FakeSolver()
    grid = [dict(light_split=ls, work_blocks=256) for ls in (1, 0)]
    r = A.tune_single(s, 0, (10, 20, 40), grid=grid, repeats=1, confirm=1)
    table = [(p["light_split"], p["delta"]) for p, _ in r["table"] if "stale_check" not in p and "prefetch" not in p]
    assert table == [(1, 10), (0, 10), (1, 20), (1, 40)]
    assert r["params"]["light_split"] == 1 and r["params"]["delta"] == 10


def test_tune_batch_returns_at_once_where_regions_answer():
    s = FakeSolver()
    r = A.tune_batch(s, np.arange(4), base=dict(delta=300))
    assert set(s.seen) == {300} and r["params"]["delta"] == 300
    s = FakeSolver(batch_by_regions=False)
    A.tune_batch(s, np.arange(4), base=dict(delta=300))
    assert len(set(s.seen)) > 1


class FakeServer:
    """Regions answer unless a bucket capacity is given: then the rate depends on
    delta, otherwise on nothing but the order of the calls."""

    def __init__(self):
        self.sizes = [(640_000, 2_400_000)]
        self.params = {}
        self.rate = 5000.0

    def set_graph_params(self, gid, **params):
        self.params = dict(params)

    def run(self, arrival, graph, src):
        n = len(arrival)
        queue = "bucket_capacity" in self.params
        assert not queue or self.params["bucket_capacity"] == 20_000
        res = np.zeros(n, dtype=[("latency_ms", "f8"), ("solver", "i4")])
        res["solver"] = 0 if queue else 1
        self.rate += 1.0
        qps = 1000.0 - abs(np.log2(self.params["delta"] / 50_000)) if queue else self.rate
        return res, {"completed": n, "mismatched": 0, "completed_qps": qps}


def test_tune_serving_scores_the_queue():
    srv = FakeServer()
    r = A.tune_serving(srv, 0, np.arange(10), base=dict(delta=200_000), repeats=1)
    assert r["params"]["delta"] == 50_000
    assert srv.params == r["params"] and "bucket_capacity" not in srv.params
    assert {k for k in r["params"] if r["params"][k] != {"prefetch": 1, "stale_check": 2}.get(k)} == {"delta"}
