"""The vertex queue on the graphs that the region and the push-pull solver answer
by themselves: it still serves live requests, allocation-free queries, crowded
lanes, large batches and whatever those two give up.  The parity, configuration
and sweep tests of the other files run again here with a bucket capacity given,
the one that the queue takes by itself: such calls are the queue's, and each
call is checked to have been answered by it (one wave per workgroup; a batch by
workgroups of batch_waves waves)."""
import numpy as np
import pytest

import test_gpu_param_sweep as sweep
from mlmq_tpds_withl3_amd import Solver, default_params
from mlmq_tpds_withl3_amd.serve import Server
# collected here again, with this module's solver
from test_gpu_configs import test_rmat22, test_road6m_delta_sweep  # noqa: F401
from test_gpu_parity import (test_back_edges, test_bfs_renumbered_graph,  # noqa: F401
                             test_errors_and_recovery, test_fixture_golden_and_source_switch,
                             test_grid_param_corners, test_heavy_piece_boundaries,
                             test_lane_pair_claims_wider_than_a_batch, test_lane_pairs_and_single_lanes,
                             test_random_graphs, test_rmat_small, test_road264k, test_zero_weight_components)

pytestmark = pytest.mark.gpu


class QueueSolver(Solver):
    def solve(self, src, params=None, **overrides):
        p = params if params is not None else default_params(**overrides)
        p.bucket_capacity = p.bucket_capacity or max(8192, self.n)
        t = super().solve(src, p)
        assert t["waves"] == t["work_blocks"]
        return t

    def solve_batch(self, sources, params=None, **overrides):
        p = params if params is not None else default_params(**overrides)
        p.bucket_capacity = p.bucket_capacity or max(8192, self.n // 8)
        t = super().solve_batch(sources, p)
        assert t["waves_per_query"] == p.batch_waves and t["graph_replay"] == (p.use_graph != 0)
        return t


class QueueServer(Server):
    def add_graph(self, graph, **params):
        params.setdefault("bucket_capacity", max(8192, (len(graph[0]) - 1) // 32))
        return super().add_graph(graph, **params)

    def run(self, *args, **kw):
        res, stats = super().run(*args, **kw)
        assert not res["solver"].any()
        return res, stats


@pytest.fixture(scope="module")
def solver():
    s = QueueSolver(0)
    yield s
    s.close()


def test_randomized_parameters(monkeypatch):
    monkeypatch.setattr(sweep, "Solver", QueueSolver)
    sweep.test_randomized_parameter_sweep(61)


def test_randomized_serving(monkeypatch):
    monkeypatch.setattr("mlmq_tpds_withl3_amd.serve.Server", QueueServer)
    sweep.test_randomized_serving_sweep(62)


def test_batch_of_a_road_graph(solver):
    from graphs_util import grid_csr
    from oracle import oracle as O
    row, col, w = grid_csr(60, 70, 5)
    solver.load_csr(row, col, w)
    src = np.random.default_rng(3).integers(0, 4200, 40)
    for pop, waves in ((32, 8), (64, 16)):
        solver.solve_batch(src, l1_pop=pop, batch_waves=waves, timeout_s=20.0)
        for i, x in enumerate(src):
            assert np.array_equal(solver.batch_dist(i), O.dijkstra(row, col, w, int(x))[0]), i
