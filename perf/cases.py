"""Performance cases: the shortest-path work this framework is used for.

A case is one graph family and size, one way of calling the solver, and the
settings a program passes.  Families are the repository's own: `road` (k
nearest neighbours of random points, symmetrised; the road-like inputs) and
`rmat` (symmetrised power-law graphs, weights 1..1000).  Ways of calling:

* `solve`: one query on a resident graph.  `out` says where the program wants
  the distances: `host` (copied out, as the command-line driver does) or
  `device` (used where they are, as the benchmark does);
* `batch`: many sources answered in one call, every row copied out;
* `serve`: a burst of requests over three resident graphs, every row copied out.

`settings` names the solver parameters: `default` (none given), `road` (the
tuned point of the road workload nearest in size) or `power` (the tuned point
of the power-law workload).
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from mlmq_tpds_withl3_amd import HostGraph, Solver, WORKLOADS, default_params
from mlmq_tpds_withl3_amd.serve import Server

UNREACHED = 0x7FFFFFFF
LARGEST_SEEDED_SCALE = 20   # larger power-law graphs take long to generate: one fixed graph each


def _case(name, family, size, call="solve", settings="default", out="host", **more):
    c = dict(name=name, family=family, size=size, call=call, settings=settings, out=out,
             ordered=True, factor=3 if family == "road" else 16, queries=1, source="random")
    c.update(more)
    return c


def listed():
    return [
        # the smallest call: a town-sized graph (the size of the known-answer
        # fixture), default settings; latency and launches are all there is
        _case("road2k", "road", 2_052, ordered=False),
        # a county with an odd vertex count, numbered at random, default settings
        _case("road50k", "road", 50_021, ordered=False),
        # the 264,346-vertex benchmark size (a city's network) at its tuned point
        _case("road264k", "road", 264_346, settings="road", ordered=False),
        # the 1,070,376-vertex benchmark size (a state's network), nothing tuned
        _case("road1m", "road", 1_070_376),
        # the largest road input: 6,262,104 vertices from the centroid at its
        # tuned point, distances used on the device: the headline query
        _case("road6m", "road", 6_262_104, settings="road", out="device", source="centroid"),
        # a small power-law graph, default settings
        _case("rmat14", "rmat", 14),
        # a power-law graph between the small and the large, tuned
        _case("rmat18", "rmat", 18, settings="power"),
        # the power-law benchmark input at its tuned point, from its hub
        _case("rmat22", "rmat", 22, settings="power", out="device", source="hub"),
        # a distance table of a small network: one batched call, 64 sources
        _case("batch_road20k", "road", 20_011, call="batch", queries=64),
        # a distance table of a city's network
        _case("batch_road264k", "road", 264_346, call="batch", queries=64),
        # a burst of 32 requests over a city, a state and a power-law graph
        # (50/30/20 %), the benchmark's serving mix at a burst's scale
        _case("serve_mix", "mix", 264_346, call="serve", queries=32),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["road", "road", "road", "rmat", "rmat", "batch", "serve"])
    if kind == "road":
        n = _log_uniform(rng, 2_000, 2_500_000)
        return dict(family="road", size=n, call="solve", settings=rng.choice(["default", "road"]),
                    out=rng.choice(["host", "device"]), ordered=rng.random() < 0.5,
                    factor=rng.choice([3, 3, 4]), queries=1, source=rng.choice(["random", "centroid"]))
    if kind == "rmat":
        return dict(family="rmat", size=rng.randint(10, 20), call="solve",
                    settings=rng.choice(["default", "power"]), out=rng.choice(["host", "device"]),
                    ordered=True, factor=rng.randint(4, 16), queries=1,
                    source=rng.choice(["random", "hub"]))
    if kind == "batch":
        n = _log_uniform(rng, 2_000, 250_000)
        return dict(family="road", size=n, call="batch", settings="default", out="host",
                    ordered=rng.random() < 0.5, factor=3, queries=rng.randint(2, 64), source="random")
    return dict(family="mix", size=_log_uniform(rng, 10_000, 250_000), call="serve", settings="default",
                out="host", ordered=True, factor=3, queries=rng.randint(1, 32), source="random")


# ---- inputs ----

def _road(n, k, seed, ordered):
    return HostGraph.knn(n, k, seed=seed, weight_scale=-50_000.0 if n > 500_000 else 1e5, morton=ordered)


def _rmat(scale, factor, seed):
    return HostGraph.rmat(scale, factor, 0.57, 0.19, 0.19, seed=seed, wmin=1, wmax=1000)


@functools.lru_cache(maxsize=1)
def _large_rmat(scale, factor):
    return _rmat(scale, factor, WORKLOADS["rmat22"]["seed"])


def _graph(case, seed):
    if case["family"] == "road":
        return _road(case["size"], case["factor"], seed, case["ordered"])
    if case["size"] > LARGEST_SEEDED_SCALE:
        return _large_rmat(case["size"], case["factor"])
    return _rmat(case["size"], case["factor"], seed)


def _sources(g, count, seed):
    """Seeded sources with several neighbours (not in one of the few-vertex
    components such graphs also have)."""
    deg = np.diff(g.arrays()[0])
    pool = np.flatnonzero(deg >= 5)
    if len(pool) == 0:
        pool = np.flatnonzero(deg == deg.max())
    return pool[np.random.default_rng(seed).integers(0, len(pool), size=count)].astype(np.int32)


def _source(case, g, seed):
    if case["source"] == "centroid":
        return int(g.centroid_vertex())
    if case["source"] == "hub" and case["size"] <= LARGEST_SEEDED_SCALE:
        return int(g.max_degree_vertex())
    if case["source"] == "hub":   # the fixed graph: one of its 64 largest hubs
        deg = np.diff(g.arrays()[0])
        return int(np.argsort(deg)[-1 - seed % 64])
    return int(_sources(g, 1, seed)[0])


def _settings(case):
    if case["settings"] == "road":
        name = "road6m" if case["size"] > 1_500_000 else "road264k"
        return dict(WORKLOADS[name]["bench_point"])
    if case["settings"] == "power":
        return dict(WORKLOADS["rmat22"]["bench_point"])
    return {}


def _mix(case, seed):
    """Three graphs (a city, a network four times as large, a power-law graph)
    and the requests over them."""
    n = case["size"]
    scale = max(10, min(18, n.bit_length()))
    graphs = [_road(n, 3, seed, False), _road(4 * n, 3, seed + 1, True), _rmat(scale, 16, seed + 2)]
    # the order of the graphs is the same for every seed, so rows keep their lengths
    which = np.random.default_rng(case["queries"]).choice(3, size=case["queries"], p=[0.5, 0.3, 0.2]).astype(np.int32)
    src = np.empty(case["queries"], dtype=np.int32)
    for i, g in enumerate(graphs):
        at = np.flatnonzero(which == i)
        src[at] = _sources(g, len(at), seed + 10 + i)
    return graphs, which, src


class _DeviceRow:
    """The distances of a solver's last query as they lie on the device."""

    def __init__(self, solver):
        self.solver = solver   # its memory
        self.__cuda_array_interface__ = dict(shape=(solver.n,), typestr="<i4", version=2, strides=None,
                                             data=(solver.dist_device_ptr(), False))


def prepare(case, seed):
    if case["call"] == "serve":
        graphs, which, src = _mix(case, seed)
        server = Server(0, hbm_budget=8 << 30)
        power = {k: v for k, v in WORKLOADS["rmat22"]["bench_point"].items()
                 if k in ("delta", "light_split", "buckets", "bucket_window", "l2_batch", "min_read", "l1_pop")}
        for g, p in zip(graphs, (WORKLOADS["road264k"]["serve_point"], {}, power)):
            server.add_graph(g, **p)
        rows = [np.empty(graphs[g].n, dtype=np.int32) for g in which]
        return dict(case=case, server=server, arrival=np.zeros(len(src)), which=which, src=src, rows=rows)
    g = _graph(case, seed)
    solver = Solver(0)
    solver.load_graph(g)
    state = dict(case=case, solver=solver, params=default_params(**_settings(case)))
    if case["call"] == "batch":
        state["src"] = _sources(g, case["queries"], seed)
    else:
        state["src"] = _source(case, g, seed)
    return state


def run(state):
    case = state["case"]
    if case["call"] == "serve":
        res, _ = state["server"].run(state["arrival"], state["which"], state["src"], dist_out=state["rows"])
        return dict(rows=state["rows"], status=np.ascontiguousarray(res["status"]))
    s = state["solver"]
    if case["call"] == "batch":
        s.solve_batch(state["src"], params=state["params"])
        return [s.batch_dist(i) for i in range(len(state["src"]))]
    s.solve(state["src"], params=state["params"])
    if case["out"] == "device":
        return dict(dist=torch.as_tensor(_DeviceRow(s), device="cuda"))
    return dict(dist=s.dist())


# ---- the work and the right answers ----

def _dims(case):
    """(vertices, edges) a graph of this case has, near enough: a symmetrised
    3-NN graph has 3.73 edges per vertex, 4-NN 4.93; RMAT loses some of its
    2 x factor per vertex to duplicates, fewer on larger graphs."""
    if case["family"] == "road":
        return case["size"], int(case["size"] * (3.73 if case["factor"] == 3 else 4.93))
    n = 1 << case["size"]
    return n, int(n * 2 * case["factor"] * min(0.96, 0.60 + 0.0166 * case["size"]))


def work(case):
    """The graph read once (offsets, destinations, weights), every distance
    written once; an addition and a comparison per edge and query."""
    if case["call"] == "serve":
        n = case["size"]
        scale = max(10, min(18, n.bit_length()))
        parts = [(0.5, dict(family="road", size=n, factor=3)), (0.3, dict(family="road", size=4 * n, factor=3)),
                 (0.2, dict(family="rmat", size=scale, factor=16))]
        total = dict(bytes=0.0, flops=0.0)
        for share, c in parts:
            v, e = _dims(c)
            total["bytes"] += 4 * v + 8 * e + 4 * v * share * case["queries"]
            total["flops"] += 2 * e * share * case["queries"]
        return total
    v, e = _dims(case)
    return dict(bytes=4 * v + 8 * e + 4 * v * case["queries"], flops=2 * e * case["queries"])


def _shortest(row, col, w, src):
    """Shortest distances by rounds of relaxation from the improved vertices."""
    n = len(row) - 1
    dist = np.full(n, np.iinfo(np.int64).max // 2, dtype=np.int64)
    dist[src] = 0
    deg = np.diff(row)
    front = np.array([src], dtype=np.int64)
    while len(front):
        d = deg[front]
        owner = np.repeat(np.arange(len(front)), d)
        at = np.arange(int(d.sum())) - np.repeat(np.cumsum(d) - d, d) + row[front][owner]
        to = col[at]
        nd = dist[front][owner] + w[at]
        better = nd < dist[to]
        to, nd = to[better], nd[better]
        np.minimum.at(dist, to, nd)
        front = np.unique(to)
    return np.where(dist < UNREACHED, dist, UNREACHED)


def exact(case, seed):
    if case["call"] == "serve" or work(case)["flops"] > 20e6:
        return None
    g = _graph(case, seed)
    row, col, w = (x.astype(np.int64) for x in g.arrays())
    if case["call"] == "batch":
        return [_shortest(row, col, w, int(s)) for s in _sources(g, case["queries"], seed)]
    return dict(dist=_shortest(row, col, w, _source(case, g, seed)))
