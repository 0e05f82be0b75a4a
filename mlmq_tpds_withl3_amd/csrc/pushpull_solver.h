// Internal interface of the push-pull solver (pushpull_kernels.hip): shortest
// paths on undirected power-law graphs.  Not part of the ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mlmq {

// Per graph: the reach of phase 1, and words 8..15 of every hop block with more
// than kInlineEdges edges = its edges of weight < (reach / 8 + 1) * (j + 1).
constexpr uint32_t kBoundSteps = 8;
// Rounds of pushes up to the bound before the pull, and of full pushes after
// it, that are launched before the host looks.
constexpr uint32_t kBoundedRounds = 12;
constexpr uint32_t kFullRounds = 5;
constexpr uint32_t kMaxRounds = 1024;   // counters per query

// Edges examined and improvements of all rounds by the workgroups of one index.
struct PushPullWork {
    uint64_t edges, improved;
};
constexpr uint32_t kWorkEntries = 2048;   // most workgroups of a launch

struct PushPullLaunch {
    const uint32_t *col;
    const uint32_t *wgt;
    const uint4 *blocks;
    uint32_t id_mask;        // vertex bits of an inline edge's destination word
    uint32_t *dist;          // n
    uint32_t *mark;          // n: last round that queued the vertex
    uint32_t *front[2];      // n each: the rounds' vertices, by parity
    uint32_t *count;         // kMaxRounds + 1: vertices of each round
    PushPullWork *work;      // a workgroup's share each (null: not counted)
    uint32_t *bound;         // distance up to which phase 1 settles
    uint32_t n;
    uint32_t reach;          // the bound lies this far beyond the nearest hub
    uint32_t hub_degree;
    uint32_t src;
    uint64_t *time;          // ticks: reset, and start of the first round or (tables) the end
};

// Queries of one sequence of launches: one, or a table of them.
struct PushPullQueries {
    PushPullLaunch one;
    const PushPullLaunch *table;   // nq entries in device memory (null: `one`)
    uint32_t nq;
    uint32_t max_n;                // most vertices of a query
    uint32_t most_groups;          // workgroups of a push or pull (0: no limit)
};

// Outcome of a query, written to host memory.
struct PushPullSummary {
    PushPullWork work;
    uint64_t time[3];               // ticks: reset, first round, now
    uint32_t count[kMaxRounds + 1];
};

// *asymmetric = 1 if some edge (u, v, w) has no edge (v, u, w).  Rows of more
// than kInlineEdges edges are sorted by (weight, destination).
hipError_t launch_symmetry_check(const uint32_t *row, const uint32_t *col, const uint32_t *wgt, uint32_t n, uint64_t m,
                                 uint32_t *asymmetric, hipStream_t s);
hipError_t launch_bound_counts(const uint32_t *row, const uint32_t *wgt, uint32_t n, uint32_t reach, uint4 *blocks,
                               hipStream_t s);
hipError_t launch_pushpull_reset(const PushPullQueries &Q, hipStream_t s);
// Workgroups of a push launch of each query, and waves of each.
uint32_t push_groups(const PushPullQueries &Q);
constexpr int kPushWaves = 8;
// Round r expands the vertices of count[r] into those of count[r + 1].
hipError_t launch_push(const PushPullQueries &Q, uint32_t round, bool bounded, hipStream_t s);
// count[0 .. rounds], work and times of a single query.
hipError_t launch_pushpull_summary(const PushPullLaunch &L, uint32_t rounds, PushPullSummary *out, hipStream_t s);
// Adds the pulled vertices to those of count[round].
hipError_t launch_pull(const PushPullQueries &Q, uint32_t round, hipStream_t s);

}  // namespace mlmq
