// Internal interface of the region solver (region_kernels.hip): shortest
// paths on a graph cut into regions (region_graph.h).  Not part of the ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "region_graph.h"

namespace mlmq {

constexpr uint32_t kRegionQueries = 1u << 20;   // queries of one launch

// A cut graph on the device.
struct RegionGraph {
    uint32_t n = 0;
    uint32_t regions = 0;
    uint32_t inbox_slots = 0;
    uint32_t width = 0;          // threshold step inside a region
    RegionHdr *hdr = nullptr;    // per region
    uint32_t *image = nullptr;
    uint32_t *verts = nullptr;   // region-ordered vertex list
    uint32_t *where = nullptr;   // vertex -> region << kRegionIdBits | local id
};

constexpr uint64_t kRegionExit = ~1ull;   // slot value that ends a workgroup

struct RegionQuerySpace {        // per-query state; query q at the strides below
    uint32_t *dist;
    uint32_t *inbox;
    uint32_t *act;
    uint64_t dist_stride, inbox_stride, act_stride;
};

// A query of a launch over several graphs, each with its own space.
struct RegionQuery {
    const RegionHdr *hdr;
    const uint32_t *image, *verts, *where;
    uint32_t *dist, *inbox, *act;   // n, inbox_slots, regions words
    uint32_t n, slots, regions, width, src;
};

// Progress of a query: its seed record, and the regions with work (credits).
struct RegionProgress {
    uint64_t seed;
    uint32_t credits;
    uint32_t pad;
};

// What a workgroup did; after a solve, what all did.
struct RegionCounts {
    uint64_t credits, activations, messages, polls, relaxations, expansions, sweeps, pad;
};
constexpr uint32_t kRegionGroups = 4096;   // most workgroups of a launch

// Outcome of a solve, written by its last workgroup.
struct RegionSummary {
    RegionCounts all;
    uint64_t reset, start, end;   // wall-clock ticks
    uint32_t error, over;         // device error; 1: every query is over
};

struct RegionLaunch {
    RegionQuerySpace space;      // nq queries on one graph, or
    const RegionQuery *table;    // nq entries in device memory (null: `space`)
    uint32_t longest;            // most vertices, inbox slots or regions of a query
    RegionProgress *progress;    // nq entries
    uint64_t *ring;
    uint32_t ring_mask;
    RegionCounts *counts;        // grid entries
    uint32_t *ctl;               // control block (device_common.h)
    RegionSummary *summary;      // optional, may be host memory
    uint64_t *qtime;             // optional: per query, wall-clock ticks of its start and end
    uint64_t timeout_ticks;
    uint32_t nq;
    uint32_t admit;              // queries in flight at once
    uint32_t relaxers;           // kFew or kMany
    uint32_t grid;
};

// Workgroups come in two sizes: with kFew relaxers many are resident, with
// kMany a hop is shorter.
constexpr uint32_t kFew = 4, kMany = 8;
hipError_t region_occupancy(uint32_t relaxers, int *blocks_per_cu);
// Relaxers of a workgroup for nq queries of `regions` regions each.
uint32_t region_relaxers(uint64_t regions, uint32_t nq, uint32_t cus);
inline int region_waves(uint32_t relaxers) { return (int)relaxers + 2; }
// Queries of `regions` regions each to have in flight on `grid` workgroups.
uint32_t region_admit(uint64_t regions, uint32_t nq, uint32_t grid);
RegionQuery region_query(const RegionGraph &g, uint32_t *dist, uint32_t *inbox, uint32_t *act, uint32_t src);
// Builds the device side of a cut (temporary device memory: 4 bytes per edge).
// Returns hipErrorInvalidValue when some region exceeds the limits or too many
// edges cross.
hipError_t region_build(const RegionPlan &plan, uint32_t n, uint64_t m, const uint32_t *row, const uint32_t *col,
                        const uint32_t *wgt, double mean_weight, hipStream_t s, RegionGraph *g);
void region_free(RegionGraph *g);
// Per-query reset (distances, inboxes, activity), the control block and the
// seed records, then the solver.  `sources` is a device array of nq vertices,
// or null: one query from `src`.  With a table, the graph and the sources are
// ignored.
hipError_t launch_region_reset(const RegionGraph &g, const RegionLaunch &L, const uint32_t *sources, uint32_t src,
                               hipStream_t s);
hipError_t launch_region_solver(const RegionGraph &g, const RegionLaunch &L, hipStream_t s);

}  // namespace mlmq
