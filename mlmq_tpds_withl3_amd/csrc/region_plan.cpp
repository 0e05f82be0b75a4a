// Cutting a graph into regions (region_graph.h), on the host.
#include "region_graph.h"

#include <algorithm>

namespace mlmq {

namespace {

// Consecutive ids are taken as regions as they are below this share of crossing
// edges (a Morton-ordered 3-NN graph crosses 4.4 %, grown regions 3.0 %, for a
// solve time within 5 % and no growth).
constexpr double kGoodCross = 0.06;

// Puts a region's `count` vertices in order of falling degree (ties keep their
// order).
void by_degree(const uint32_t *row, uint32_t *verts, uint32_t count) {
    uint32_t at[kRegionMaxDegree + 1] = {}, old[kRegionVerts];
    uint8_t degree[kRegionVerts];
    for (uint32_t i = 0; i < count; ++i) {
        old[i] = verts[i];
        degree[i] = (uint8_t)(row[old[i] + 1] - row[old[i]]);
        ++at[degree[i]];
    }
    uint32_t before = 0;
    for (uint32_t d = kRegionMaxDegree + 1; d-- > 0;) {
        const uint32_t k = at[d];
        at[d] = before;
        before += k;
    }
    for (uint32_t i = 0; i < count; ++i) verts[at[degree[i]]++] = old[i];
}

// Grown regions: breadth-first from a seed until the region is full; the
// vertices left at its rim seed the next ones, so regions pack closely.  A
// growth that ends early (a pocket between full regions, a small component)
// continues in the next pocket while the region is under three quarters full.
//
// The growth takes one core, beside the rest of a load, and is bound by memory
// latency where ids are scattered: ms on 50k / 264k / 1.07M shuffled vertices
// 0.5 / 2.6 / 13.7, before (a region number per vertex instead of a bit, a
// branch per edge) 1.0 / 6 / 24.
void grow(uint32_t n, const uint32_t *row, const uint32_t *col, RegionPlan *plan) {
    constexpr uint32_t kNone = 0xFFFFFFFFu, kAhead = 8;
    plan->order.resize((size_t)n + 1);   // (one place behind the last is written)
    uint32_t *order = plan->order.data();
    std::vector<uint64_t> taken((size_t)n / 64 + 1, 0);
    std::vector<uint32_t> rim;
    size_t rim_head = 0;
    uint32_t next = 0, placed = 0, first = 0;
    auto is_taken = [&](uint32_t v) { return (taken[v / 64] >> (v % 64) & 1u) != 0; };
    auto take = [&](uint32_t v) { taken[v / 64] |= 1ull << (v % 64); };
    auto close = [&]() {
        by_degree(row, order + first, placed - first);
        plan->first.push_back(placed);
        first = placed;
    };
    while (placed < n) {
        uint32_t seed = kNone;
        while (rim_head < rim.size() && seed == kNone) {
            const uint32_t x = rim[rim_head++];
            if (!is_taken(x)) seed = x;
        }
        if (rim_head == rim.size()) {
            rim.clear();
            rim_head = 0;
        }
        if (seed == kNone) {
            while (is_taken(next)) ++next;
            seed = next;
        }
        if (placed - first > kRegionVerts * 3 / 4) close();
        const uint32_t full = first + kRegionVerts;
        uint32_t head = placed;
        take(seed);
        order[placed++] = seed;
        for (; head < placed; ++head) {
            if (head + kAhead < placed) __builtin_prefetch(&col[row[order[head + kAhead]]]);
            const uint32_t lo = row[order[head]], hi = row[order[head] + 1];
            if (placed + (hi - lo) <= full) {
                // whether a neighbour is taken can't be predicted: it is written
                // behind the last vertex in any case
                for (uint32_t e = lo; e < hi; ++e) {
                    const uint32_t v = col[e];
                    const bool was = is_taken(v);
                    take(v);
                    __builtin_prefetch(&row[v]);
                    order[placed] = v;
                    placed += was ? 0u : 1u;
                }
                continue;
            }
            for (uint32_t e = lo; e < hi; ++e) {
                const uint32_t v = col[e];
                if (is_taken(v)) continue;
                if (placed < full) {
                    take(v);
                    order[placed++] = v;
                } else {
                    rim.push_back(v);
                }
            }
        }
    }
    close();
    plan->order.resize(n);
}

}  // namespace

bool region_plan(uint32_t n, const uint32_t *row, const uint32_t *col, RegionPlan *plan) {
    const uint64_t m = row[n];
    if (n == 0 || m > 8ull * n) return false;
    for (uint32_t u = 0; u < n; ++u)
        if (row[u + 1] - row[u] > kRegionMaxDegree) return false;
    plan->first.assign(1, 0);
    // consecutive ids, unless too many of their edges cross
    const double most = kGoodCross * (double)m;
    uint64_t cross = 0;
    for (uint32_t u = 0; u < n && (double)cross <= most; ++u)
        for (uint32_t e = row[u]; e < row[u + 1]; ++e) cross += col[e] / kRegionVerts != u / kRegionVerts;
    if ((double)cross > most) {
        grow(n, row, col, plan);
        return true;
    }
    plan->order.resize(n);
    for (uint32_t u = 0; u < n; ++u) plan->order[u] = u;
    for (uint64_t lo = 0; lo < n; lo += kRegionVerts) {
        const uint32_t hi = (uint32_t)std::min<uint64_t>(lo + kRegionVerts, n);
        by_degree(row, plan->order.data() + lo, hi - (uint32_t)lo);
        plan->first.push_back(hi);
    }
    return true;
}

}  // namespace mlmq
