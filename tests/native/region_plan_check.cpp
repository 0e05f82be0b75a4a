// The cut of a graph (region_plan.cpp) for tests without a GPU.
#include <algorithm>

#include "region_graph.h"

// Regions, with order[n] and first[regions + 1] filled in; -1: not cut.
extern "C" int region_plan_check(uint32_t n, const uint32_t *row, const uint32_t *col, uint32_t *order,
                                 uint32_t *first) {
    mlmq::RegionPlan plan;
    if (!mlmq::region_plan(n, row, col, &plan)) return -1;
    if (plan.order.size() != n || plan.first.size() > (size_t)n + 1) return -2;
    std::copy(plan.order.begin(), plan.order.end(), order);
    std::copy(plan.first.begin(), plan.first.end(), first);
    return (int)plan.first.size() - 1;
}
