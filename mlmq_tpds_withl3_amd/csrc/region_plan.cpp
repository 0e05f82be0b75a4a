// Cutting a graph into regions (region_graph.h), on the host.
#include "region_graph.h"

#include <algorithm>
#include <atomic>
#include <thread>

namespace mlmq {

namespace {

// Above this share of crossing edges the solver's messages between regions
// outweigh the relaxations kept inside them.  Road-like graphs cut at 2-5 %,
// graphs without locality at 80 % and more; nothing measured lies between.
constexpr double kMaxCross = 0.12;
// Consecutive ids are taken as regions as they are below this share (a
// Morton-ordered 3-NN graph crosses 4.4 %, grown regions 3.0 %, for a solve
// time within 5 % and a tenth of the cutting time).
constexpr double kGoodCross = 0.06;

int thread_count(uint64_t items) {
    const uint64_t want = items / 100000 + 1;
    return (int)std::min<uint64_t>({want, 16, std::max(1u, std::thread::hardware_concurrency())});
}

template <typename F>
void in_parallel(uint64_t n, F &&f) {
    const int nt = thread_count(n);
    if (nt == 1) return f((uint64_t)0, n);
    std::vector<std::thread> th;
    for (int t = 0; t < nt; ++t) th.emplace_back([&, t]() { f(n * t / nt, n * (t + 1) / nt); });
    for (auto &x : th) x.join();
}

// Edges whose ends lie in different regions.
uint64_t crossing(uint32_t n, const uint32_t *row, const uint32_t *col, const uint32_t *reg) {
    std::atomic<uint64_t> total{0};
    in_parallel(n, [&](uint64_t lo, uint64_t hi) {
        uint64_t c = 0;
        for (uint64_t u = lo; u < hi; ++u)
            for (uint32_t e = row[u]; e < row[u + 1]; ++e) c += reg[col[e]] != reg[u];
        total += c;
    });
    return total;
}

constexpr uint32_t kNone = 0xFFFFFFFFu;

// Each region's vertices by falling degree (stable: ties keep their order).
void by_degree(const uint32_t *row, RegionPlan *plan) {
    const uint64_t regions = plan->first.size() - 1;
    in_parallel(regions * 1000, [&](uint64_t lo, uint64_t hi) {
        for (uint64_t r = (lo + 999) / 1000; r < (hi + 999) / 1000; ++r)
            std::stable_sort(plan->order.begin() + plan->first[r], plan->order.begin() + plan->first[r + 1],
                             [&](uint32_t a, uint32_t b) { return row[a + 1] - row[a] > row[b + 1] - row[b]; });
    });
}

}  // namespace

bool region_plan(uint32_t n, const uint32_t *row, const uint32_t *col, RegionPlan *plan) {
    const uint64_t m = row[n];
    if (n == 0 || m > 8ull * n) return false;
    for (uint32_t u = 0; u < n; ++u)
        if (row[u + 1] - row[u] > kRegionMaxDegree) return false;
    std::vector<uint32_t> reg(n);
    plan->order.resize(n);
    plan->first.assign(1, 0);

    // consecutive ids
    for (uint32_t u = 0; u < n; ++u) {
        reg[u] = u / kRegionVerts;
        plan->order[u] = u;
    }
    for (uint64_t u = kRegionVerts; u < n; u += kRegionVerts) plan->first.push_back((uint32_t)u);
    plan->first.push_back(n);
    if (m == 0 || (double)crossing(n, row, col, reg.data()) <= kGoodCross * (double)m) {
        by_degree(row, plan);
        return true;
    }

    // Grown regions: breadth-first from a seed until the region is full; the
    // vertices left at its rim seed the next ones, so regions pack closely.
    // A growth that ends early (a pocket between full regions, a small
    // component) continues in the next pocket while the region is under
    // three quarters full.
    std::fill(reg.begin(), reg.end(), kNone);
    plan->first.assign(1, 0);
    constexpr uint32_t kAhead = 16;
    std::vector<uint32_t> rim;
    size_t rim_head = 0;
    uint32_t next = 0, placed = 0, r = 0;
    auto size = [&]() { return placed - plan->first.back(); };
    auto put = [&](uint32_t v) {
        __builtin_prefetch(&row[v]);
        reg[v] = r;
        plan->order[placed++] = v;
    };
    while (placed < n) {
        uint32_t seed = kNone;
        while (rim_head < rim.size() && seed == kNone) {
            const uint32_t x = rim[rim_head++];
            if (reg[x] == kNone) seed = x;
        }
        if (rim_head == rim.size()) {
            rim.clear();
            rim_head = 0;
        }
        if (seed == kNone) {
            while (reg[next] != kNone) ++next;
            seed = next;
        }
        if (size() > kRegionVerts * 3 / 4) {
            plan->first.push_back(placed);
            ++r;
        }
        uint32_t head = placed;
        put(seed);
        for (; head < placed; ++head) {
            // (what the next vertices need: the ids are scattered over memory)
            if (head + kAhead < placed) __builtin_prefetch(&col[row[plan->order[head + kAhead]]]);
            if (head + kAhead / 2 < placed) {
                const uint32_t x = plan->order[head + kAhead / 2];
                for (uint32_t e = row[x]; e < row[x + 1]; ++e) __builtin_prefetch(&reg[col[e]], 1);
            }
            const uint32_t u = plan->order[head];
            for (uint32_t e = row[u]; e < row[u + 1]; ++e) {
                const uint32_t v = col[e];
                if (reg[v] != kNone) continue;
                if (size() < kRegionVerts) put(v);
                else rim.push_back(v);
            }
        }
    }
    plan->first.push_back(n);
    if ((double)crossing(n, row, col, reg.data()) > kMaxCross * (double)m) return false;
    by_degree(row, plan);
    return true;
}

}  // namespace mlmq
