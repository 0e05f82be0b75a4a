// Push-pull solver: shortest paths on undirected power-law graphs.
//
// Most of such a graph's edges are heavy edges of hubs, and they lower nothing:
// on RMAT-22 (weights 1..1000) every vertex of degree 30 is reached at a
// distance of 10-100, so a hub's edges of weight 100-1000 only matter to the
// few vertices that have no lighter way in.  The vertex queue still relaxes
// each of the 128 M edges once.  Here
//   1. rounds of pushes settle vertices up to a bound B only: a vertex at
//      distance d reads its edges of weight <= B - d, a prefix of its sorted
//      adjacency whose length comes from its hop block.  B is the distance of
//      the nearest hub pushed so far plus the graph's `reach` (until a hub is
//      met there is no bound: a source at the rim first finds its way in);
//   2. one pull: every vertex beyond B looks at its own few edges, lightest
//      first, until the weight alone exceeds the best sum;
//   3. rounds of full pushes from the vertices beyond B, and from what phase 1
//      may have left, finish the rest.
// Edges examined on RMAT-22: about 25 % of the graph (reach = the 5 % quantile
// of the weights), against 105 % before.  Any B gives the same distances, also
// one that falls while phase 1 runs: a vertex lowered to at most B is pushed
// to everything it can bring to at most B, what it could bring further is
// pulled from the other end, and a vertex beyond B is pushed in phase 3.  The
// graph must be undirected (checked edge by edge when it is loaded): the pull
// reads out-edges as in-edges.
//
// Every round is one launch, and no workgroup waits for another.  A round that
// finds nothing costs its launch (40 more of them: 63-88 us, RMAT-13 to 20).
//
// Measured, device us of one query, vertex queue / here: RMAT-14 400 / 165,
// RMAT-18 2900 / 330, RMAT-22 11000 / 1130 (0.6 TB/s of scattered line fetches;
// the pull 200 us, the largest round of pushes 190).
#include "device_common.h"
#include "hop_block.h"
#include "pushpull_solver.h"

namespace mlmq {

namespace {

constexpr uint32_t kGroup = 512;        // threads of a workgroup
constexpr uint32_t kBuffer = 4096;      // queued vertices a workgroup gathers
constexpr uint32_t kUnroll = 4;

struct OutBuffer {
    uint32_t n;
    uint32_t base;
    uint32_t v[kBuffer];
};

__device__ __forceinline__ void queue_vertex(OutBuffer &B, uint32_t *out, uint32_t *count, uint32_t v) {
    const uint32_t p = atomicAdd(&B.n, 1u);
    if (p < kBuffer) B.v[p] = v;
    else out[fetch_add(count, 1u)] = v;
}

// All threads of the workgroup.
__device__ __forceinline__ void flush_buffer(OutBuffer &B, uint32_t *out, uint32_t *count) {
    __syncthreads();
    const uint32_t have = min(B.n, kBuffer);
    if (threadIdx.x == 0 && have) B.base = fetch_add(count, have);
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < have; i += kGroup) out[B.base + i] = B.v[i];
    __syncthreads();
}

// All threads of the workgroup: adds to its entry (thousands of workgroups that
// add to the same two words take longer than most rounds' work).
__device__ __forceinline__ void count_work(const PushPullLaunch &L, uint32_t *s_work, uint32_t edges, uint32_t improved) {
    if (!L.work) return;
    edges = wave_sum(edges);
    improved = wave_sum(improved);
    if (lane_id() == 0) {
        atomicAdd(&s_work[0], edges);
        atomicAdd(&s_work[1], improved);
    }
    __syncthreads();
    if (threadIdx.x != 0 || s_work[0] == 0) return;
    L.work[blockIdx.x].edges += s_work[0];
    L.work[blockIdx.x].improved += s_work[1];
}

// Lower v[k] to nd[k] where it was above nd[k]; queue each vertex once a round
// when that succeeds.  All k are under way at once: one after another (two
// dependent atomics of about 1.5 us each) they were most of a round's time.
// Returns how many fell.
template <uint32_t kN>
__device__ __forceinline__ uint32_t lower(const PushPullLaunch &L, OutBuffer &B, uint32_t *out, uint32_t *count,
                                          uint32_t round, uint32_t bound, const uint32_t (&v)[kN],
                                          const uint32_t (&nd)[kN], const uint32_t (&was)[kN]) {
    uint32_t old[kN], seen[kN], fell = 0;
#pragma unroll
    for (uint32_t k = 0; k < kN; ++k) {
        old[k] = 0;
        if (nd[k] < was[k] && nd[k] <= bound) old[k] = fetch_min(L.dist + v[k], nd[k]);
    }
#pragma unroll
    for (uint32_t k = 0; k < kN; ++k) asm volatile("" : "+v"(old[k]));
#pragma unroll
    for (uint32_t k = 0; k < kN; ++k) {
        seen[k] = round + 1u;
        if (old[k] > nd[k]) {
            seen[k] = __hip_atomic_exchange(L.mark + v[k], round + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            ++fell;
        }
    }
#pragma unroll
    for (uint32_t k = 0; k < kN; ++k) asm volatile("" : "+v"(seen[k]));
#pragma unroll
    for (uint32_t k = 0; k < kN; ++k)
        if (seen[k] != round + 1u) queue_vertex(B, out, count, v[k]);
    return fell;
}

// This workgroup's query.
template <bool kTable>
__device__ __forceinline__ PushPullLaunch query_of(const PushPullLaunch &one, const PushPullLaunch *table) {
    if constexpr (kTable) return table[blockIdx.y];
    else return one;
}

// A workgroup takes its share of the round's vertices, at most one per thread:
// few vertices of many edges are spread over all workgroups.  Inline vertices
// are pushed by their thread; the others' edges are numbered through and
// dealt out to all threads.
template <bool kTable, bool kBounded>
__global__ __launch_bounds__(kGroup) void push_kernel(PushPullLaunch one, const PushPullLaunch *table, uint32_t round) {
    const PushPullLaunch L = query_of<kTable>(one, table);
    __shared__ OutBuffer B;
    __shared__ uint32_t s_first[kGroup + 1], s_start[kGroup], s_dist[kGroup], s_wave[kGroup / kWave];
    __shared__ uint32_t s_work[2];
    const uint32_t count = L.count[round];
    if (count == 0) return;
    if (!kTable && round == 0 && blockIdx.x == 0 && threadIdx.x == 0) L.time[1] = wall_clock64();
    const uint32_t bound = kBounded ? *L.bound : kUnreached - 1u;
    const uint32_t *in = (round & 1u ? L.front[1] : L.front[0]);
    uint32_t *out = (round & 1u ? L.front[0] : L.front[1]), *out_count = L.count + round + 1;
    const uint32_t share = min(kGroup, (count + gridDim.x - 1) / gridDim.x);
    if (blockIdx.x * share >= count) return;
    // half of the places that are searched for an edge's vertex
    const uint32_t half = share > 1 ? 1u << (31 - __builtin_clz(share - 1)) : 0u;
    if (threadIdx.x == 0) {
        B.n = 0;
        s_work[0] = s_work[1] = 0;
    }
    uint32_t edges = 0, improved = 0;
    for (uint32_t b = blockIdx.x * share; b < count; b += gridDim.x * share) {
        const bool have = threadIdx.x < share && b + threadIdx.x < count;
        uint32_t len = 0, start = 0, d = 0;
        __syncthreads();
        // (loads without conditions: under one each they would wait for the last)
        const uint32_t v = in[have ? b + threadIdx.x : b];
        const uint4 *p = L.blocks + 4ull * v;
        const uint4 q0 = p[0], q1 = p[1], q2 = p[2], q3 = p[3];
        d = L.dist[v];
        if (have) {
            if (d > bound) {
                // beyond the bound by now: phase 3 pushes it
            } else if (q0.x <= kInlineEdges) {
                const uint32_t word[14] = {q0.z, q0.w, q1.x, q1.y, q1.z, q1.w, q2.x,
                                           q2.y, q2.z, q2.w, q3.x, q3.y, q3.z, q3.w};
                uint32_t to[kInlineEdges], nd[kInlineEdges], was[kInlineEdges];
#pragma unroll
                for (uint32_t k = 0; k < kInlineEdges; ++k) {
                    to[k] = word[2 * k] & L.id_mask;
                    nd[k] = d + word[2 * k + 1];
                    was[k] = L.dist[k < q0.x ? to[k] : v];
                }
#pragma unroll
                for (uint32_t k = 0; k < kInlineEdges; ++k) was[k] = k < q0.x ? was[k] : 0u;
                improved += lower(L, B, out, out_count, round, bound, to, nd, was);
                edges += q0.x;
            } else {
                start = q0.y;
                len = q0.x;
                if (kBounded) {
                    uint32_t limit = bound;
                    if (q0.x >= L.hub_degree && d + L.reach < limit) {
                        limit = d + L.reach;
                        (void)fetch_min(L.bound, limit);
                    }
                    // the least step that covers every weight up to limit - d
                    const uint32_t room = limit - d;
                    const uint32_t step = L.reach / kBoundSteps + 1u;
                    const uint32_t j = room / step;
                    const uint32_t word[8] = {q2.x, q2.y, q2.z, q2.w, q3.x, q3.y, q3.z, q3.w};
#pragma unroll
                    for (uint32_t k = 0; k < kBoundSteps; ++k)
                        if (k == j) len = word[k];
                }
            }
        }
        // number the edges
        const uint32_t incl = wave_incl_add(len);
        const uint32_t wave = threadIdx.x / kWave;
        if (lane_id() == kWave - 1) s_wave[wave] = incl;
        s_start[threadIdx.x] = start;
        s_dist[threadIdx.x] = d;
        __syncthreads();
        uint32_t before = 0, total = 0;
#pragma unroll
        for (uint32_t k = 0; k < kGroup / kWave; ++k) {
            before += k < wave ? s_wave[k] : 0u;
            total += s_wave[k];
        }
        s_first[threadIdx.x] = before + incl - len;
        if (threadIdx.x == 0) s_first[kGroup] = total;
        __syncthreads();
        edges += threadIdx.x == 0 ? total : 0u;
        for (uint32_t e0 = 0; e0 < total; e0 += kUnroll * kGroup) {
            uint32_t at[kUnroll], c[kUnroll], nd[kUnroll], was[kUnroll];
#pragma unroll
            for (uint32_t j = 0; j < kUnroll; ++j) {
                at[j] = 0;
                nd[j] = kUnreached;
                if (e0 + j * kGroup >= total) continue;   // (uniform)
                const uint32_t e = e0 + j * kGroup + threadIdx.x;
                // the last vertex whose first edge is <= e
                uint32_t lo = 0;
                for (uint32_t k = half; k; k /= 2)
                    if (s_first[lo + k] <= e) lo += k;
                at[j] = e < total ? s_start[lo] + (e - s_first[lo]) : s_start[lo];
                nd[j] = e < total ? s_dist[lo] : kUnreached;
            }
#pragma unroll
            for (uint32_t j = 0; j < kUnroll; ++j) {
                c[j] = L.col[at[j]];
                nd[j] = min(nd[j] + L.wgt[at[j]], kUnreached);   // (no edge: not below any distance)
            }
#pragma unroll
            for (uint32_t j = 0; j < kUnroll; ++j) was[j] = L.dist[c[j]];
            improved += lower(L, B, out, out_count, round, bound, c, nd, was);
        }
    }
    flush_buffer(B, out, out_count);
    count_work(L, s_work, edges, improved);
    // (its last round's other workgroups end at about the same time)
    if (kTable && blockIdx.x == 0 && threadIdx.x == 0) L.time[1] = wall_clock64();
}

// Every vertex beyond the bound takes the best distance over its edges.
template <bool kTable>
__global__ __launch_bounds__(kGroup) void pull_kernel(PushPullLaunch one, const PushPullLaunch *table, uint32_t round) {
    const PushPullLaunch L = query_of<kTable>(one, table);
    __shared__ OutBuffer B;
    __shared__ uint32_t s_work[2];
    uint32_t *out = (round & 1u ? L.front[1] : L.front[0]), *out_count = L.count + round;
    if (threadIdx.x == 0) {
        B.n = 0;
        s_work[0] = s_work[1] = 0;
    }
    __syncthreads();
    uint32_t edges = 0, improved = 0;
    const uint32_t bound = *L.bound;
    for (uint32_t base = blockIdx.x * kGroup; base < L.n; base += gridDim.x * kGroup) {
        const uint32_t v = base + threadIdx.x;
        const uint32_t d = v < L.n ? L.dist[v] : 0u;
        uint32_t best = d, deg = 0, start = 0;
        if (d > bound) {
            const uint4 *p = L.blocks + 4ull * v;
            const uint4 q0 = p[0];
            if (q0.x > kInlineEdges) {
                deg = q0.x;
                start = q0.y;
            } else if (q0.x) {
                const uint4 q1 = p[1], q2 = p[2], q3 = p[3];
                const uint32_t word[14] = {q0.z, q0.w, q1.x, q1.y, q1.z, q1.w, q2.x,
                                           q2.y, q2.z, q2.w, q3.x, q3.y, q3.z, q3.w};
                uint32_t from[kInlineEdges];
#pragma unroll
                for (uint32_t k = 0; k < kInlineEdges; ++k) from[k] = L.dist[k < q0.x ? word[2 * k] & L.id_mask : v];
#pragma unroll
                for (uint32_t k = 0; k < kInlineEdges; ++k)
                    if (k < q0.x && from[k] < kUnreached) best = min(best, from[k] + word[2 * k + 1]);
                edges += q0.x;
            }
        }
        // the others one after another, 64 edges at a time, lightest first
        for (uint64_t rest = ballot(deg != 0); rest; rest &= rest - 1) {
            const uint32_t l = (uint32_t)__builtin_ctzll(rest);
            const uint32_t s = read_lane(start, l), n = read_lane(deg, l);
            uint32_t b = read_lane(best, l);
            for (uint32_t at = 0; at < n; at += kWave) {
                const bool in = at + lane_id() < n;
                const uint32_t e = s + (in ? at + lane_id() : n - 1u);
                const uint32_t c = L.col[e], w = L.wgt[e];
                const uint32_t from = L.dist[c];
                uint32_t x = in && from < kUnreached ? from + w : ~0u;
                x = ~read_lane(wave_incl_max(~x), kWave - 1);
                b = min(b, x);
                edges += in ? 1u : 0u;
                if (read_lane(w, kWave - 1) >= b) break;
            }
            if (lane_id() == l) best = b;
        }
        if (v < L.n && d > bound && best < kUnreached) {
            // (only this thread lowers v in this launch)
            if (best < d) {
                L.dist[v] = best;
                ++improved;
            }
            // phase 1 may have left it in the list
            if (L.mark[v] != round) queue_vertex(B, out, out_count, v);
        }
    }
    flush_buffer(B, out, out_count);
    count_work(L, s_work, edges, improved);
}

template <bool kTable>
__global__ __launch_bounds__(256) void pushpull_reset_kernel(PushPullLaunch one, const PushPullLaunch *table) {
    const PushPullLaunch L = query_of<kTable>(one, table);
    const uint32_t src = L.src;
    const uint32_t stride = gridDim.x * blockDim.x, t = blockIdx.x * blockDim.x + threadIdx.x;
    for (uint32_t i = t; i < L.n; i += stride) {
        L.dist[i] = i == src ? 0u : kUnreached;
        L.mark[i] = 0;
    }
    for (uint32_t i = t; i <= kMaxRounds; i += stride) L.count[i] = i == 0 ? 1u : 0u;
    if (L.work)
        for (uint32_t i = t; i < kWorkEntries; i += stride) L.work[i] = PushPullWork{0, 0};
    if (t == 0) {
        L.front[0][0] = src;
        *L.bound = kUnreached - 1u;
        L.time[0] = L.time[1] = wall_clock64();
    }
}

__global__ __launch_bounds__(1024) void pushpull_summary_kernel(PushPullLaunch L, uint32_t groups, uint32_t rounds,
                                                                PushPullSummary *out) {
    for (uint32_t i = threadIdx.x; i <= rounds; i += blockDim.x) out->count[i] = L.count[i];
    __shared__ unsigned long long s_edges, s_improved;
    if (threadIdx.x == 0) s_edges = s_improved = 0;
    __syncthreads();
    uint64_t edges = 0, improved = 0;
    for (uint32_t i = threadIdx.x; i < groups; i += blockDim.x) {
        edges += L.work[i].edges;
        improved += L.work[i].improved;
    }
    if (edges) atomicAdd(&s_edges, (unsigned long long)edges);
    if (improved) atomicAdd(&s_improved, (unsigned long long)improved);
    __syncthreads();
    if (threadIdx.x < 2) out->time[threadIdx.x] = L.time[threadIdx.x];
    if (threadIdx.x == 0) out->work = PushPullWork{s_edges, s_improved};
    if (threadIdx.x == 0) out->time[2] = wall_clock64();
}

// A workgroup checks kSymEdges consecutive edges, whoever's they are: with a
// wave per vertex the largest hub of RMAT-22 took 0.3 s.
constexpr uint32_t kSymEdges = 4096;
__global__ __launch_bounds__(256) void symmetry_kernel(const uint32_t *row, const uint32_t *col, const uint32_t *wgt,
                                                       uint32_t n, uint32_t *asymmetric) {
    const uint64_t first = (uint64_t)blockIdx.x * kSymEdges;
    const uint32_t m = row[n], end = (uint32_t)min((uint64_t)m, first + kSymEdges);
    // the vertices of the first and the last edge: the last with row[u] <= e
    uint32_t range[2];
    for (uint32_t i = 0; i < 2; ++i) {
        const uint32_t e = i ? end - 1u : (uint32_t)first;
        uint32_t lo = 0, hi = n;
        while (hi - lo > 1) {
            const uint32_t mid = lo + (hi - lo) / 2;
            if (row[mid] <= e) lo = mid;
            else hi = mid;
        }
        range[i] = lo;
    }
    bool bad = false;
    for (uint32_t e = (uint32_t)first + threadIdx.x; e < end; e += blockDim.x) {
        uint32_t u = range[0], hi = range[1] + 1u;
        while (hi - u > 1) {
            const uint32_t mid = u + (hi - u) / 2;
            if (row[mid] <= e) u = mid;
            else hi = mid;
        }
        const uint32_t v = col[e], w = wgt[e], top = row[v + 1];
        uint32_t a = row[v], b = top;
        bool found = false;
        if (b - a > kInlineEdges) {
            while (a < b) {   // first entry >= (w, u)
                const uint32_t mid = a + (b - a) / 2, mw = wgt[mid];
                if (mw < w || (mw == w && col[mid] < u)) a = mid + 1;
                else b = mid;
            }
            found = a < top && wgt[a] == w && col[a] == u;
        } else {
            for (; a < b; ++a) found = found || (wgt[a] == w && col[a] == u);
        }
        bad = bad || !found;
    }
    if (ballot(bad) && lane_id() == 0) *asymmetric = 1;
}

__global__ __launch_bounds__(256) void bound_count_kernel(const uint32_t *row, const uint32_t *wgt, uint32_t n,
                                                          uint32_t reach, uint4 *blocks) {
    const uint32_t stride = gridDim.x * blockDim.x;
    const uint32_t step = reach / kBoundSteps + 1u;
    for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += stride) {
        const uint32_t s = row[v], e = row[v + 1];
        if (e - s <= kInlineEdges) continue;
        uint32_t at = s;
        for (uint32_t j = 0; j < kBoundSteps; ++j) {
            // edges of weight < step * (j + 1); the last step covers the reach
            const uint32_t top = step * (j + 1);
            uint32_t lo = at, hi = e;
            while (lo < hi) {
                const uint32_t mid = lo + (hi - lo) / 2;
                if (wgt[mid] < top) lo = mid + 1;
                else hi = mid;
            }
            at = lo;
            reinterpret_cast<uint32_t *>(blocks + 4ull * v)[8 + j] = at - s;
        }
    }
}

uint32_t groups_for(uint64_t items, uint32_t most) {
    const uint64_t g = (items + kGroup - 1) / kGroup;
    return (uint32_t)(g < 1 ? 1 : g > most ? most : g);
}

uint32_t limited(const PushPullQueries &Q, uint32_t groups) {
    return Q.most_groups && Q.most_groups < groups ? Q.most_groups : groups;
}

}  // namespace

hipError_t launch_symmetry_check(const uint32_t *row, const uint32_t *col, const uint32_t *wgt, uint32_t n, uint64_t m,
                                 uint32_t *asymmetric, hipStream_t s) {
    if (m == 0) return hipSuccess;
    hipLaunchKernelGGL(symmetry_kernel, dim3((uint32_t)((m + kSymEdges - 1) / kSymEdges)), dim3(256), 0, s, row, col,
                       wgt, n, asymmetric);
    return hipGetLastError();
}

hipError_t launch_bound_counts(const uint32_t *row, const uint32_t *wgt, uint32_t n, uint32_t reach, uint4 *blocks,
                               hipStream_t s) {
    hipLaunchKernelGGL(bound_count_kernel, dim3(groups_for(n, 16384)), dim3(256), 0, s, row, wgt, n, reach, blocks);
    return hipGetLastError();
}

hipError_t launch_pushpull_reset(const PushPullQueries &Q, hipStream_t s) {
    const dim3 grid(groups_for(Q.max_n, 4096), Q.nq);
    if (Q.table) hipLaunchKernelGGL(pushpull_reset_kernel<true>, grid, dim3(256), 0, s, Q.one, Q.table);
    else hipLaunchKernelGGL(pushpull_reset_kernel<false>, grid, dim3(256), 0, s, Q.one, Q.table);
    return hipGetLastError();
}

// A workgroup reserves its places in the next round's list by one atomic, and
// those of all workgroups, on the one word, take about 15 ns each: with 2048
// workgroups of 256 threads some waited 30 us of a 35 us round of RMAT-18.  So
// the workgroups are few and large; four per CU where a round has enough work
// for them (us, RMAT-18 / 20 / 22: 2048 of 256 358 / 626 / 1119, 1024 of 512
// 304 / 537 / 1089, 512 of 512 280 / 557 / 1114, 512 of 1024 314 / 559 / 1131).
// A graph of few vertices never fills two per CU.
static uint32_t groups_of_push(uint32_t n) {
    const uint32_t most = n / 1024 < 512 ? 512 : n / 1024 < 1024 ? n / 1024 : 1024;
    return groups_for((uint64_t)n * 8, most);
}

uint32_t push_groups(const PushPullQueries &Q) {
    // several queries share the device, but a round of one may be most of the work
    const uint32_t share = 1024 / Q.nq > 128 ? 1024 / Q.nq : 128;
    const uint32_t x = limited(Q, groups_of_push(Q.max_n));
    return x < share ? x : share;
}

hipError_t launch_push(const PushPullQueries &Q, uint32_t round, bool bounded, hipStream_t s) {
    const dim3 grid(push_groups(Q), Q.nq), group(kGroup);
    if (Q.table && bounded) hipLaunchKernelGGL((push_kernel<true, true>), grid, group, 0, s, Q.one, Q.table, round);
    else if (Q.table) hipLaunchKernelGGL((push_kernel<true, false>), grid, group, 0, s, Q.one, Q.table, round);
    else if (bounded) hipLaunchKernelGGL((push_kernel<false, true>), grid, group, 0, s, Q.one, Q.table, round);
    else hipLaunchKernelGGL((push_kernel<false, false>), grid, group, 0, s, Q.one, Q.table, round);
    return hipGetLastError();
}

hipError_t launch_pushpull_summary(const PushPullLaunch &L, uint32_t rounds, PushPullSummary *out, hipStream_t s) {
    const uint32_t pushes = groups_of_push(L.n), pulls = groups_for(L.n, 2048);
    const uint32_t groups = pushes > pulls ? pushes : pulls;   // entries in use
    hipLaunchKernelGGL(pushpull_summary_kernel, dim3(1), dim3(1024), 0, s, L, groups, rounds, out);
    return hipGetLastError();
}

hipError_t launch_pull(const PushPullQueries &Q, uint32_t round, hipStream_t s) {
    const dim3 grid(limited(Q, groups_for(Q.max_n, 2048)), Q.nq), group(kGroup);
    if (Q.table) hipLaunchKernelGGL(pull_kernel<true>, grid, group, 0, s, Q.one, Q.table, round);
    else hipLaunchKernelGGL(pull_kernel<false>, grid, group, 0, s, Q.one, Q.table, round);
    return hipGetLastError();
}

}  // namespace mlmq
