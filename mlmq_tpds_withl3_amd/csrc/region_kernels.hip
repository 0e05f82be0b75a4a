// Region solver: shortest paths on a graph cut into regions that fit LDS.
//
// The vertex queue of sssp_kernels.hip pays one batch of dependent round
// trips to memory per hop of the longest shortest path (about 2.3 us), and a
// road graph has thousands of hops.  Here a hop inside a region costs a few
// LDS round trips (about 0.3 us); only the 3-4 % of edges that leave a region
// go through memory.
//
// A workgroup serves one region at a time.  Its waves share LDS words only and
// never meet at a barrier while the region is served:
//   * the relaxers own the region's vertices, two or four per lane, and hold
//     their edges in registers.  A relaxer reads its vertices' distances (8-byte
//     LDS reads), and a lane whose vertex is lower than it last
//     expanded it lowers the heads by one LDS atomicMin per edge.  There is no
//     queue: the comparison is the queue.  A lone wave issues one instruction
//     per 8 cycles and an LDS round trip takes 64, so the hop costs what its
//     instructions cost, and these are few;
//   * the sender holds the exits.  When an exit's tail fell it lowers the
//     target region's inbox slot with an agent-scope atomicMin, then marks that
//     region active;
//   * the poller reads its own region's inbox and activity word over and
//     over, applies what improves, and adopts, settles and leaves regions.
// Neighbouring served regions thus exchange distances at the latency of one
// atomic and one poll.
//
// Quiet: LDS word `version` is raised by a relaxer after the atomicMins of an
// expansion and by the poller after it applied news.  A relaxer or sender that
// finds nothing to do publishes the version it read before it looked
// (`checked`).  When every wave has checked the current version nothing is
// left: whoever had work to do has not checked a version as new as the one
// its cause raised, and a cause that has not raised the version yet is itself
// such a wave.
//
// Activity word of a region, per query, in bits:
//   kWork     has work: one credit is or will be outstanding for it
//   kCounted  that credit has been counted
//   kServed   a workgroup serves the region and polls this word
//   kVisited  its distances are in the row
//   kOver     the query is over
// A sender completes its inbox write, then sets kWork.  If it was clear, the
// sender counts a credit, only then sets kCounted, and publishes a record in
// the ring unless the region is served.  A poller that finds its region quiet
// and counted clears both bits and then reads the inbox once more: whatever was
// written by a sender that found kWork set is seen now, and the poller sets
// kWork again and keeps its credit, unless a sender did first.  Otherwise it
// returns the credit.  Leaving writes the distances back and then clears
// kServed, which fails if kWork came first.
//
// Ring: a workgroup without a region takes the next ticket (kHeadOff) and
// polls that slot alone; a sender takes the next position (kRingTailOff) and
// publishes there.  A region is left as soon as it has returned its credit.
// (Regions that keep a workgroup were tried where every region has one: to
// poll an idle region's word is faster than a record, a ticket and the region's
// edges from L2 anew, but the pollers slow everyone: road 264k 631 against
// 595 us, 4-NN 700k 1335 against 965 us.)  No workgroup ever waits for another
// one to become resident.
//
// Termination: a query's credits are counted before they can be returned.  Work
// in a region is covered by its own credit, or by that of the sender whose
// message caused it and which has not finished marking; a region returns its
// credit only when it is quiet and everything it sent is marked.  So the return
// that leaves none proves that the query is over; its workgroup publishes seeds
// of queries that wait, by how many workgroups wait for a record, and marks every
// region of this one kOver.
// Whoever ends the last query publishes one exit record per workgroup of the
// grid, for the ticket each of them takes last.
//
// Errors: a workgroup that sees the error word set or its deadline passed ends.
// In a launch over a table of queries it writes its region's distances out
// first: a region that is left this way with work keeps its credit outstanding,
// so a query that was over by then has all of its distances in the row, and no
// other one ends any more (qtime tells which).  Launches on one graph answer all
// of their queries or none; there the write costs road 6.26M 1.4 % by what the
// compiler makes of the poller's registers.
//
// Measured, device us of one query, vertex queue / here: 2,052 vertices 190 / 41,
// 264k 1250 / 430, 1.06M 4500 / 800-1000, 6.26M 5850 / 1850; 64 queries on 264k
// 14100 / 2600.  Bound: hops one after another (about 0.25 us each inside a
// region) and crossings between regions (about 8 us: inbox, mark, credit, ring
// record, adoption); LDS bank conflicts are below 1 % of the cycles and memory
// traffic (0.7 GB on 6.26M) is 5 % of the peak.
#include <algorithm>
#include <cmath>
#include "device_common.h"
#include "region_solver.h"
#include "solver_internal.h"

namespace mlmq {

namespace {

constexpr uint32_t kRingTailOff = kHungryOff;   // ring positions taken
constexpr uint32_t kNextOff = kHeadOff + kStride;           // queries admitted
constexpr uint32_t kFinishedOff = kHeadOff + 2 * kStride;   // queries over
constexpr uint32_t kLeftOff = kHeadOff + 3 * kStride;       // workgroups that are done
constexpr uint32_t kResetOff = kHeadOff + 4 * kStride;      // ticks of the reset and the
constexpr uint32_t kStartOff = kHeadOff + 5 * kStride;      // solver's start (64 bits)
constexpr uint32_t kWork = 1, kCounted = 2, kServed = 4, kVisited = 8, kOver = 16;
// Quiet polls before an active region returns its credit.
constexpr uint32_t kSettle = 2;
// Record: low word region | flags, high word query | seed's local id << 20.
constexpr uint32_t kSeedFlag = 0x80000000u;
constexpr uint32_t kVisitFlag = 0x40000000u;    // the region's distances are in the row
constexpr uint32_t kQueryBits = 20;
static_assert(kRegionQueries == 1u << kQueryBits && kQueryBits + kRegionIdBits <= 32, "record");

// Threads of a workgroup with kR relaxing waves and its waves resident per SIMD.
template <uint32_t kR> constexpr uint32_t kThreads = (kR + 2) * kWave;
template <uint32_t kR> constexpr uint32_t kPerSimd = kR == kFew ? 6 : 5;

struct RegionArgs {
    const RegionHdr *hdr;        // nq queries on one graph ...
    const uint32_t *image;
    const uint32_t *verts;
    RegionQuerySpace space;
    const RegionQuery *table;    // ... or each on its own
    RegionProgress *progress;    // per query
    uint32_t nq, admit;
    uint64_t *ring;
    uint32_t ring_mask;
    RegionCounts *counts;
    uint32_t *ctl;
    RegionSummary *summary;
    uint64_t *qtime;
    uint64_t timeout_ticks;
    uint32_t regions;
    uint32_t width;          // window of a wave's expansions
};

constexpr uint32_t kCounters = sizeof(RegionCounts) / sizeof(uint64_t);

struct RegionLds {
    alignas(16) uint32_t dist[kRegionVerts];
    uint32_t version;
    uint32_t over;                     // the region is left: a wave without work returns
    uint32_t checked[kMany + 1];       // relaxers, sender
    uint32_t rec[2];                   // adopted record
    uint32_t last;                     // this workgroup is the last one
    unsigned long long total[kCounters];
};

__device__ __forceinline__ uint32_t sh_ld(uint32_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void sh_st(uint32_t *p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ uint32_t sh_min(uint32_t *p, uint32_t v) {
    return __hip_atomic_fetch_min(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void sh_add(uint32_t *p, uint32_t v) {
    (void)__hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ uint32_t fetch_or(uint32_t *p, uint32_t v) {
    return __hip_atomic_fetch_or(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Rank of this lane among the set lanes of `m`.
__device__ __forceinline__ uint32_t rank_of(uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}
// This lane's id, computed anew: keeps one wave's address arithmetic out of the
// other waves' registers.
__device__ __forceinline__ uint32_t fresh_lane() {
    uint32_t lane = lane_id();
    asm volatile("" : "+v"(lane));
    return lane;
}
// Every outstanding load, store and atomic of this wave is complete.
__device__ __forceinline__ void wait_memory() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// LDS accesses of a wave execute in order; this keeps the compiler's order too.
__device__ __forceinline__ void lds_order() { asm volatile("" ::: "memory"); }
__device__ __forceinline__ uint32_t *at_offset(uint32_t *base, uint32_t bytes) {
    return reinterpret_cast<uint32_t *>(reinterpret_cast<char *>(base) + bytes);
}

// ---- a relaxer ----

struct RelaxStats {
    uint32_t relax, improve, sweeps;
};

typedef uint32_t Pair __attribute__((ext_vector_type(2)));

// Waits for a version other than `checked`.  A wave that has waited a while
// naps longer: it leaves the issue slots to the waves of active regions.
__device__ __forceinline__ void wait_version(RegionLds &S, uint32_t checked) {
    for (uint32_t turn = 0; uniform(sh_ld(&S.version)) == checked; ++turn) {
        if (turn < 32) __builtin_amdgcn_s_sleep(1);
        else __builtin_amdgcn_s_sleep(8);
    }
}

// Least value of the wave.
__device__ __forceinline__ uint32_t wave_least(uint32_t x) {
    // as a maximum of the complements: lanes outside a row keep the identity 0
    return ~read_lane(wave_incl_max(~x), kWave - 1);
}

// More lowered vertices than this in a wave are expanded in order.
constexpr uint32_t kWindowCount = 16;

// Lower the heads of edges kFrom .. kTo - 1 of this lane's vertex at distance d.
template <uint32_t kFrom, uint32_t kTo>
__device__ __forceinline__ void lower_heads(RegionLds &S, const uint32_t (&edge)[kLaneEdges], uint32_t mask,
                                            uint32_t shift, uint32_t d) {
#pragma unroll
    for (uint32_t k = kFrom; k < kTo; ++k) (void)sh_min(at_offset(S.dist, edge[k] & mask), d + (edge[k] >> shift));
}

template <uint32_t kR>
__device__ __forceinline__ void run_relaxer(RegionLds &S, const RegionHdr &h, const uint32_t *image,
                                            const uint32_t *verts, uint32_t *dist, bool visited, uint32_t w,
                                            uint32_t width, RelaxStats &st) {
    const uint32_t lane = fresh_lane();
    constexpr uint32_t kLaneVerts = kRegionVerts / (kR * kWave);
    constexpr uint32_t kStep = kR * kWave;   // from one of a lane's vertices to the next
    const uint32_t thread = w * kWave + lane;
    uint32_t edge[kLaneVerts][kLaneEdges], last[kLaneVerts], most[kLaneVerts];
    uint32_t degrees = 0;   // edges of each vertex, 8 bits each
    // the distances, by way of the vertex list, beside the edges
    uint32_t start[kLaneVerts], vert[kLaneVerts];
#pragma unroll
    for (uint32_t i = 0; i < kLaneVerts; ++i) start[i] = kUnreached;
    if (visited) {
#pragma unroll
        for (uint32_t i = 0; i < kLaneVerts; ++i) vert[i] = verts[min(i * kStep + thread, h.nv - 1u)];
    }
#pragma unroll
    for (uint32_t i = 0; i < kLaneVerts; ++i)
#pragma unroll
        for (uint32_t k = 0; k < kLaneEdges; ++k) edge[i][k] = image[k * kRegionVerts + i * kStep + thread];
    if (visited) {
#pragma unroll
        for (uint32_t i = 0; i < kLaneVerts; ++i) {
            const uint32_t x = ld_relaxed(dist + vert[i]);
            start[i] = i * kStep + thread < h.nv ? x : kUnreached;
        }
    }
    // pair j: this lane's vertices j and j + kPairs
    constexpr uint32_t kPairs = kLaneVerts / 2;
    Pair *own = reinterpret_cast<Pair *>(S.dist) + thread;
#pragma unroll
    for (uint32_t j = 0; j < kPairs; ++j) own[j * kStep] = Pair{start[j], start[j + kPairs]};
#pragma unroll
    for (uint32_t i = 0; i < kLaneVerts; ++i) {
        most[i] = image[kImageMost + i * kR + w];
        // a vertex is expanded below `last` (a region that was left is expanded
        // as far as it has distances); past the end: never
        last[i] = i * kStep + thread < h.nv ? start[i] : 0u;
#pragma unroll
        for (uint32_t k = 0; k < kLaneEdges; ++k) {
            if (edge[i][k] >> kWeightShift != kNoWeight) degrees += 1u << 8 * i;
        }
    }
    __syncthreads();
    if (visited) __syncthreads();   // until the sender has read them
    uint32_t checked = 0, expanded = 0, sweeps = 0;
    for (;;) {
        // the version before the distances
        const uint32_t seen = sh_ld(&S.version);
        lds_order();
        uint32_t cur[kLaneVerts];
#pragma unroll
        for (uint32_t j = 0; j < kPairs; ++j) {
            const Pair now = own[j * kStep];
            cur[j] = now[0];
            cur[j + kPairs] = now[1];
        }
        lds_order();
        // edges are decoded as they are used: kept decoded, they would not fit
        // the registers (the compiler must not see the constants)
        uint32_t mask = kOffsetMask, shift = kWeightShift;
        asm volatile("" : "+s"(mask), "+s"(shift));
        uint64_t low[kLaneVerts], any = 0;
        uint32_t count = 0;
#pragma unroll
        for (uint32_t i = 0; i < kLaneVerts; ++i) {
            low[i] = ballot(cur[i] < last[i]);
            any |= low[i];
            count += popc(low[i]);
        }
        if (any == 0) {
            checked = uniform(seen);
            if (uniform(sh_ld(&S.over))) break;
            if (lane == 0) sh_st(&S.checked[w], checked);
            wait_version(S, checked);
            continue;
        }
        // Many at once: only those within `width` of the least (the others
        // stay lower than last expanded, and come up again)
        uint32_t limit = kUnreached;
        if (count > kWindowCount) {
            uint32_t least = kUnreached;
#pragma unroll
            for (uint32_t i = 0; i < kLaneVerts; ++i) least = min(least, cur[i] < last[i] ? cur[i] : kUnreached);
            limit = wave_least(least) + width;
#pragma unroll
            for (uint32_t i = 0; i < kLaneVerts; ++i) low[i] = ballot(cur[i] < last[i] && cur[i] <= limit);
        }
#pragma unroll
        for (uint32_t i = 0; i < kLaneVerts; ++i) {
            if (low[i] == 0) continue;
            expanded += popc(low[i]);
            if (cur[i] < last[i] && cur[i] <= limit) {
                last[i] = cur[i];
                st.relax += (degrees >> 8 * i) & 0xFFu;   // per lane
                lower_heads<0, kLaneEdges / 2>(S, edge[i], mask, shift, cur[i]);
                if (most[i] > kLaneEdges / 2) lower_heads<kLaneEdges / 2, kLaneEdges>(S, edge[i], mask, shift, cur[i]);
            }
        }
        sweeps += 1;
        lds_order();
        if (lane == 0) sh_add(&S.version, 1u);
    }
    st.improve += expanded;
    st.sweeps += sweeps;
}

// ---- the sender and the poller ----

struct MessageStats {
    uint32_t credits, activations, messages, polls;
};

__device__ __forceinline__ void region_raise(const RegionArgs &a, uint32_t code) {
    if (lane_id() == 0) {
        cas32(a.ctl + kErrOff, kErrNone, code);
    }
}

// Publish the records of the lanes with `valid` set.
__device__ __forceinline__ void ring_push(const RegionArgs &a, bool valid, uint64_t rec) {
    const uint64_t m = ballot(valid);
    if (m == 0) return;
    uint32_t pos0 = 0;
    if (lane_id() == 0) pos0 = fetch_add(a.ctl + kRingTailOff, popc(m));
    const uint32_t pos = read_lane(pos0, 0) + rank_of(m);
    bool ok = true;
    if (valid) {
        uint64_t *slot = a.ring + (pos & a.ring_mask);
        uint32_t spins = 0;
        while (!cas64(slot, kEmpty, rec)) {
            if (++spins > kSpinLimit) {
                ok = false;
                break;
            }
            __builtin_amdgcn_s_sleep(2);
        }
    }
    if (ballot(!ok)) region_raise(a, kErrOverflow);
}

template <uint32_t kR, int kG>
__device__ __forceinline__ void run_sender(const RegionArgs &a, RegionLds &S, const RegionHdr &h,
                                           const uint32_t *image, bool visited, uint32_t query, uint32_t *inbox_all,
                                           uint32_t *act, MessageStats &st) {
    const uint32_t lane = fresh_lane();
    const uint32_t *exits = image + kImageExits;
    uint32_t edge[kG], slot[kG], reg[kG], last[kG];   // last: least distance sent
#pragma unroll
    for (int g = 0; g < kG; ++g) {
        const uint32_t x = g * kWave + lane;
        edge[g] = x < h.nx ? exits[x] : 0u;
        slot[g] = x < h.nx ? exits[h.nx + x] : 0u;
        reg[g] = x < h.nx ? exits[2 * h.nx + x] : 0u;
        last[g] = x < h.nx ? kUnreached : 0u;         // 0: never sends
    }
    __syncthreads();
    if (visited) {   // what the adopted distances give was sent before
#pragma unroll
        for (int g = 0; g < kG; ++g)
            last[g] = min(last[g], sh_ld(at_offset(S.dist, edge[g] & kOffsetMask)) + (edge[g] >> kWeightShift));
        __syncthreads();
    }
    for (;;) {
        const uint32_t version = uniform(sh_ld(&S.version));
        if (uniform(sh_ld(&S.over))) break;
        lds_order();
        uint32_t d[kG], was[kG], state[kG];
#pragma unroll
        for (int g = 0; g < kG; ++g) d[g] = sh_ld(at_offset(S.dist, edge[g] & kOffsetMask));
        bool send = false;
#pragma unroll
        for (int g = 0; g < kG; ++g) {
            d[g] += edge[g] >> kWeightShift;
            send = send || d[g] < last[g];
        }
        if (ballot(send) == 0) {
            if (lane == 0) sh_st(&S.checked[kR], version);
            wait_version(S, version);
            continue;
        }
#pragma unroll
        for (int g = 0; g < kG; ++g) {
            was[g] = 0;
            if (d[g] < last[g]) {
                was[g] = fetch_min(inbox_all + slot[g], d[g]);
                last[g] = d[g];
                st.messages += 1;   // per lane
            }
        }
#pragma unroll
        for (int g = 0; g < kG; ++g) asm volatile("" : "+v"(was[g])::"memory");   // complete before the marks
#pragma unroll
        for (int g = 0; g < kG; ++g) {
            state[g] = kWork;
            if (was[g] > d[g]) state[g] = fetch_or(act + reg[g], kWork);
        }
#pragma unroll
        for (int g = 0; g < kG; ++g) asm volatile("" : "+v"(state[g])::"memory");
        uint32_t woken = 0;
#pragma unroll
        for (int g = 0; g < kG; ++g) woken += popc(ballot(!(state[g] & kWork)));
        if (woken) {
            st.activations += lane == 0 ? woken : 0u;
            uint32_t t = 0;
            if (lane == 0) t = fetch_add(&a.progress[query].credits, woken);
            asm volatile("" : "+v"(t)::"memory");   // counted before it can be returned
#pragma unroll
            for (int g = 0; g < kG; ++g) {
                const bool wake = !(state[g] & kWork);
                if (wake) (void)fetch_or(act + reg[g], kCounted);
            }
#pragma unroll
            for (int g = 0; g < kG; ++g)
                ring_push(a, !(state[g] & (kWork | kServed)),
                          (uint64_t)query << 32 | reg[g] | (state[g] & kVisited ? kVisitFlag : 0u));
            wait_memory();
        }
    }
}

// Return a credit.  The query's last one ends it: the next query is admitted,
// and the last query ends the solve.
__device__ __forceinline__ void return_credit(const RegionArgs &a, uint32_t query, uint32_t *act, uint32_t regions,
                                              MessageStats &st) {
    const uint32_t lane = fresh_lane();
    st.credits += lane == 0 ? 1u : 0u;
    uint32_t held = 0;
    if (lane == 0) held = fetch_add(&a.progress[query].credits, ~0u);
    asm volatile("" : "+v"(held)::"memory");
    if (read_lane(held, 0) != 1u) return;
    if (a.qtime && lane == 0) a.qtime[2 * query + 1] = wall_clock64();
    uint32_t over = 0;
    if (lane == 0) over = fetch_add(a.ctl + kFinishedOff, 1u) + 1u;
    over = read_lane(over, 0);
    if (a.admit < a.nq) {
        // For this query the next one, in general; two while a third of the
        // workgroups wait for a record, and none while hardly any does (other
        // launches may have kept some from starting), unless none is left.
        // (64 queries on 100k 1168 us one for one, 1053 this way; on 264k 2705 and
        // 2830; lanes at 2000 queries/s offered: 790 and 1411 served.)
        const uint32_t admitted = uniform(ld_relaxed(a.ctl + kNextOff));
        const int32_t idle = (int32_t)(uniform(ld_relaxed(a.ctl + kHeadOff)) - uniform(ld_relaxed(a.ctl + kRingTailOff)));
        uint32_t want = idle >= (int32_t)gridDim.x / 3 ? 2u : idle > (int32_t)gridDim.x / 64 ? 1u : 0u;
        if (over == admitted) want = max(want, 1u);
        for (uint32_t k = 0; k < want && admitted < a.nq; ++k) {
            uint32_t next = 0;
            if (lane == 0) next = fetch_add(a.ctl + kNextOff, 1u);
            next = read_lane(next, 0);
            if (next >= a.nq) break;
            if (a.qtime && lane == 0) a.qtime[2 * next] = wall_clock64();
            ring_push(a, lane == 0, a.progress[next].seed);
        }
    }
    for (uint32_t i = lane; i < regions; i += kWave) st_relaxed(act + i, kOver);
    wait_memory();
    if (over != a.nq) return;
    const uint32_t ring_tail = uniform(ld_relaxed(a.ctl + kRingTailOff));
    for (uint32_t i = lane; i < gridDim.x; i += kWave) {
        uint64_t *slot = a.ring + ((ring_tail + i) & a.ring_mask);
        __hip_atomic_store(slot, kRegionExit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Serves the adopted region until it is left or the solve is over.
template <bool kTable, uint32_t kR, int kG>
__device__ __forceinline__ void run_poller(const RegionArgs &a, RegionLds &S, const RegionHdr &h,
                                           const uint32_t *image, const uint32_t *verts, uint32_t region,
                                           uint32_t query, uint32_t *dist, uint32_t *inbox, uint32_t *act,
                                           uint32_t regions, uint32_t seed, bool visited, uint64_t deadline,
                                           MessageStats &st) {
    const uint32_t lane = fresh_lane();
    uint32_t to[kG], seen[kG], val[kG];
#pragma unroll
    for (int g = 0; g < kG; ++g) {
        const uint32_t x = g * kWave + lane;
        to[g] = x < h.nin ? image[image_inbox(h) + x] : 0u;
        seen[g] = x < h.nin ? kUnreached : 0u;   // 0: never news
    }
    // slots past the end repeat the last one (a region without any reads the
    // spare word behind the inboxes or its neighbour's, and ignores it)
    uint32_t at[kG];
#pragma unroll
    for (int g = 0; g < kG; ++g) at[g] = min(g * kWave + lane, h.nin ? h.nin - 1u : 0u);
    uint32_t quiet = 0;
    bool dirty = false, idle = false;
    const uint32_t base = kServed | (visited ? kVisited : 0u);
    __syncthreads();
    if (visited) __syncthreads();
    // the waves look once at the adopted distances in any case: a version they
    // have not checked
    if (lane == 0) {
        if (seed) sh_st(S.dist + (seed - 1u), 0u);
        lds_order();
        sh_add(&S.version, 1u);
    }
    dirty = seed != 0;
    for (uint32_t turn = 0;; ++turn) {
        if ((turn & 31u) == 0) {
            bool stop = uniform(ld_relaxed(a.ctl + kErrOff)) != 0;
            if (!stop && wall_clock64() > deadline) {
                region_raise(a, kErrTimeout);
                stop = true;
            }
            if (stop) {
                // (this query may be over, and others be asked for)
                if constexpr (kTable) break;
                else return;
            }
        }
        st.polls += lane == 0 ? 1u : 0u;
        if (idle) {
            const uint32_t state = uniform(ld_relaxed(act + region));
            if (state & kOver) break;
            if (!(state & kWork)) {
                if (dirty) {
                    for (uint32_t i = lane; i < h.nv; i += kWave) {
                        const uint32_t x = sh_ld(S.dist + local_id(i));
                        if (x < kUnreached) st_relaxed(dist + verts[i], x);
                    }
                    dirty = false;
                }
                wait_memory();
                uint32_t left = 0;
                if (lane == 0) left = cas32(act + region, base, kVisited) ? 1u : 0u;
                if (read_lane(left, 0)) return;
                continue;
            }
            // (a sender marks the region after its message)
            idle = false;
        }
#pragma unroll
        for (int g = 0; g < kG; ++g) val[g] = ld_relaxed(inbox + at[g]);
        bool news = false, lower = false;
#pragma unroll
        for (int g = 0; g < kG; ++g) {
            if (val[g] < seen[g]) {
                news = true;
                seen[g] = val[g];
                lower = sh_min(at_offset(S.dist, to[g]), val[g]) > val[g] || lower;
            }
        }
        if (ballot(lower)) {
            lds_order();
            if (lane == 0) sh_add(&S.version, 1u);
        }
        if (ballot(news)) {
            dirty = true;
            quiet = 0;
            continue;
        }
        // the checks before the version: it only grows
        const uint32_t done = sh_ld(&S.checked[min(lane, kR)]);
        lds_order();
        if (ballot(done != uniform(sh_ld(&S.version)))) {
            quiet = 0;
            continue;
        }
        if (++quiet < kSettle) continue;
        quiet = 0;
        uint32_t cleared = 0;
        if (lane == 0) cleared = cas32(act + region, base | kWork | kCounted, base) ? 1u : 0u;
        asm volatile("" : "+v"(cleared)::"memory");
        if (!read_lane(cleared, 0)) continue;   // its sender is about to count the credit
        bool more = false;
#pragma unroll
        for (int g = 0; g < kG; ++g) val[g] = ld_relaxed(inbox + at[g]);
#pragma unroll
        for (int g = 0; g < kG; ++g) more = more || val[g] < seen[g];
        if (ballot(more) == 0) {
            idle = true;
            return_credit(a, query, act, regions, st);
            continue;
        }
        uint32_t was = 0;
        if (lane == 0) was = fetch_or(act + region, kWork);
        asm volatile("" : "+v"(was)::"memory");
        if (read_lane(was, 0) & kWork) return_credit(a, query, act, regions, st);   // a sender's credit covers the news
        else if (lane == 0) (void)fetch_or(act + region, kCounted);
    }
    // the query or the solve is over
    if (dirty)
        for (uint32_t i = lane; i < h.nv; i += kWave) {
            const uint32_t x = sh_ld(S.dist + local_id(i));
            if (x < kUnreached) dist[verts[i]] = x;
        }
}

template <bool kTable, uint32_t kR>
__global__ __launch_bounds__(kThreads<kR>, kPerSimd<kR>) void region_solver_kernel(RegionArgs a) {
    __shared__ RegionLds S;
    const uint32_t wave = uniform(threadIdx.x / kWave);
    const uint32_t lane = lane_id();
    const uint64_t deadline = wall_clock64() + a.timeout_ticks;
    RelaxStats rs{};
    MessageStats ms{};
    if (blockIdx.x == 0 && threadIdx.x == 0)
        __hip_atomic_store(reinterpret_cast<uint64_t *>(a.ctl + kStartOff), (uint64_t)wall_clock64(), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    for (;;) {
        // adopt the next ticket's region
        if (wave == kR && lane == 0) {
            uint64_t *slot = a.ring + (fetch_add(a.ctl + kHeadOff, 1u) & a.ring_mask);
            uint64_t rec;
            for (uint32_t turn = 1;; ++turn) {
                rec = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (rec != kEmpty) {
                    xchg64(slot, kEmpty);
                    break;
                }
                // after an error no record will come; a finished solve has put
                // this ticket's exit record in place
                if ((turn & 15u) == 0 && (ld_relaxed(a.ctl + kErrOff) || wall_clock64() > deadline)) {
                    rec = kRegionExit;
                    break;
                }
                __builtin_amdgcn_s_sleep(4);
            }
            if (rec != kRegionExit) {
                // (its word: kWork, kCounted and perhaps kVisited)
                const uint32_t q = (uint32_t)(rec >> 32) & (kRegionQueries - 1u);
                const uint32_t r = (uint32_t)rec & ~(kSeedFlag | kVisitFlag);
                (void)fetch_or((kTable ? a.table[q].act : a.space.act + q * a.space.act_stride) + r, kServed);
            }
            S.rec[0] = (uint32_t)rec;
            S.rec[1] = (uint32_t)(rec >> 32);
            S.version = S.over = 0;
            for (uint32_t i = 0; i <= kR; ++i) S.checked[i] = 0;
        }
        __syncthreads();
        const uint32_t rec_lo = uniform(S.rec[0]), rec_hi = uniform(S.rec[1]);
        if (((uint64_t)rec_hi << 32 | rec_lo) == kRegionExit) break;
        const uint32_t region = rec_lo & ~(kSeedFlag | kVisitFlag);
        const uint32_t query = rec_hi & ((1u << kQueryBits) - 1u);
        const uint32_t seed = rec_lo & kSeedFlag ? (rec_hi >> kQueryBits) + 1u : 0u;
        const RegionQuery *of = kTable ? a.table + query : nullptr;
        uint32_t *dist = kTable ? of->dist : a.space.dist + query * a.space.dist_stride;
        uint32_t *inbox = kTable ? of->inbox : a.space.inbox + query * a.space.inbox_stride;
        uint32_t *act = kTable ? of->act : a.space.act + query * a.space.act_stride;
        const RegionHdr h = (kTable ? of->hdr : a.hdr)[region];
        const uint32_t *image = (kTable ? of->image : a.image) + h.image;
        const uint32_t *verts = (kTable ? of->verts : a.verts) + h.first;
        const uint32_t width = kTable ? of->width : a.width;
        const uint32_t regions = kTable ? of->regions : a.regions;
        const bool visited = (rec_lo & kVisitFlag) != 0;
        // (each role loads what it holds, then meets the others once)
        if (wave < kR) {
            run_relaxer<kR>(S, h, image, verts, dist, visited, wave, width, rs);
        } else if (wave == kR) {
            uint32_t *in = inbox + h.inbox;
            if (h.nin <= 2 * kWave) run_poller<kTable, kR, 2>(a, S, h, image, verts, region, query, dist, in, act, regions, seed, visited, deadline, ms);
            else if (h.nin <= 4 * kWave) run_poller<kTable, kR, 4>(a, S, h, image, verts, region, query, dist, in, act, regions, seed, visited, deadline, ms);
            else run_poller<kTable, kR, 6>(a, S, h, image, verts, region, query, dist, in, act, regions, seed, visited, deadline, ms);
            if (lane == 0) {
                sh_st(&S.over, 1u);
                lds_order();
                sh_add(&S.version, 1u);   // wakes the waiting waves
            }
        } else if (wave == kR + 1) {
            if (h.nx <= 2 * kWave) run_sender<kR, 2>(a, S, h, image, visited, query, inbox, act, ms);
            else if (h.nx <= 4 * kWave) run_sender<kR, 4>(a, S, h, image, visited, query, inbox, act, ms);
            else run_sender<kR, 6>(a, S, h, image, visited, query, inbox, act, ms);
        }
        __syncthreads();
    }
    // What the workgroup did goes to its own entry; whoever is last adds them up
    // (a thousand workgroups that add to the same words take tens of us).
    if (threadIdx.x < kCounters) S.total[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t mine[kCounters] = {ms.credits, ms.activations, ms.messages, ms.polls, rs.relax, 0, 0, 0};
#pragma unroll
    for (uint32_t k = 0; k < kCounters; ++k)
        if (mine[k]) atomicAdd(&S.total[k], (unsigned long long)mine[k]);
    if (wave < kR && lane == 0) {
        atomicAdd(&S.total[5], (unsigned long long)rs.improve);
        atomicAdd(&S.total[6], (unsigned long long)rs.sweeps);
    }
    __syncthreads();
    auto *entry = reinterpret_cast<uint64_t *>(a.counts + blockIdx.x);
    if (wave == 0) {
        if (lane < kCounters)
            __hip_atomic_store(entry + lane, (uint64_t)S.total[lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        wait_memory();
        if (lane == 0) S.last = fetch_add(a.ctl + kLeftOff, 1u) == gridDim.x - 1 ? 1u : 0u;
        if (lane < kCounters) S.total[lane] = 0;
    }
    __syncthreads();
    if (!S.last) return;
    for (uint32_t i = threadIdx.x; i < gridDim.x * kCounters; i += kThreads<kR>) {
        const uint64_t x = __hip_atomic_load(reinterpret_cast<uint64_t *>(a.counts) + i, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
        if (x) atomicAdd(&S.total[i % kCounters], (unsigned long long)x);
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    RegionSummary out;
    out.all = {S.total[0], S.total[1], S.total[2], S.total[3], S.total[4], S.total[5], S.total[6], 0};
    out.reset = *reinterpret_cast<uint64_t *>(a.ctl + kResetOff);
    out.start = __hip_atomic_load(reinterpret_cast<uint64_t *>(a.ctl + kStartOff), __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT);
    out.error = ld_relaxed(a.ctl + kErrOff);
    out.over = ld_relaxed(a.ctl + kFinishedOff) == a.nq ? 1u : 0u;
    a.ctl[kTailOff] = a.nq + (uint32_t)out.all.activations;
    a.ctl[kTakenOff] = a.ctl[kDoneOff] = (uint32_t)out.all.credits;
    a.ctl[kExitOff] = out.over;
    out.end = wall_clock64();
    if (a.summary) *a.summary = out;
}

// ---- reset ----

template <bool kTable>
__global__ __launch_bounds__(256) void region_reset_kernel(RegionArgs a, uint32_t n, uint32_t slots,
                                                           const uint32_t *sources, uint32_t src,
                                                           const uint32_t *where) {
    const uint32_t stride = gridDim.x * blockDim.x;
    const uint32_t t0 = blockIdx.x * blockDim.x + threadIdx.x;
    for (uint32_t q = blockIdx.y; q < a.nq; q += gridDim.y) {
        uint32_t s, *dist, *inbox, *act, at, regions = a.regions;
        if constexpr (kTable) {
            const RegionQuery &of = a.table[q];
            s = of.src;
            dist = of.dist;
            inbox = of.inbox;
            act = of.act;
            at = of.where[s];
            n = of.n;
            slots = of.slots;
            regions = of.regions;
        } else {
            s = sources ? sources[q] : src;
            dist = a.space.dist + q * a.space.dist_stride;
            inbox = a.space.inbox + q * a.space.inbox_stride;
            act = a.space.act + q * a.space.act_stride;
            at = where[s];
        }
        for (uint32_t i = t0; i < n; i += stride) dist[i] = i == s ? 0u : kUnreached;
        for (uint32_t i = t0; i < slots; i += stride) inbox[i] = kUnreached;
        for (uint32_t i = t0; i < regions; i += stride) act[i] = i == at >> kRegionIdBits ? kWork | kCounted : 0u;
        if (t0 == 0) {
            const uint64_t seed = (uint64_t)((at & (kRegionVerts - 1u)) << kQueryBits | q) << 32 | kSeedFlag | at >> kRegionIdBits;
            a.progress[q] = {seed, 1u, 0u};
            if (q < a.admit) a.ring[q] = seed;
            if (a.qtime) {
                a.qtime[2 * q] = wall_clock64();
                a.qtime[2 * q + 1] = 0;
            }
        }
    }
    if (blockIdx.y == 0)
        for (uint32_t i = t0; i < kCtlWords; i += stride) {
            if (i == kResetOff) *reinterpret_cast<uint64_t *>(a.ctl + i) = wall_clock64();
            else if (i != kResetOff + 1) a.ctl[i] = i == kRingTailOff || i == kNextOff ? a.admit : 0u;
        }
}

// ---- building ----

__global__ __launch_bounds__(256) void region_where_kernel(const uint32_t *verts, const uint32_t *first,
                                                           uint32_t *where) {
    const uint32_t r = blockIdx.x, lo = first[r], hi = first[r + 1];
    for (uint32_t i = lo + threadIdx.x; i < hi; i += blockDim.x)
        where[verts[i]] = r << kRegionIdBits | local_id(i - lo);
}

// Per region: exits and crossing edges.  Each exit takes an inbox slot of the region it enters:
// tmp[e] = its number there.
__global__ __launch_bounds__(256) void region_count_kernel(const uint32_t *row, const uint32_t *col,
                                                           const uint32_t *verts, const uint32_t *where,
                                                           RegionHdr *hdr, uint32_t *tmp) {
    __shared__ uint32_t nx, cross;
    RegionHdr &h = hdr[blockIdx.x];
    if (threadIdx.x == 0) nx = cross = 0;
    __syncthreads();
    uint32_t mx = 0, mine = 0;
    for (uint32_t i = threadIdx.x; i < h.nv; i += blockDim.x) {
        const uint32_t u = verts[h.first + i], lo = row[u], hi = row[u + 1];
        uint32_t inside = 0;
        for (uint32_t e = lo; e < hi; ++e) {
            const uint32_t r = where[col[e]] >> kRegionIdBits;
            mine += r != blockIdx.x ? 1u : 0u;
            if (r == blockIdx.x && inside++ < kLaneEdges) continue;
            ++mx;
            tmp[e] = atomicAdd(&hdr[r].nin, 1u);
        }
    }
    atomicAdd(&nx, mx);
    atomicAdd(&cross, mine);
    __syncthreads();
    if (threadIdx.x == 0) {
        h.nx = nx;
        h.cross = cross;
    }
}

__global__ __launch_bounds__(256) void region_image_kernel(const uint32_t *row, const uint32_t *col,
                                                                      const uint32_t *wgt, const uint32_t *verts,
                                                                      const uint32_t *where, const RegionHdr *hdr,
                                                                      const uint32_t *tmp, uint32_t *image) {
    __shared__ uint32_t most[kBlocks], exits;
    const RegionHdr h = hdr[blockIdx.x];
    uint32_t *img = image + h.image;
    if (threadIdx.x < kBlocks) most[threadIdx.x] = 0;
    if (threadIdx.x == 0) exits = 0;
    __syncthreads();
    uint32_t *xedge = img + kImageExits, *xslot = xedge + h.nx, *xreg = xslot + h.nx;
    for (uint32_t p = threadIdx.x; p < kRegionVerts; p += blockDim.x) {
        const uint32_t own = 4 * local_id(p);
        uint32_t inside = 0;
        if (p < h.nv) {
            const uint32_t u = verts[h.first + p], lo = row[u], hi = row[u + 1];
            for (uint32_t e = lo; e < hi; ++e) {
                const uint32_t to = where[col[e]], r = to >> kRegionIdBits, head = 4 * (to & (kRegionVerts - 1u));
                if (r == blockIdx.x && inside < kLaneEdges) {
                    img[inside * kRegionVerts + p] = head | wgt[e] << kWeightShift;
                    ++inside;
                    continue;
                }
                const RegionHdr &t = hdr[r];
                const uint32_t x = atomicAdd(&exits, 1u);
                xedge[x] = own | wgt[e] << kWeightShift;
                xslot[x] = t.inbox + tmp[e];
                xreg[x] = r;
                image[t.image + image_inbox(t) + tmp[e]] = head;
            }
        }
        atomicMax(&most[p / kWave], inside);
        // absent edges: to the vertex itself, which they cannot lower
        for (uint32_t k = inside; k < kLaneEdges; ++k)
            img[k * kRegionVerts + p] = own | kNoWeight << kWeightShift;
    }
    __syncthreads();
    if (threadIdx.x < kBlocks) img[kImageMost + threadIdx.x] = most[threadIdx.x];
}

RegionArgs make_region_args(const RegionGraph &g, const RegionLaunch &L) {
    RegionArgs a;
    a.hdr = g.hdr;
    a.image = g.image;
    a.verts = g.verts;
    a.space = L.space;
    a.table = L.table;
    a.progress = L.progress;
    a.nq = L.nq;
    a.admit = L.admit;
    a.ring = L.ring;
    a.ring_mask = L.ring_mask;
    a.counts = L.counts;
    a.ctl = L.ctl;
    a.summary = L.summary;
    a.qtime = L.qtime;
    a.timeout_ticks = L.timeout_ticks;
    a.regions = g.regions;
    a.width = g.width;
    return a;
}

}  // namespace

hipError_t region_occupancy(uint32_t relaxers, int *blocks_per_cu) {
    // (with and without a table the kernels need the same)
    const void *k = relaxers == kMany ? reinterpret_cast<const void *>(&region_solver_kernel<true, kMany>)
                                      : reinterpret_cast<const void *>(&region_solver_kernel<true, kFew>);
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(
        blocks_per_cu, k, (int)(relaxers == kMany ? kThreads<kMany> : kThreads<kFew>), 0);
}

// A hop is shorter where eight waves with two vertices per lane do what four
// waves with four do (their loop has half the instructions, and a lone wave
// issues one per 8 cycles), but only two such workgroups fit a CU, not four.
// So few relaxers once the wavefronts of all queries (see region_admit) may
// fill those, also from the middle of the graph.  us at 4 / 8 relaxers, by
// nq sqrt(regions): a query on 2k 57 / 41 (1.4), 50k 250 / 186 (7), 264k from
// its middle 414 / 372 (16), 1.06M 908 / 787 (32), 2.5M 1303 / 1183 (49), 4M
// 1604 / 1814 (62), 6.26M 1987 / 3263 (78); 3 queries on 264k 842 / 673 (48),
// 20 on 50k 493 / 626 (140), 64 on 20k 417 / 553 (286).
uint32_t region_relaxers(uint64_t regions, uint32_t nq, uint32_t cus) {
    return nq * std::sqrt((double)regions) <= 0.21 * cus ? kMany : kFew;
}

// A query's wavefront has work in about as many regions at once as a few times
// the square root of their number.  With more queries in flight than workgroups can follow
// a region waits in the ring, is expanded from distances that are far from
// final, and again when they fall: 64 queries on road 264k all at once expand
// each vertex 7.4 times, a few at a time 2.2 times, as a lone query does.
// Batch on 264k / 1.06M (24 queries), ms, at kAdmit = 0.15, 0.2, 0.25, 0.3,
// 0.4, all at once: 4.2, 3.5, 3.0, 2.9, 3.8, 5.9 / 7.0, 4.9, 4.6, 4.1, 5.7,
// 11.9.  Graphs of few regions: enough of them for every workgroup.
uint32_t region_admit(uint64_t regions, uint32_t nq, uint32_t grid) {
    constexpr double kAdmit = 0.27, kAdmitTasks = 1.5;
    const double r = regions ? (double)regions : 1.0;
    const uint64_t k = (uint64_t)(grid * std::max(kAdmitTasks / r, kAdmit / std::sqrt(r)));
    return (uint32_t)(k < 1 ? 1 : k < nq ? k : nq);
}

RegionQuery region_query(const RegionGraph &g, uint32_t *dist, uint32_t *inbox, uint32_t *act, uint32_t src) {
    return {g.hdr, g.image, g.verts, g.where, dist, inbox, act, g.n, g.inbox_slots, g.regions, g.width, src};
}

void region_free(RegionGraph *g) {
    for (void *p : {(void *)g->hdr, (void *)g->image, (void *)g->verts, (void *)g->where})
        if (p) (void)hipFree(p);
    *g = RegionGraph{};
}

hipError_t region_build(const RegionPlan &plan, uint32_t n, uint64_t m, const uint32_t *row, const uint32_t *col,
                        const uint32_t *wgt, double mean_weight, hipStream_t s, RegionGraph *g) {
    *g = RegionGraph{};
    const uint32_t nr = (uint32_t)plan.first.size() - 1;
    if (nr > (1u << (32 - kRegionIdBits))) return hipErrorInvalidValue;
    std::vector<RegionHdr> hdr(nr);
    for (uint32_t r = 0; r < nr; ++r) hdr[r] = RegionHdr{plan.first[r], plan.first[r + 1] - plan.first[r], 0, 0, 0, 0, 0, 0};
    uint32_t *tmp = nullptr, *first = nullptr;
    hipError_t e = hipMalloc(&g->hdr, sizeof(RegionHdr) * nr);
    if (e == hipSuccess) e = hipMalloc(&g->verts, sizeof(uint32_t) * (size_t)n);
    if (e == hipSuccess) e = hipMalloc(&g->where, sizeof(uint32_t) * (size_t)n);
    if (e == hipSuccess) e = hipMalloc(&tmp, sizeof(uint32_t) * (size_t)(m ? m : 1));
    if (e == hipSuccess) e = hipMalloc(&first, sizeof(uint32_t) * ((size_t)nr + 1));
    if (e == hipSuccess) e = hipMemcpy(g->hdr, hdr.data(), sizeof(RegionHdr) * nr, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(g->verts, plan.order.data(), sizeof(uint32_t) * (size_t)n, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(first, plan.first.data(), sizeof(uint32_t) * ((size_t)nr + 1), hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(region_where_kernel, dim3(nr), dim3(256), 0, s, g->verts, first, g->where);
        hipLaunchKernelGGL(region_count_kernel, dim3(nr), dim3(256), 0, s, row, col, g->verts, g->where, g->hdr, tmp);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(hdr.data(), g->hdr, sizeof(RegionHdr) * nr, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    uint64_t slots = 0, words = 0, cross = 0;
    if (e == hipSuccess) {
        for (RegionHdr &h : hdr) {
            cross += h.cross;
            if (h.nx > kRegionExits || h.nin > kRegionInbox) e = hipErrorInvalidValue;
            h.inbox = (uint32_t)slots;
            h.image = (uint32_t)words;
            slots += h.nin;
            words += image_words(h);
        }
        g->n = n;
        g->regions = nr;
        g->inbox_slots = (uint32_t)slots;
        // eight mean edge weights
        g->width = (uint32_t)std::min(1e9, std::max(1.0, 8.0 * mean_weight));
        if (words > 0xFFFFFFF0ull || (double)cross > kMaxCross * (double)m) e = hipErrorInvalidValue;
    }
    if (e == hipSuccess) e = hipMalloc(&g->image, sizeof(uint32_t) * words);
    if (e == hipSuccess) e = hipMemcpy(g->hdr, hdr.data(), sizeof(RegionHdr) * nr, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(region_image_kernel, dim3(nr), dim3(256), 0, s, row, col, wgt, g->verts, g->where, g->hdr,
                           tmp, g->image);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (tmp) (void)hipFree(tmp);
    if (first) (void)hipFree(first);
    if (e != hipSuccess) region_free(g);
    return e;
}

hipError_t launch_region_reset(const RegionGraph &g, const RegionLaunch &L, const uint32_t *sources, uint32_t src,
                               hipStream_t s) {
    const uint32_t longest = L.longest > kCtlWords ? L.longest : kCtlWords;
    uint32_t x = (longest + 1023) / 1024;
    if (x > 2048) x = 2048;
    const dim3 grid(x, L.nq < 1024 ? L.nq : 1024);
    const RegionArgs a = make_region_args(g, L);
    if (L.table)
        hipLaunchKernelGGL(region_reset_kernel<true>, grid, dim3(256), 0, s, a, 0u, 0u, nullptr, 0u, nullptr);
    else
        hipLaunchKernelGGL(region_reset_kernel<false>, grid, dim3(256), 0, s, a, g.n, g.inbox_slots, sources, src,
                           g.where);
    return hipGetLastError();
}

hipError_t launch_region_solver(const RegionGraph &g, const RegionLaunch &L, hipStream_t s) {
    const RegionArgs a = make_region_args(g, L);
    if (L.table && L.relaxers == kMany)
        hipLaunchKernelGGL((region_solver_kernel<true, kMany>), dim3(L.grid), dim3(kThreads<kMany>), 0, s, a);
    else if (L.table)
        hipLaunchKernelGGL((region_solver_kernel<true, kFew>), dim3(L.grid), dim3(kThreads<kFew>), 0, s, a);
    else if (L.relaxers == kMany)
        hipLaunchKernelGGL((region_solver_kernel<false, kMany>), dim3(L.grid), dim3(kThreads<kMany>), 0, s, a);
    else
        hipLaunchKernelGGL((region_solver_kernel<false, kFew>), dim3(L.grid), dim3(kThreads<kFew>), 0, s, a);
    return hipGetLastError();
}

}  // namespace mlmq
