// Device-side building blocks of the BFS level kernels for gfx950 (wave64).
//
//  * LdsQueue: frontier-queue allocation.  Waves reserve slots in an LDS
//    buffer with one ballot + one LDS atomic per wave; the workgroup flushes
//    the buffer to the global queue with ONE global atomic per flush
//    (replaces CooperativeTileScan::ScanTileWithEnqueue's per-tile atomic,
//    b40c/util/scan/cooperative_scan.cuh:173-229).  A wave that finds the LDS
//    buffer full spills straight to the global queue (one atomic per wave).
//  * positional_gather: neighbour gathering by edge position over a tile's
//    lists laid end to end, several edges per thread in flight, replacing
//    ExpandByCta / ExpandByWarp / ExpandByScan
//    (b40c/graph/bfs/two_phase/expand_atomic/cta.cuh:215-423, 606-719): one
//    form for every degree.
//  * mark_claim: an agent-scope atomic on the visited bitmask, or on the depth
//    label of a small graph, so each vertex has exactly one discoverer (the
//    reference's best-effort bitmask RMW, contract_expand_atomic/cta.cuh:237-252,
//    lets duplicates through).
//  * HistoryHash: per-workgroup LDS hash of recently seen ids that culls
//    duplicates before they reach the atomic (the reference's warp/history
//    culls, contract_expand_atomic/cta.cuh:363-387,
//    two_phase/contract_atomic/cta.cuh:276-297, sized for wave64 + LDS).
#pragma once

#include <cstddef>

#include "common.hpp"

namespace b40c {

constexpr int BFS_THREADS = 256;
constexpr int BFS_WAVES = BFS_THREADS / kWave;
constexpr int LQ_CAP = 2048;          // LDS queue entries
constexpr int HIST_SIZE = 1024;       // history hash entries

struct BfsArgs {
    const int32_t* offs;
    const int32_t* cols;
    int32_t* depth;
    int32_t* pred;
    uint32_t* visited;       // 1 bit per vertex
    uint32_t* fbm[3];        // frontier bitmaps (direction-optimizing), rotating by level % 3
    int2* heavy;             // grid-tier entries (vertex, first chunk), in chunk order
    int32_t* chunk_map;      // grid-tier chunk -> entry index
    uint32_t heavy_cap;      // capacity of heavy[] (entries)
    uint32_t chunk_cap;      // capacity of chunk_map[]
    int32_t* qk[2];          // frontier queue keys (ping-pong)
    int32_t* qv[2];          // frontier queue values (predecessors), edge frontiers only
    uint32_t qcap[2];        // capacities of qk[i] (elements)
    DevCounters* ctr;
    uint32_t* bar_arrive;    // persistent kernels: grid-barrier arrival word per workgroup
    unsigned long long* bar_words;  // ... of the all-to-all barrier, [2][kAllToAllMax]
    int32_t* regions;        // narrow persistent kernel: frontier pieces, [2][kAllToAllMax][region]
    uint32_t region;         // entries of a piece
    DevCounters* hctr;       // device address of the pinned host mirror of *ctr
    uint32_t* max_depth;     // deepest depth label written
    unsigned long long* wg_stats;  // instrumented: [grid][2] (busy clocks, lifetime clocks)
    int32_t n;
    int32_t words;           // ceil(n / 32)
    int32_t cta_th;          // set by callers that drive the bodies themselves; no body reads them
    int32_t wave_th;
    int32_t grid_th;         // degree >= this: grid tier (split across workgroups)
    int32_t symmetric;       // graph has every reverse edge (bottom-up allowed)
    int32_t do_alpha;
    int32_t do_beta;
    int32_t td_grid;         // direction-optimizing: workgroups of a top-down step
    const uint32_t* iso;     // symmetric graphs: isolated-vertex bitmap, pre-marked visited (else null)
    int32_t dev_base;        // 1: phase = ctr->ph_base + kernel argument (captured, replayed level loops)
    int32_t persistent;      // 1 inside a persistent (single-launch) search
    int32_t coh_in;          // persistent: frontier inputs are read with coh_ld
    int32_t coh_out;         // persistent: outputs (queue, grid-tier entries) are written with coh_st
    long long edges;
    int32_t by_label;        // small graphs: the depth labels mark visited vertices, not the bitmask (mark_claim)
    unsigned long long* spread;  // direction-optimizing (else null): per-level sums of what the steps found (spread_at)
};

// Same-address traffic is serialised at memory: every workgroup's atomic add
// (or plain agent-scope store) to one 256-byte line costs 11.4 ns (33 ns), so
// a counter that all 1,536 workgroups of a launch update costs 17.5 us per
// launch, and 1.1 us when they update 16 counters 256 bytes apart.  Per-level
// sums are therefore kept as SPREAD partial sums per level slot
// (level & 3), one per 256-byte line; the next launch's readers add them up.
// A partial sum is (edges << 32) | vertices (each fits: E < 2^31, V < 2^31).
constexpr int SPREAD = 16;
constexpr int SPREAD_STRIDE = 256 / (int)sizeof(unsigned long long);
constexpr int SPREAD_WORDS = 4 * SPREAD * SPREAD_STRIDE;
__device__ __forceinline__ unsigned long long* spread_at(unsigned long long* spread, int level, int i) {
    return spread + ((level & 3) * SPREAD + i) * SPREAD_STRIDE;
}

// Frontier data that other workgroups of the same persistent launch read
// after a grid barrier (queue entries, grid-tier entries and chunk maps).
// With `coh` the accesses are agent-scope atomic ones, which the GPU keeps
// coherent across XCDs without any cache maintenance, so the persistent
// kernels' barrier only has to wait for each wave's stores to complete
// (grid_sync's light mode) instead of writing back and invalidating its
// XCD's L2 once per workgroup.  Without `coh` (separate launches) they are
// plain accesses.
__device__ __forceinline__ void coh_st(int32_t* p, int32_t v, bool coh) {
    if (coh) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else *p = v;
}
__device__ __forceinline__ int32_t coh_ld(const int32_t* p, bool coh) {
    return coh ? __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : *p;
}
__device__ __forceinline__ void coh_st2(int2* p, int2 v, bool coh) {
    if (coh) {
        const unsigned long long w = (unsigned long long)(uint32_t)v.x | ((unsigned long long)(uint32_t)v.y << 32);
        __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
        *p = v;
    }
}
__device__ __forceinline__ int2 coh_ld2(const int2* p, bool coh) {
    if (!coh) return *p;
    const unsigned long long w = __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p), __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
    return make_int2((int32_t)(uint32_t)w, (int32_t)(uint32_t)(w >> 32));
}

constexpr int HEAVY_CHUNK = 256;     // most grid-tier edges per work item

// ---------------------------------------------------------------------------
// LDS-buffered queue.  VCAP is the capacity of the value array: LQ_CAP for a
// queue that can carry (key, value) pairs, 1 for a keys-only queue.  A
// pair-capable queue also serves keys-only appends (VALS = false), so one
// kernel that alternates key and pair steps uses ONE queue object; no other
// field ever shares storage with `count` or `gbase`.
// ---------------------------------------------------------------------------
template <int VCAP>
struct LdsQueueT {
    int32_t keys[LQ_CAP];
    int32_t vals[VCAP];
    uint32_t count;
    uint32_t gbase;
};
using LdsKeyQueue = LdsQueueT<1>;
using LdsPairQueue = LdsQueueT<LQ_CAP>;
static_assert(offsetof(LdsKeyQueue, count) >= sizeof(int32_t) * (LQ_CAP + 1), "key queue count overlaps its arrays");
static_assert(offsetof(LdsPairQueue, count) >= sizeof(int32_t) * 2 * LQ_CAP, "pair queue count overlaps its arrays");

struct GlobalQueue {
    int32_t* keys;
    int32_t* vals;
    uint32_t* len;
    uint32_t cap;
    uint32_t* overflow;
    bool coh = false;  // entries written with agent-scope stores (persistent launches)
};

// Wave-uniform call: every lane of the wave must be active.
template <bool VALS, int VCAP>
__device__ __forceinline__ void lq_append(LdsQueueT<VCAP>& q, const GlobalQueue& g, bool want, int32_t k,
                                          int32_t v) {
    static_assert(!VALS || VCAP == LQ_CAP, "pair appends need a pair queue");
    const uint64_t m = __ballot(want);
    if (m == 0) return;
    const int lane = lane_id();
    const int cnt = __popcll(m);
    const int leader = __ffsll((unsigned long long)m) - 1;
    uint32_t base = 0;
    if (lane == leader) base = atomicAdd(&q.count, (uint32_t)cnt);
    base = (uint32_t)wave_bcast((int)base, leader);
    const uint32_t pos = base + (uint32_t)lane_prefix(m);
    if (want && pos < (uint32_t)LQ_CAP) {
        q.keys[pos] = k;
        if (VALS) q.vals[pos] = v;
    }
    if (base + (uint32_t)cnt > (uint32_t)LQ_CAP) {
        const uint32_t spill_start = base > (uint32_t)LQ_CAP ? base : (uint32_t)LQ_CAP;
        const uint32_t nspill = base + (uint32_t)cnt - spill_start;
        uint32_t gb = 0;
        if (lane == leader) gb = atomic_add_u32(g.len, nspill);
        gb = (uint32_t)wave_bcast((int)gb, leader);
        if (want && pos >= (uint32_t)LQ_CAP) {
            const uint32_t gp = gb + (pos - spill_start);
            if (gp < g.cap) {
                coh_st(&g.keys[gp], k, g.coh);
                if (VALS) coh_st(&g.vals[gp], v, g.coh);
            } else {
                st_relaxed(g.overflow, 1u);
            }
        }
    }
}

// lq_append of K entries per lane: one ballot per entry, but a single LDS
// atomic for the wave.  Wave-uniform call.
template <bool VALS, int K, int VCAP>
__device__ __forceinline__ void lq_append_batch(LdsQueueT<VCAP>& q, const GlobalQueue& g, const bool (&want)[K],
                                                const int32_t (&k)[K], const int32_t (&v)[K]) {
    static_assert(!VALS || VCAP == LQ_CAP, "pair appends need a pair queue");
    uint64_t m[K];
    uint32_t cnt = 0;
#pragma unroll
    for (int r = 0; r < K; ++r) {
        m[r] = __ballot(want[r]);
        cnt += (uint32_t)__popcll(m[r]);
    }
    if (cnt == 0) return;
    uint32_t base = 0;
    if (lane_id() == 0) base = atomicAdd(&q.count, cnt);
    base = (uint32_t)wave_bcast((int)base, 0);
    // Entries past the LDS buffer go straight to the global queue.
    const bool spills = base + cnt > (uint32_t)LQ_CAP;
    const uint32_t spill_start = base > (uint32_t)LQ_CAP ? base : (uint32_t)LQ_CAP;
    uint32_t gb = 0;
    if (spills) {
        if (lane_id() == 0) gb = atomic_add_u32(g.len, base + cnt - spill_start);
        gb = (uint32_t)wave_bcast((int)gb, 0);
    }
    uint32_t at = base;
#pragma unroll
    for (int r = 0; r < K; ++r) {
        const uint32_t pos = at + (uint32_t)lane_prefix(m[r]);
        at += (uint32_t)__popcll(m[r]);
        if (!want[r]) continue;
        if (pos < (uint32_t)LQ_CAP) {
            q.keys[pos] = k[r];
            if (VALS) q.vals[pos] = v[r];
        } else {
            const uint32_t gp = gb + (pos - spill_start);
            if (gp < g.cap) {
                coh_st(&g.keys[gp], k[r], g.coh);
                if (VALS) coh_st(&g.vals[gp], v[r], g.coh);
            } else {
                st_relaxed(g.overflow, 1u);
            }
        }
    }
}

// Workgroup-uniform call.  Flushes when the buffer holds at least `min_fill`
// entries (min_fill = 1: flush whatever is there).
template <bool VALS, int VCAP>
__device__ __forceinline__ void lq_flush(LdsQueueT<VCAP>& q, const GlobalQueue& g, uint32_t min_fill) {
    static_assert(!VALS || VCAP == LQ_CAP, "pair flushes need a pair queue");
    __syncthreads();
    uint32_t cnt = q.count;
    __syncthreads();
    if (cnt > (uint32_t)LQ_CAP) cnt = LQ_CAP;
    if (cnt < min_fill || cnt == 0) return;
    if (threadIdx.x == 0) q.gbase = atomic_add_u32(g.len, cnt);
    __syncthreads();
    const uint32_t gb = q.gbase;
    for (uint32_t j = threadIdx.x; j < cnt; j += BFS_THREADS) {
        const uint32_t gp = gb + j;
        if (gp < g.cap) {
            coh_st(&g.keys[gp], q.keys[j], g.coh);
            if (VALS) coh_st(&g.vals[gp], q.vals[j], g.coh);
        }
    }
    if (threadIdx.x == 0 && gb + cnt > g.cap) st_relaxed(g.overflow, 1u);
    __syncthreads();
    if (threadIdx.x == 0) q.count = 0;
    __syncthreads();
}

// ---------------------------------------------------------------------------
// Culling.
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool visited_test(const uint32_t* visited, int32_t v) {
    return (visited[v >> 5] >> (v & 31)) & 1u;
}

// Exactly one caller per vertex returns true.
__device__ __forceinline__ bool claim_exact(uint32_t* visited, int32_t v) {
    uint32_t* w = visited + (v >> 5);
    const uint32_t bit = 1u << (v & 31);
    if (*w & bit) return false;
    return (atomic_or_u32(w, bit) & bit) == 0;
}

// Marks of visited vertices.  Normally the bitmask: 32 times smaller than the
// labels, so probes stay in L2.  But atomics on one 64-byte line are
// serialised (11.4 ns each), a line of the bitmask holds 512 vertices, and a
// graph of 4,096 vertices has only eight such lines: its widest top-down level
// spent 23 us in claims.  Small graphs (by_label) therefore claim on the depth
// label itself, 16 vertices to a line: an unsigned minimum, -1 being the
// largest, which also labels the vertex.
__device__ __forceinline__ uint32_t mark_load(const BfsArgs& a, int32_t v) {
    return a.by_label ? (uint32_t)a.depth[v] : a.visited[v >> 5];
}
__device__ __forceinline__ bool mark_seen(const BfsArgs& a, int32_t v, uint32_t mark) {
    return a.by_label ? mark != 0xFFFFFFFFu : ((mark >> (v & 31)) & 1u) != 0u;
}
// Returns the mark before the claim (mark_seen tells whether it was taken);
// with by_label the winner's label is then already written.
__device__ __forceinline__ uint32_t mark_claim(const BfsArgs& a, int32_t v, int32_t depth) {
    if (a.by_label)
        return __hip_atomic_fetch_min(reinterpret_cast<uint32_t*>(&a.depth[v]), (uint32_t)depth, __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
    return atomic_or_u32(&a.visited[v >> 5], 1u << (v & 31));
}

struct HistoryHash {
    int32_t slot[HIST_SIZE];
};

__device__ __forceinline__ void history_init(HistoryHash& h) {
    for (int i = threadIdx.x; i < HIST_SIZE; i += BFS_THREADS) h.slot[i] = -1;
}

// True when `v` was seen recently by this workgroup (a duplicate to drop).
// Racing writers may both miss: the hash only thins duplicates, the exact
// claim decides.
__device__ __forceinline__ bool history_seen(HistoryHash& h, int32_t v) {
    const uint32_t idx = ((uint32_t)v * 2654435761u) >> (32 - 10);
    if (h.slot[idx] == v) return true;
    h.slot[idx] = v;
    return false;
}

// ---------------------------------------------------------------------------
// Positional gather: the lists of one tile (one per thread) laid end to end,
// each thread taking K positions per step, BFS_THREADS apart.  A position is
// mapped back to its list by binary search over the tile's ranks in LDS, so
// work per step follows edges whatever the degrees, and the K edges' loads,
// probes and claims (sink.step) are in flight together: a gather step is a
// chain of dependent accesses and latency, not bandwidth, bounds it.
// ---------------------------------------------------------------------------
struct ListSmem {
    int32_t rank[BFS_THREADS];  // first position of each list
    int32_t base[BFS_THREADS];  // column index of position p of the list is base + p
    int32_t src[BFS_THREADS];
    int s_wave[BFS_WAVES];
    uint32_t reserved;  // sinks that write in place: the tile's first output position
};

template <int K, typename Sink>
__device__ __forceinline__ void gather_step(const int32_t* __restrict__ cols, const ListSmem& g, uint32_t p0,
                                            uint32_t total, Sink& sink) {
    int lo[K];
    int32_t v[K], src[K];
    bool valid[K];
#pragma unroll
    for (int r = 0; r < K; ++r) {
        lo[r] = 0;
        valid[r] = p0 + (uint32_t)(r * BFS_THREADS) + threadIdx.x < total;
    }
    // Last list with rank <= p; the K searches run side by side.
#pragma unroll
    for (int h = BFS_THREADS / 2; h >= 1; h >>= 1) {
#pragma unroll
        for (int r = 0; r < K; ++r) {
            const int32_t p = (int32_t)(p0 + (uint32_t)(r * BFS_THREADS) + threadIdx.x);
            if (g.rank[lo[r] + h] <= p) lo[r] += h;
        }
    }
#pragma unroll
    for (int r = 0; r < K; ++r) {
        const int32_t p = (int32_t)(p0 + (uint32_t)(r * BFS_THREADS) + threadIdx.x);
        src[r] = g.src[lo[r]];
        v[r] = valid[r] ? cols[g.base[lo[r]] + p] : 0;
    }
    sink.template step<K>(p0, valid, v, src);
}

// Workgroup-uniform call.  sink.reserve(total, g) runs in thread 0 when the
// tile has edges, sink.step wave-uniformly, sink.step_end() workgroup-
// uniformly after every step.  With `parts` > 1 the
// same tile is gathered by that many workgroups, each taking every parts-th
// step (this one the part-th).
constexpr int GATHER_K = 8;
template <int KMAX, typename Sink>
__device__ __forceinline__ void positional_gather(const int32_t* __restrict__ cols, int32_t src, int32_t start,
                                                  int32_t deg, ListSmem& g, Sink& sink, uint32_t part = 0,
                                                  uint32_t parts = 1) {
    constexpr uint32_t STEP = (uint32_t)(KMAX * BFS_THREADS);
    int sum;
    const int rank = wg_exclusive_scan<BFS_THREADS>(deg, sum, g.s_wave);
    const uint32_t total = (uint32_t)sum;
    if ((uint64_t)part * STEP >= total) return;
    g.rank[threadIdx.x] = rank;
    g.base[threadIdx.x] = start - rank;
    g.src[threadIdx.x] = src;
    if (threadIdx.x == 0) sink.reserve(total, g);
    __syncthreads();
    for (uint64_t p0 = (uint64_t)part * STEP; p0 < total; p0 += (uint64_t)parts * STEP) {
        if (total - (uint32_t)p0 <= 2u * BFS_THREADS)
            gather_step<2>(cols, g, (uint32_t)p0, total, sink);
        else
            gather_step<KMAX>(cols, g, (uint32_t)p0, total, sink);
        sink.step_end();
    }
    __syncthreads();
}

// ---------------------------------------------------------------------------
// Per-workgroup clock instrumentation (KernelRuntimeStats,
// b40c/util/kernel_runtime_stats.cuh:77-113): busy clocks and lifetime.
// ---------------------------------------------------------------------------
__device__ __forceinline__ unsigned long long wg_clock() { return wall_clock64(); }

}  // namespace b40c
