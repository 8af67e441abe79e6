// Device side of the single-GPU BFS for gfx950: the level step bodies and
// every kernel's body as a __device__ function that takes its LDS block by
// reference.  bfs.hip wraps each body in a __global__ kernel that declares
// the LDS block; keeping the bodies here lets a CPU replay build (tests/
// cpu_replay) run the very same code with bounds-checked buffers.
//
// Reference counterparts (b40c):
//   level kernels             b40c/graph/bfs/{expand_contract_atomic,
//                             contract_expand_atomic, two_phase}/kernel.cuh
//   persistent kernels        contract_expand_atomic/kernel.cuh:281-554,
//                             two_phase/kernel.cuh:60-313
//
// Queue protocol: a "phase" is one kernel step that reads one frontier queue
// and writes the next.  Phase ph reads buffer ph&1 with its length in
// counter slot ph&3, appends to buffer (ph+1)&1 / slot (ph+1)&3 and clears
// slot (ph+2)&3.  Expand-contract and contract-expand use one phase per BFS
// level, two-phase uses two (contract, expand) or three (filter, contract,
// expand).  Depth labels are carried separately from the phase index.
//
// Grid tier: an expanding phase defers vertices whose degree reaches
// grid_th to a list (length slot ph&1); the k_heavy launch that follows the
// phase splits those adjacency lists into HEAVY_CHUNK-edge pieces spread over
// every workgroup, so one hub no longer serializes a level on one workgroup.
#pragma once

#include <climits>

#include "bfs_device.hpp"

namespace b40c {

// ===========================================================================
// Level bodies (device).
// ===========================================================================

constexpr int CONTRACT_K = 4;  // pairs per thread of a wide contraction

// LDS of a level step.  Keys-only steps (two-phase contraction) and pair
// steps (contract-expand, two-phase filter) append to the same pair-capable
// queue, so a persistent kernel that alternates them keeps one valid count.
struct PairLevelShared {
    LdsPairQueue q;
    ListSmem l;
    HistoryHash hist;
    unsigned long long red[BFS_WAVES];
    uint32_t ctl;  // persistent kernels: loop control, read by one thread per workgroup
};

// Contract-expand steps also hold the survivors of one wide tile.
struct LevelShared : PairLevelShared {
    int32_t kept_v[CONTRACT_K * BFS_THREADS];
    int32_t kept_start[CONTRACT_K * BFS_THREADS];
    int32_t kept_deg[CONTRACT_K * BFS_THREADS];
};

// Expand-contract and two-phase expand steps only ever append keys, if
// anything, and keep no history: less than half the LDS, so more workgroups
// stay resident.
struct TdLevelShared {
    LdsKeyQueue q;
    ListSmem l;
    unsigned long long red[BFS_WAVES];
    uint32_t ctl;
};

__device__ __forceinline__ void shared_init(PairLevelShared& s) {
    if (threadIdx.x == 0) s.q.count = 0;
    history_init(s.hist);
    __syncthreads();
}
__device__ __forceinline__ void shared_init(TdLevelShared& s) {
    if (threadIdx.x == 0) s.q.count = 0;
    __syncthreads();
}

// Frontier entries are validated before they are used as addresses: an id
// outside [0, n) is dropped and flagged, so a corrupt queue surfaces as an
// error status instead of an out-of-bounds access.
__device__ __forceinline__ bool valid_vertex(const BfsArgs& a, int32_t v) {
    if ((uint32_t)v < (uint32_t)a.n) return true;
    st_relaxed(&a.ctr->corrupt, 1u);
    return false;
}

__device__ __forceinline__ uint32_t phase_input_len(const BfsArgs& a, int ph) {
    uint32_t n = ld_relaxed(&a.ctr->qlen[ph & 3]);
    if (n > a.qcap[ph & 1]) n = 0;  // an overflowed queue counts as empty
    return n;
}

// A phase body's n_in argument: the input frontier's length when the caller
// already has it (the persistent kernels get it with the grid barrier), or
// this value to read it from the counters.
constexpr uint32_t kLenFromCounters = 0xFFFFFFFFu;
__device__ __forceinline__ uint32_t input_len(const BfsArgs& a, int ph, uint32_t n_in) {
    return n_in == kLenFromCounters ? phase_input_len(a, ph) : n_in;
}

// `frontier_depth` >= 0: the phase's input vertices carry that label, so a
// nonempty input makes it the deepest one before this phase (told by workgroup
// 0 alone: updates by every workgroup would be serialised at one address).  With
// `raised` other workgroups of the launch may have raised it to the phase's own
// label already (raise_max_depth), so it takes a maximum; elsewhere a store, which
// is 0.15 us sooner done (a launch per level of a 2,000-vertex path: 6.4 and 6.55 us).
__device__ __forceinline__ void phase_begin(const BfsArgs& a, int ph, uint32_t n_in, int32_t frontier_depth = -1,
                                            bool raised = false) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (frontier_depth >= 0 && n_in) {
            if (raised)
                atomic_max_u32(a.max_depth, (uint32_t)frontier_depth);
            else
                st_relaxed(a.max_depth, (uint32_t)frontier_depth);
        }
        st_relaxed(&a.ctr->qlen[(ph + 2) & 3], 0u);
        __hip_atomic_store(&a.ctr->heavy_alloc[(ph + 1) & 1], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (n_in) atomic_add_u64(&a.ctr->queued, n_in);
    }
}

// How a gathering phase deals its input entries out to the `wgs` workgroups
// taking part: in turns of 2^turn consecutive entries.  Neighbouring entries
// thus go to different workgroups: discovery order puts an RMAT graph's hubs
// (low ids, first in every sorted list) next to each other, and with
// contiguous tiles the workgroup that got them was the level (RMAT-20's widest
// level: 489 us for the slowest of 512 workgroups, 181 us on average).
// Longer turns read the queue in fewer lines: single entries while a
// workgroup gets fewer than 16 of them, 16 bytes (a line of an edge
// frontier, which has more entries and culls most) up to a full tile (with
// single entries there, a 100^3 lattice search is 5 % slower), then a line
// of a vertex frontier; an edge frontier that wide is read in whole tiles
// (with single entries RMAT-22 contract-expand took 5.9 instead of 4.4 ms),
// since its culled tiles differ little.
struct Deal {
    uint32_t wgs, turn;
    __device__ __forceinline__ uint32_t entry(uint32_t base, uint32_t wg) const {
        const uint32_t t = threadIdx.x;
        return base + ((((t >> turn) * wgs + wg) << turn) | (t & ((1u << turn) - 1u)));
    }
};
__device__ __forceinline__ Deal deal_out(uint32_t n_in, uint32_t wgs, bool edges) {
    const uint64_t w = wgs;
    const uint32_t mid = edges ? 4u : 2u, wide = edges ? 8u : 4u;
    return Deal{wgs, n_in < 16 * w ? 0u : n_in < BFS_THREADS * w ? mid : wide};
}

// Workgroups taking part.  Level launches use no more than there are full
// tiles; a persistent launch uses all of its grid, so that on the narrow
// levels of a high-diameter graph every workgroup gathers its few lists in one
// step.  Level launches run four times as many workgroups, and there the extra
// workgroups' same-address queue atomics cost more than the steps saved
// (200^3 lattice: 25 instead of 17 us per level).
__device__ __forceinline__ uint32_t sharing_wgs(const BfsArgs& a, uint32_t n_in, uint32_t nblocks) {
    if (a.persistent) return nblocks;
    return min(nblocks, (n_in + BFS_THREADS - 1) / BFS_THREADS);
}

__device__ __forceinline__ GlobalQueue out_queue(const BfsArgs& a, int ph) {
    GlobalQueue q;
    q.keys = a.qk[(ph + 1) & 1];
    q.vals = a.qv[(ph + 1) & 1];
    q.len = &a.ctr->qlen[(ph + 1) & 3];
    q.cap = a.qcap[(ph + 1) & 1];
    q.overflow = &a.ctr->overflow;
    q.coh = a.coh_out != 0;
    return q;
}

// Workgroup sum of a per-thread u64, added once to *dst.
__device__ __forceinline__ void wg_add_u64(unsigned long long v, unsigned long long* dst, unsigned long long* red) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, kWave);
    __syncthreads();
    if (lane_id() == 0) red[threadIdx.x / kWave] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long t = 0;
        for (int w = 0; w < BFS_WAVES; ++w) t += red[w];
        if (t) atomic_add_u64(dst, t);
    }
}

// Grid-tier deferral (wave-uniform): lanes whose vertex has degree >= grid_th
// hand its adjacency list to the grid tier of phase ph and drop their own
// expansion.  One 64-bit atomic per wave allocates, in the same order, entry
// slots (high word) and HEAVY_CHUNK-edge chunk ranges (low word); each lane
// records (vertex, first chunk) and points its chunks at its entry, so the
// grid-tier kernel maps any chunk to its vertex with one load.
__device__ __forceinline__ void defer_heavy(const BfsArgs& a, int ph, int32_t v, int32_t& deg, int32_t grid_th) {
    const bool heavy = deg >= grid_th;
    const uint64_t m = __ballot(heavy);
    if (m == 0) return;
    const int lane = lane_id();
    const int leader = __ffsll((unsigned long long)m) - 1;
    const uint32_t nch = heavy ? (uint32_t)((deg + HEAVY_CHUNK - 1) / HEAVY_CHUNK) : 0u;
    const uint32_t ch_incl = (uint32_t)wave_inclusive_scan((int)nch);
    const uint32_t ch_total = (uint32_t)__shfl((int)ch_incl, kWave - 1, kWave);
    unsigned long long base = 0;
    if (lane == leader)
        base = __hip_atomic_fetch_add(&a.ctr->heavy_alloc[ph & 1],
                                      ((unsigned long long)__popcll(m) << 32) | (unsigned long long)ch_total,
                                      __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t base_lo = (uint32_t)wave_bcast((int)(uint32_t)base, leader);
    const uint32_t base_hi = (uint32_t)wave_bcast((int)(uint32_t)(base >> 32), leader);
    if (heavy) {
        const uint32_t entry = base_hi + (uint32_t)lane_prefix(m);
        const uint32_t c0 = base_lo + ch_incl - nch;
        if (entry < a.heavy_cap && c0 + nch <= a.chunk_cap) {
            const bool coh = a.coh_out != 0;
            coh_st2(&a.heavy[entry], make_int2(v, (int)c0), coh);
            for (uint32_t c = 0; c < nch; ++c) coh_st(&a.chunk_map[c0 + c], (int32_t)entry, coh);
        } else {
            st_relaxed(&a.ctr->overflow, 1u);
        }
        deg = 0;
    }
}

// Top-down discovery: exact claims and labels of the K edges of a gather
// step, each access for all of them together; `won` marks the edges that
// discovered their neighbour.
template <int K>
__device__ __forceinline__ void td_claim(const BfsArgs& a, const bool (&valid)[K], const int32_t (&v)[K],
                                         const int32_t (&src)[K], int32_t depth_next, bool (&won)[K]) {
    uint32_t seen[K];
#pragma unroll
    for (int r = 0; r < K; ++r) {
        seen[r] = 0u;
        if (valid[r]) seen[r] = mark_load(a, v[r]);
        won[r] = valid[r] && !mark_seen(a, v[r], seen[r]);
    }
#pragma unroll
    for (int r = 0; r < K; ++r)
        if (won[r]) seen[r] = mark_claim(a, v[r], depth_next);
#pragma unroll
    for (int r = 0; r < K; ++r) {
        won[r] = won[r] && !mark_seen(a, v[r], seen[r]);
        if (won[r]) {
            if (!a.by_label) a.depth[v[r]] = depth_next;
            a.pred[v[r]] = src[r];
        }
    }
}

// Top-down sink: optional frontier bitmap bit and degree accounting for the
// direction switch, then the LDS queue.
template <int VCAP>
struct TdSink {
    const BfsArgs& a;
    LdsQueueT<VCAP>& q;
    const GlobalQueue& out;
    uint32_t* next_bm;
    int32_t depth_next;
    bool count_edges;
    unsigned long long eacc;
    __device__ __forceinline__ void reserve(uint32_t, ListSmem&) {}
    template <int K>
    __device__ __forceinline__ void step(uint32_t, const bool (&valid)[K], const int32_t (&v)[K],
                                         const int32_t (&src)[K]) {
        bool won[K];
        td_claim(a, valid, v, src, depth_next, won);
        if (next_bm) {
#pragma unroll
            for (int r = 0; r < K; ++r)
                if (won[r]) atomic_or_u32(&next_bm[v[r] >> 5], 1u << (v[r] & 31));
        }
        if (count_edges) {
#pragma unroll
            for (int r = 0; r < K; ++r)
                if (won[r]) eacc += (unsigned long long)(a.offs[v[r] + 1] - a.offs[v[r]]);
        }
        lq_append_batch<false>(q, out, won, v, v);
    }
    __device__ __forceinline__ void step_end() { lq_flush<false>(q, out, LQ_CAP / 2); }
};

// Every edge as a (neighbour, source) pair through the LDS queue.
struct PairSink {
    LdsPairQueue& q;
    const GlobalQueue& out;
    __device__ __forceinline__ void reserve(uint32_t, ListSmem&) {}
    template <int K>
    __device__ __forceinline__ void step(uint32_t, const bool (&valid)[K], const int32_t (&nbr)[K],
                                         const int32_t (&src)[K]) {
        lq_append_batch<true>(q, out, valid, nbr, src);
    }
    __device__ __forceinline__ void step_end() { lq_flush<true>(q, out, LQ_CAP / 2); }
};

// Every edge as a pair, written in place: all of a tile's edges are output,
// so one atomic reserves them and position p goes to slot reserved + p.
struct InPlaceSink {
    const GlobalQueue& out;
    ListSmem& g;
    __device__ __forceinline__ void reserve(uint32_t total, ListSmem& l) {
        const uint32_t base = atomic_add_u32(out.len, total);
        if ((uint64_t)base + total > out.cap) st_relaxed(out.overflow, 1u);
        l.reserved = base;
    }
    template <int K>
    __device__ __forceinline__ void step(uint32_t p0, const bool (&valid)[K], const int32_t (&nbr)[K],
                                         const int32_t (&src)[K]) {
        const uint64_t base = (uint64_t)g.reserved + p0 + threadIdx.x;
#pragma unroll
        for (int r = 0; r < K; ++r) {
            const uint64_t pos = base + (uint32_t)(r * BFS_THREADS);
            if (valid[r] && pos < out.cap) {
                coh_st(&out.keys[pos], nbr[r], out.coh);
                coh_st(&out.vals[pos], src[r], out.coh);
            }
        }
    }
    __device__ __forceinline__ void step_end() {}
};

// Workgroup sum of a per-thread degree count, added to the level's partial
// sums of the degrees of discovered vertices.
__device__ __forceinline__ void add_level_edges(const BfsArgs& a, int ph, unsigned long long edges,
                                                unsigned long long* red) {
    wg_add_u64(edges << 32, spread_at(a.spread, ph + 1, blockIdx.x % SPREAD), red);
}

template <int VCAP>
__device__ __forceinline__ void td_finish(const BfsArgs& a, int ph, TdSink<VCAP>& sink, unsigned long long* red) {
    lq_flush<false>(sink.q, sink.out, 1);
    if (sink.count_edges) add_level_edges(a, ph, sink.eacc, red);
}

// Expand-contract (vertex frontier -> vertex frontier).  Neighbours are
// culled and labelled at discovery (depth = depth_next), as in
// expand_contract_atomic/cta.cuh:212-214, and compacted into the next vertex
// frontier.
// `nblocks` workgroups (the first ones of the launch) share the frontier;
// lists of at least `grid_th` edges go to the grid tier (k_heavy), or, with
// `split`, no list does: while the frontier has fewer tiles than half the
// workgroups, several workgroups read the same tile and share its edges.
// That replaces the grid tier's launch (4 us even when it finds nothing) on
// the narrow levels where a hub would keep one workgroup busy.
template <int KMAX, int VCAP>
__device__ void td_phase(const BfsArgs& a, int ph, int32_t depth_next, uint32_t* next_bm, bool count_edges,
                         LdsQueueT<VCAP>& q, ListSmem& g, unsigned long long* red, uint32_t nblocks,
                         int32_t grid_th, uint32_t n_in_arg = kLenFromCounters, bool split = false) {
    const uint32_t n_in = input_len(a, ph, n_in_arg);
    phase_begin(a, ph, n_in, a.persistent ? -1 : depth_next - 1);
    const int32_t* qin = a.qk[ph & 1];
    const GlobalQueue out = out_queue(a, ph);
    TdSink<VCAP> sink{a, q, out, next_bm, depth_next, count_edges, 0ull};
    uint32_t wgs = sharing_wgs(a, n_in, nblocks), wg = blockIdx.x, part = 0, parts = 1;
    if (split && wgs && nblocks >= 2 * wgs) {
        // The remainder of the division takes no part.
        parts = nblocks / wgs;
        part = blockIdx.x / wgs;
        wg = part < parts ? blockIdx.x % wgs : wgs;
    }
    const Deal deal = deal_out(n_in, wgs, false);
    for (uint32_t base = 0; wg < wgs && base < n_in; base += wgs * BFS_THREADS) {
        const uint32_t i = deal.entry(base, wg);
        int32_t u = -1, start = 0, deg = 0;
        if (i < n_in) {
            u = coh_ld(&qin[i], a.coh_in != 0);
            if (valid_vertex(a, u)) {
                start = a.offs[u];
                deg = a.offs[u + 1] - start;
            }
        }
        if (!split) defer_heavy(a, ph, u, deg, grid_th);
        positional_gather<KMAX>(a.cols, u, start, deg, g, sink, part, parts);
    }
    td_finish(a, ph, sink, red);
}

// The same step over a frontier held as a bitmap (a bottom-up step leaves no
// vertex queue): each workgroup takes 256-word pieces of the bitmap, lists
// their vertices in LDS and gathers them 256 at a time.
constexpr int BM_LIST = 1024;
template <int KMAX, int VCAP>
__device__ void td_bitmap_phase(const BfsArgs& a, int ph, int32_t depth_next, const uint32_t* cur, uint32_t* next_bm,
                                LdsQueueT<VCAP>& q, ListSmem& g, int32_t* list, unsigned long long* red,
                                uint32_t nblocks, int32_t grid_th, uint32_t n_in) {
    phase_begin(a, ph, n_in, depth_next - 1);
    const GlobalQueue out = out_queue(a, ph);
    TdSink<VCAP> sink{a, q, out, next_bm, depth_next, true, 0ull};
    for (int32_t w0 = (int32_t)blockIdx.x * BFS_THREADS; w0 < a.words; w0 += (int32_t)nblocks * BFS_THREADS) {
        const int32_t w = w0 + (int32_t)threadIdx.x;
        uint32_t bits = w < a.words ? cur[w] : 0u;
        int total;
        int at = wg_exclusive_scan<BFS_THREADS>(__popcll((unsigned long long)bits), total, g.s_wave);
        for (int l0 = 0; l0 < total; l0 += BM_LIST) {
            while (bits && at < l0 + BM_LIST) {
                list[at - l0] = w * 32 + (__ffsll((unsigned long long)bits) - 1);
                bits &= bits - 1;
                ++at;
            }
            __syncthreads();
            const int cnt = min(BM_LIST, total - l0);
            for (int i0 = 0; i0 < cnt; i0 += BFS_THREADS) {
                const int i = i0 + (int)threadIdx.x;
                int32_t u = -1, start = 0, deg = 0;
                if (i < cnt) {
                    u = list[i];
                    if (valid_vertex(a, u)) {
                        start = a.offs[u];
                        deg = a.offs[u + 1] - start;
                    }
                }
                defer_heavy(a, ph, u, deg, grid_th);
                positional_gather<KMAX>(a.cols, u, start, deg, g, sink);
            }
            __syncthreads();
        }
    }
    td_finish(a, ph, sink, red);
}

// Contract-expand (edge frontier -> edge frontier).  Incoming (vertex,
// predecessor) pairs are culled (bitmask, history hash, exact claim) and
// labelled at contraction (depth = depth_here), then the survivors'
// neighbour lists are expanded into the outgoing edge frontier
// (contract_expand_atomic/cta.cuh:573-709).
//
// Wide frontiers are contracted CONTRACT_K pairs per thread, each access of
// the chain (pair, mark, claim, row offsets) for all of them together; the
// few survivors are compacted in LDS and their lists gathered 256 at a time.

// Contracts K pairs per thread; returns what each lane keeps.
template <int K>
__device__ __forceinline__ void contract_pairs(const BfsArgs& a, int ph, const uint32_t (&i)[K], uint32_t n_in,
                                               int32_t depth_here, HistoryHash& hist, bool (&keep)[K],
                                               int32_t (&v)[K]) {
    const int32_t* qk = a.qk[ph & 1];
    const int32_t* qv = a.qv[ph & 1];
    int32_t p[K];
    uint32_t mark[K];
#pragma unroll
    for (int r = 0; r < K; ++r) {
        v[r] = i[r] < n_in ? coh_ld(&qk[i[r]], a.coh_in != 0) : -1;
        p[r] = i[r] < n_in ? coh_ld(&qv[i[r]], a.coh_in != 0) : 0;
    }
#pragma unroll
    for (int r = 0; r < K; ++r) {
        keep[r] = i[r] < n_in && valid_vertex(a, v[r]);
        mark[r] = keep[r] ? mark_load(a, v[r]) : 0u;
    }
#pragma unroll
    for (int r = 0; r < K; ++r) keep[r] = keep[r] && !mark_seen(a, v[r], mark[r]) && !history_seen(hist, v[r]);
#pragma unroll
    for (int r = 0; r < K; ++r)
        if (keep[r]) mark[r] = mark_claim(a, v[r], depth_here);
#pragma unroll
    for (int r = 0; r < K; ++r) {
        keep[r] = keep[r] && !mark_seen(a, v[r], mark[r]);
        if (keep[r]) {
            if (!a.by_label) a.depth[v[r]] = depth_here;
            a.pred[v[r]] = p[r];
        }
    }
}

// The deepest label: vertices that a contraction labels are the next phases'
// frontier, or their edges are, so a later phase sees that there were some.
// Only those without out-edges leave nothing behind (`sinks`).
__device__ __forceinline__ void raise_max_depth(const BfsArgs& a, bool sinks, int32_t depth) {
    if (__syncthreads_or(sinks) && threadIdx.x == 0) atomic_max_u32(a.max_depth, (uint32_t)depth);
}

template <bool PERSISTENT>
__device__ void ce_phase(const BfsArgs& a, int ph, int32_t depth_here, LevelShared& s,
                         uint32_t n_in_arg = kLenFromCounters) {
    const uint32_t n_in = input_len(a, ph, n_in_arg);
    // (Symmetric graphs, which have a.iso, have no vertex without out-edges to raise
    // it.  The persistent loop keeps the depth itself; its form of this call, without
    // the test of a.iso and with that of a.persistent, is the one whose code is
    // fastest: 46^3 lattice 1,210 us, without either 1,252.)
    if constexpr (PERSISTENT)
        phase_begin(a, ph, n_in, a.persistent ? -1 : depth_here - 1);
    else
        phase_begin(a, ph, n_in, depth_here - 1, a.iso == nullptr);
    const GlobalQueue out = out_queue(a, ph);
    PairSink sink{s.q, out};
    bool sinks = false;
    const uint32_t wgs = sharing_wgs(a, n_in, gridDim.x);
    const Deal deal = deal_out(n_in, wgs, true);
    uint32_t base = 0;
    for (; blockIdx.x < wgs && n_in - base >= wgs * (uint32_t)(CONTRACT_K * BFS_THREADS);
         base += wgs * (uint32_t)(CONTRACT_K * BFS_THREADS)) {
        uint32_t i[CONTRACT_K];
        bool keep[CONTRACT_K];
        int32_t v[CONTRACT_K], start[CONTRACT_K], deg[CONTRACT_K];
#pragma unroll
        for (int r = 0; r < CONTRACT_K; ++r) i[r] = deal.entry(base + (uint32_t)r * wgs * BFS_THREADS, blockIdx.x);
        contract_pairs<CONTRACT_K>(a, ph, i, n_in, depth_here, s.hist, keep, v);
        int cnt = 0;
#pragma unroll
        for (int r = 0; r < CONTRACT_K; ++r) {
            start[r] = deg[r] = 0;
            if (keep[r]) {
                start[r] = a.offs[v[r]];
                deg[r] = a.offs[v[r] + 1];
            }
        }
#pragma unroll
        for (int r = 0; r < CONTRACT_K; ++r) {
            deg[r] -= start[r];
            sinks |= keep[r] && deg[r] == 0;
            cnt += deg[r] > 0 ? 1 : 0;
        }
        int kept;
        int at = wg_exclusive_scan<BFS_THREADS>(cnt, kept, s.l.s_wave);
#pragma unroll
        for (int r = 0; r < CONTRACT_K; ++r)
            if (deg[r] > 0) {
                s.kept_v[at] = v[r];
                s.kept_start[at] = start[r];
                s.kept_deg[at] = deg[r];
                ++at;
            }
        __syncthreads();
        for (int k0 = 0; k0 < kept; k0 += BFS_THREADS) {
            const int k = k0 + (int)threadIdx.x;
            int32_t u = -1, us = 0, ud = 0;
            if (k < kept) {
                u = s.kept_v[k];
                us = s.kept_start[k];
                ud = s.kept_deg[k];
            }
            defer_heavy(a, ph, u, ud, a.grid_th);
            positional_gather<GATHER_K>(a.cols, u, us, ud, s.l, sink);
        }
        __syncthreads();
    }
    for (; blockIdx.x < wgs && base < n_in; base += wgs * BFS_THREADS) {
        const uint32_t i[1] = {deal.entry(base, blockIdx.x)};
        bool keep[1];
        int32_t v[1], start = 0, deg = 0;
        contract_pairs<1>(a, ph, i, n_in, depth_here, s.hist, keep, v);
        if (keep[0]) {
            start = a.offs[v[0]];
            deg = a.offs[v[0] + 1] - start;
            sinks |= deg == 0;
        }
        defer_heavy(a, ph, v[0], deg, a.grid_th);
        positional_gather<GATHER_K>(a.cols, v[0], start, deg, s.l, sink);
    }
    lq_flush<true>(s.q, out, 1);
    raise_max_depth(a, sinks, depth_here);
}

// Two-phase contract (edge frontier -> vertex frontier + labels),
// two_phase/contract_atomic/cta.cuh:494-572.
__device__ void tp_contract_phase(const BfsArgs& a, int ph, int32_t depth_here, PairLevelShared& s,
                                  uint32_t n_in_arg = kLenFromCounters) {
    const uint32_t n_in = input_len(a, ph, n_in_arg);
    phase_begin(a, ph, n_in);
    const GlobalQueue out = out_queue(a, ph);
    for (uint64_t base = (uint64_t)blockIdx.x * BFS_THREADS; base < n_in;
         base += (uint64_t)gridDim.x * BFS_THREADS * CONTRACT_K) {
        uint32_t i[CONTRACT_K];
        bool keep[CONTRACT_K];
        int32_t v[CONTRACT_K];
#pragma unroll
        for (int r = 0; r < CONTRACT_K; ++r)
            i[r] = (uint32_t)min<uint64_t>(base + (uint64_t)r * gridDim.x * BFS_THREADS + threadIdx.x, n_in);
        contract_pairs<CONTRACT_K>(a, ph, i, n_in, depth_here, s.hist, keep, v);
        lq_append_batch<false>(s.q, out, keep, v, v);
        lq_flush<false>(s.q, out, LQ_CAP / 2);
    }
    lq_flush<false>(s.q, out, 1);
}

// A workgroup takes at least this many vertices: each reserves its output at one
// address (11.4 ns apiece), which on narrow levels, dealt out to all workgroups
// of a persistent launch one vertex each, took longer than the expansion.  One-
// launch searches with 1 / 4 / 16 vertices at least: 10^3 lattice 308 / 266 / 248 us,
// 20^3 668 / 640 / 549, a comb of 400 vertices a level 11.9 / 10.8 / 9.1 ms; RMAT-12,
// whose few vertices have long lists, 104 / 105 / 110 us, RMAT-14 131 / 133 / 136.
constexpr uint32_t TP_EXPAND_ENTRIES = 16;

// Two-phase expand (vertex frontier -> edge frontier of (neighbour, pred)),
// two_phase/expand_atomic/cta.cuh:606-719.  No culling: lists below the
// grid threshold are expanded in place per tile, longer ones by k_heavy.
__device__ void tp_expand_phase(const BfsArgs& a, int ph, int32_t depth_here, ListSmem& l,
                                uint32_t n_in_arg = kLenFromCounters) {
    const uint32_t n_in = input_len(a, ph, n_in_arg);
    phase_begin(a, ph, n_in, depth_here);
    const int32_t* qin = a.qk[ph & 1];
    const GlobalQueue out = out_queue(a, ph);
    InPlaceSink sink{out, l};
    const uint32_t wgs = min(sharing_wgs(a, n_in, gridDim.x), (n_in + TP_EXPAND_ENTRIES - 1) / TP_EXPAND_ENTRIES);
    const Deal deal = deal_out(n_in, wgs, false);
    for (uint32_t base = 0; blockIdx.x < wgs && base < n_in; base += wgs * BFS_THREADS) {
        const uint32_t i = deal.entry(base, blockIdx.x);
        int32_t u = -1, start = 0, deg = 0;
        if (i < n_in) {
            u = coh_ld(&qin[i], a.coh_in != 0);
            if (valid_vertex(a, u)) {
                start = a.offs[u];
                deg = a.offs[u + 1] - start;
            }
        }
        defer_heavy(a, ph, u, deg, a.grid_th);
        positional_gather<GATHER_K>(a.cols, u, start, deg, l, sink);
    }
}

// Two-phase filter (edge frontier -> edge frontier), bitmask and history
// culls only, no labelling (two_phase/filter_atomic/cta.cuh:308-388).
__device__ void tp_filter_phase(const BfsArgs& a, int ph, PairLevelShared& s) {
    const uint32_t n_in = phase_input_len(a, ph);
    phase_begin(a, ph, n_in);
    const int32_t* qk = a.qk[ph & 1];
    const int32_t* qv = a.qv[ph & 1];
    const GlobalQueue out = out_queue(a, ph);
    for (uint64_t base = (uint64_t)blockIdx.x * BFS_THREADS; base < n_in;
         base += (uint64_t)gridDim.x * BFS_THREADS * CONTRACT_K) {
        bool keep[CONTRACT_K];
        int32_t v[CONTRACT_K], p[CONTRACT_K];
        uint32_t mark[CONTRACT_K];
#pragma unroll
        for (int r = 0; r < CONTRACT_K; ++r) {
            const uint64_t i = base + (uint64_t)r * gridDim.x * BFS_THREADS + threadIdx.x;
            keep[r] = i < n_in;
            v[r] = keep[r] ? coh_ld(&qk[i], a.coh_in != 0) : -1;
            p[r] = keep[r] ? coh_ld(&qv[i], a.coh_in != 0) : 0;
        }
#pragma unroll
        for (int r = 0; r < CONTRACT_K; ++r) {
            keep[r] = keep[r] && valid_vertex(a, v[r]);
            mark[r] = keep[r] ? mark_load(a, v[r]) : 0u;
        }
#pragma unroll
        for (int r = 0; r < CONTRACT_K; ++r)
            keep[r] = keep[r] && !mark_seen(a, v[r], mark[r]) && !history_seen(s.hist, v[r]);
        lq_append_batch<true>(s.q, out, keep, v, p);
        lq_flush<true>(s.q, out, LQ_CAP / 2);
    }
    lq_flush<true>(s.q, out, 1);
}

// Bottom-up step of the direction-optimizing traversal (no counterpart in
// the reference): every unvisited vertex looks for a neighbour in the current
// frontier bitmap and stops at the first hit.  Only valid on symmetric
// graphs.  The step is a chain of dependent loads (visited word -> offsets
// -> column -> bitmap word), so latency, not bandwidth, bounds it; every
// wave therefore works on its own 64-vertex tiles with no workgroup
// barriers, so a stalled wave never holds the others:
//  * a tile whose 64 vertices are all visited is skipped after one load per
//    lane (isolated vertices of symmetric graphs are pre-marked visited by
//    the reset, so late levels skip almost every tile);
//  * stage 1: each lane checks the first BU_FIRST neighbours of its vertex
//    with independent loads;
//  * stage 2: vertices still unresolved with neighbours left are scanned by
//    BU_GROUP-lane groups of the wave, BU_GROUP neighbours per step, lowest
//    lane wins (the first frontier neighbour in list order).
// A wave owns the two bitmap words of its 64 vertices, so visited/next words
// are written without atomics.  The next frontier is only its bitmap: a
// top-down step that follows lists it itself (td_bitmap_phase), so a
// bottom-up step reserves no queue space and its one atomic per workgroup is
// the partial sum of what it found.
// Measured on RMAT-22 (ms per search): BU_FIRST 1-3 within 1 % of each
// other, 4 about 2 % slower, 6 and 8 4-10 % slower; BU_GROUP 4 and 16 no
// better than 8.
constexpr int BU_FIRST = 2;
constexpr int BU_GROUP = 8;
constexpr int BU_WAVE_GROUPS = kWave / BU_GROUP;
constexpr int BU_LISTS = 4;  // lists each group scans side by side

struct BuWave {
    int32_t start[kWave];  // pending entry: next edge to scan
    int32_t end[kWave];
    int32_t parent[kWave];
};

struct BuShared {
    BuWave w[BFS_WAVES];
    unsigned long long red[BFS_WAVES];
};

// LDS written by some lanes of a wave and read by others after it: keep the
// compiler from reordering across this point (a wave's LDS operations
// complete in program order).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// LDS of a direction-optimizing level: the top-down step's queue and gather
// staging or the bottom-up step's per-wave scratch (about 15 KB: eight
// workgroups of 256 threads can stay resident per CU).
constexpr int DO_GATHER_K = 4;
struct DoTdShared {
    LdsKeyQueue qv;
    ListSmem g;
    int32_t list[BM_LIST];
    unsigned long long red[BFS_WAVES];
};
// Start state of a level (do_level_in).
struct DoLevelIn {
    int32_t ph;
    uint32_t n_f;      // frontier vertices: queued by a top-down step, or found by a bottom-up one
    uint32_t prev_dir;
    long long m_f;     // their degree sum
    long long vis;     // degree sum of the vertices visited before them
};
struct DoShared {
    union {
        DoTdShared td;
        BuShared bu;
    };
    DoLevelIn in;
};

__device__ __forceinline__ bool bm_test(const uint32_t* bm, int32_t u) { return (bm[u >> 5] >> (u & 31)) & 1u; }

__device__ void bu_waves(const BfsArgs& a, int ph, int32_t depth_next, const uint32_t* cur, uint32_t* next,
                         BuShared& s) {
    const int lane = lane_id();
    const int wid = threadIdx.x / kWave;
    BuWave& W = s.w[wid];
    const int grp = lane / BU_GROUP, sub = lane % BU_GROUP;
    const int gbase = lane & ~(BU_GROUP - 1);
    unsigned long long acc = 0;  // (degree sum << 32) | vertices found by this lane
    // The frontier by its labels in a small graph, else by its bitmap (which
    // small graphs' top-down steps do not set).
    auto in_frontier = [&](int32_t u) -> bool {
        return a.by_label ? a.depth[u] == depth_next - 1 : bm_test(cur, u);
    };
    // Tiles go round by round over the launch's waves, each round rotated
    // against the last: with equal residues every wave would get tiles of like
    // ids, and in an RMAT graph ids with the same low bits zero are hubs
    // together (the slowest wave of the first bottom-up level of RMAT-22 took
    // 85 us, the average one 51).
    const int64_t nw = (int64_t)gridDim.x * BFS_WAVES;
    const int64_t turn = (nw * 5 / 13) | 1;
    int64_t pos = (int64_t)blockIdx.x * BFS_WAVES + wid, round0 = 0;
    // The next tile's visited word and row offsets are loaded one iteration
    // ahead (whether or not the vertex turns out to be visited), so the
    // current tile's scan overlaps the next tile's first two round trips.
    int64_t vb = pos * kWave;
    uint32_t nvw = 0u;
    int32_t noff0 = 0, noff1 = 0;
    if (vb + lane < a.n) {
        const int32_t v = (int32_t)(vb + lane);
        nvw = mark_load(a, v);
        noff0 = a.offs[v];
        noff1 = a.offs[v + 1];
    }
    while (round0 * kWave < a.n) {
        const int64_t vcur = vb;
        const int32_t v = (int32_t)(vb + lane);
        const uint32_t vw = nvw;
        const int32_t off0 = noff0, off1 = noff1;
        round0 += nw;
        pos += turn;
        if (pos >= nw) pos -= nw;
        vb = (round0 + pos) * kWave;
        if (vb + lane < a.n) {
            const int32_t vn = (int32_t)(vb + lane);
            nvw = mark_load(a, vn);
            noff0 = a.offs[vn];
            noff1 = a.offs[vn + 1];
        }
        const bool active = (vcur + lane < a.n) && !mark_seen(a, v, vw);
        if (__ballot(active) == 0) continue;
        int32_t start = 0, deg = 0, parent = -1;
        if (active) {
            start = off0;
            deg = off1 - off0;
        }
        // Stage 1: the first BU_FIRST neighbours, loads issued together.
        if (deg > 0) {
            int32_t u[BU_FIRST];
#pragma unroll
            for (int k = 0; k < BU_FIRST; ++k) u[k] = (k < deg) ? a.cols[start + k] : -1;
#pragma unroll
            for (int k = BU_FIRST - 1; k >= 0; --k)
                if (u[k] >= 0 && in_frontier(u[k])) parent = u[k];
        }
        // Stage 2: the wave's unresolved lists, one per BU_GROUP-lane group.
        const bool pend = parent < 0 && deg > BU_FIRST;
        const uint64_t pm = __ballot(pend);
        if (pm) {
            const int slot = lane_prefix(pm);
            if (pend) {
                W.start[slot] = start + BU_FIRST;
                W.end[slot] = start + deg;
            }
            wave_lds_sync();
            const int np = __popcll(pm);
            for (int i0 = grp; i0 - grp < np; i0 += BU_LISTS * BU_WAVE_GROUPS) {
                int32_t e[BU_LISTS], e1[BU_LISTS], hit_u[BU_LISTS];
#pragma unroll
                for (int k = 0; k < BU_LISTS; ++k) {
                    const int i = i0 + k * BU_WAVE_GROUPS;
                    e[k] = i < np ? W.start[i] + sub : 0;
                    e1[k] = i < np ? W.end[i] : 0;
                    hit_u[k] = -1;
                }
                uint64_t live;
                do {
                    int32_t u[BU_LISTS];
                    bool hit[BU_LISTS];
                    bool more = false;
#pragma unroll
                    for (int k = 0; k < BU_LISTS; ++k) u[k] = e[k] < e1[k] ? a.cols[e[k]] : -1;
#pragma unroll
                    for (int k = 0; k < BU_LISTS; ++k) hit[k] = u[k] >= 0 && in_frontier(u[k]);
#pragma unroll
                    for (int k = 0; k < BU_LISTS; ++k) {
                        const uint32_t hm = (uint32_t)(__ballot(hit[k]) >> gbase) & ((1u << BU_GROUP) - 1);
                        const int32_t first = __shfl(u[k], gbase + (hm ? __ffsll((unsigned long long)hm) - 1 : 0), kWave);
                        if (hm) {
                            hit_u[k] = first;
                            e1[k] = 0;  // resolved
                        }
                        e[k] += BU_GROUP;
                        more |= e[k] < e1[k];
                    }
                    live = __ballot(more);
                } while (live);
#pragma unroll
                for (int k = 0; k < BU_LISTS; ++k) {
                    const int i = i0 + k * BU_WAVE_GROUPS;
                    if (sub == 0 && i < np) W.parent[i] = hit_u[k];
                }
            }
            wave_lds_sync();
            if (pend) parent = W.parent[slot];
            wave_lds_sync();  // the next tile rewrites the scratch
        }
        const bool found = parent >= 0;
        if (found) {
            a.depth[v] = depth_next;
            a.pred[v] = parent;
            acc += ((unsigned long long)deg << 32) | 1ull;
        }
        const uint64_t fm = __ballot(found);
        if ((lane & 31) == 0) {
            const int64_t w = v >> 5;
            if (w < a.words) {
                const uint32_t bits = (lane == 0) ? (uint32_t)fm : (uint32_t)(fm >> 32);
                next[w] = bits;
                if (bits && !a.by_label) a.visited[w] = vw | bits;
            }
        }
    }
    wg_add_u64(acc, spread_at(a.spread, ph + 1, blockIdx.x % SPREAD), s.red);
}

// Direction for level ph of the direction-optimizing traversal (Beamer,
// Asanovic, Patterson, SC 2012).  Every workgroup evaluates the same counters
// (finalized by the previous launch), so all agree without host involvement.
// m_f = degree sum of the frontier, m_u = edges of unvisited vertices;
// top-down -> bottom-up when m_f > m_u / alpha, back when n_f < n / beta.
__device__ __forceinline__ uint32_t do_direction(const BfsArgs& a, uint32_t n_f, long long m_f, long long vis,
                                                 uint32_t prev) {
    if (!a.symmetric) return 0;
    long long m_u = a.edges - vis - m_f;
    if (m_u < 0) m_u = 0;
    if (prev == 0) return (m_f * (long long)a.do_alpha > m_u) ? 1u : 0u;
    return ((long long)n_f * (long long)a.do_beta < (long long)a.n) ? 0u : 1u;
}

// ===========================================================================
// Kernel bodies.
// ===========================================================================

enum SeedMode { SEED_VERTEX = 0, SEED_EDGE = 1, SEED_DO = 2 };

// Reset's label initialisation fused with the search prologue (the
// reference's MemsetKernel x 2, csr_problem.cuh:723-745, then the
// iteration-0 prologue of contract_expand_atomic/kernel.cuh:307-332 and
// expand_contract_atomic/kernel.cuh:305-319) in one launch: depth and
// predecessor := -1, visited mask and the first two frontier bitmaps := 0,
// except the source, which vertex modes label at once (depth 0, pred -2,
// visited, and its frontier bit for the direction-optimizing mode); edge
// mode leaves it unlabelled and enqueues (src, -2) for contraction.  Every
// value is written by exactly one thread, so no ordering is needed inside
// the launch.  Workgroup 0 also resets the counters; the grid barrier's
// release epoch is left alone (it grows over the problem's lifetime).
__device__ void reset_seed_body(const BfsArgs& a, int ph, int32_t src, int mode) {
    const bool label_src = mode != SEED_EDGE;
    const int32_t stride = gridDim.x * blockDim.x;
    for (int32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < a.n; i += stride) {
        const bool s = label_src && i == src;
        a.depth[i] = s ? 0 : -1;
        a.pred[i] = s ? -2 : -1;
    }
    const uint32_t sbit = label_src ? (1u << (src & 31)) : 0u;
    const int32_t sw = src >> 5;
    uint32_t* fcur = a.fbm[ph % 3];
    uint32_t* fnext = a.fbm[(ph + 1) % 3];
    for (int32_t w = blockIdx.x * blockDim.x + threadIdx.x; w < a.words; w += stride) {
        // Isolated vertices of a symmetric graph can never be reached:
        // marking them visited lets bottom-up steps skip them (their labels
        // stay -1).  The source keeps only its own seeding.
        uint32_t vis = a.iso ? a.iso[w] : 0u;
        if (w == sw) vis = (vis & ~(1u << (src & 31))) | sbit;
        a.visited[w] = vis;
        fcur[w] = (mode == SEED_DO && w == sw) ? sbit : 0u;
        fnext[w] = 0u;
    }
    if (blockIdx.x != 0) return;
    if (mode == SEED_DO && threadIdx.x < 4 * SPREAD) {
        const int level = (int)threadIdx.x / SPREAD, i = (int)threadIdx.x % SPREAD;
        const bool first = level == (ph & 3) && i == 0;
        *spread_at(a.spread, level, i) = first ? (unsigned long long)(a.offs[src + 1] - a.offs[src]) << 32 : 0ull;
    }
    if (threadIdx.x != 0) return;
    DevCounters* c = a.ctr;
    for (int i = 0; i < 4; ++i) {
        c->qlen[i] = 0;
        c->vis_edges[i] = 0;
        c->dir[i] = 0;
    }
    c->heavy_alloc[0] = 0;
    c->heavy_alloc[1] = 0;
    c->ph_base = 0;
    c->overflow = 0;
    c->last_level = 0;
    c->levels_run = 0;
    c->saturated = 0;
    c->queued = 0;
    c->bar_abort = 0;
    c->corrupt = 0;
    *a.max_depth = 0;
    a.qk[ph & 1][0] = src;
    if (mode == SEED_EDGE) a.qv[ph & 1][0] = -2;
    c->qlen[ph & 3] = 1;
}

__device__ __forceinline__ void stats_begin(unsigned long long& t0, const BfsArgs& a) {
    if (a.wg_stats && threadIdx.x == 0) t0 = wg_clock();
}
__device__ __forceinline__ void stats_end(unsigned long long t0, const BfsArgs& a, int slot) {
    if (a.wg_stats && threadIdx.x == 0) {
        const unsigned long long t1 = wg_clock();
        atomic_add_u64(&a.wg_stats[0], t1 - t0);
        // per-launch span: [2 + 2*slot] = min start, [3 + 2*slot] = max end
        __hip_atomic_fetch_min(&a.wg_stats[2 + 2 * slot], t0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_fetch_max(&a.wg_stats[3 + 2 * slot], t1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// In a captured, replayed level loop (dev_base set) a kernel's phase
// argument is relative to ctr->ph_base, which the loop's last node advances,
// and its depth argument is relative to that phase.
__device__ __forceinline__ void resolve_phase(const BfsArgs& a, int& ph, int32_t& depth) {
    if (a.dev_base) {
        ph += (int)ld_relaxed(&a.ctr->ph_base);
        depth += ph;
    }
}

enum PhaseKind { PK_TD = 0, PK_CE = 2, PK_TP_CONTRACT = 3, PK_TP_EXPAND = 4, PK_TP_FILTER = 5 };
template <int KIND>
struct PhaseShared {
    typedef PairLevelShared type;
};
template <>
struct PhaseShared<PK_TD> {
    typedef TdLevelShared type;
};
template <>
struct PhaseShared<PK_TP_EXPAND> {
    typedef TdLevelShared type;
};
template <>
struct PhaseShared<PK_CE> {
    typedef LevelShared type;
};

template <int KIND, typename Shared>
__device__ void phase_body(BfsArgs a, int ph, int32_t depth, int slot, Shared& s) {
    resolve_phase(a, ph, depth);
    unsigned long long t0 = 0;
    stats_begin(t0, a);
    shared_init(s);
    if constexpr (KIND == PK_TD) td_phase<GATHER_K>(a, ph, depth, nullptr, false, s.q, s.l, s.red, gridDim.x, a.grid_th);
    if constexpr (KIND == PK_CE) ce_phase<false>(a, ph, depth, s);
    if constexpr (KIND == PK_TP_CONTRACT) tp_contract_phase(a, ph, depth, s);
    if constexpr (KIND == PK_TP_EXPAND) tp_expand_phase(a, ph, depth, s.l);
    if constexpr (KIND == PK_TP_FILTER) tp_filter_phase(a, ph, s);
    stats_end(t0, a, slot);
}

// What a level kernel of the direction-optimizing traversal needs to know
// before it can start, read in one round trip: one wave of the workgroup loads
// every counter word and every partial sum of all four level slots together
// (following the phase base to the level's slot would be three dependent round
// trips, about 2.5 us of a 7 us level).
constexpr int CTR_WORDS = (int)(sizeof(DevCounters) / 4);
static_assert(CTR_WORDS == kWave && 4 * SPREAD == kWave, "one counter word and one partial sum per lane");

__device__ __forceinline__ void do_level_in(const BfsArgs& a, int ph, DoLevelIn& in) {
    if (threadIdx.x < kWave) {
        const int lane = lane_id();
        const uint32_t w = reinterpret_cast<const uint32_t*>(a.ctr)[lane];
        unsigned long long part = *spread_at(a.spread, lane / SPREAD, lane % SPREAD);
        constexpr int kPh = (int)(offsetof(DevCounters, ph_base) / 4), kDir = (int)(offsetof(DevCounters, dir) / 4),
                      kVis = (int)(offsetof(DevCounters, vis_edges) / 4);
        if (a.dev_base) ph += (int)__shfl(w, kPh, kWave);
        if (lane / SPREAD != (ph & 3)) part = 0ull;
#pragma unroll
        for (int d = kWave / 2; d >= 1; d >>= 1) part += __shfl_xor(part, d, kWave);
        uint32_t n_q = __shfl(w, ph & 3, kWave);
        if (n_q > a.qcap[ph & 1]) n_q = 0;  // an overflowed queue counts as empty
        const uint32_t dir = __shfl(w, kDir + ((ph + 3) & 3), kWave);
        const uint32_t lo = __shfl(w, kVis + 2 * (ph & 3), kWave), hi = __shfl(w, kVis + 2 * (ph & 3) + 1, kWave);
        if (lane == 0) {
            in.ph = ph;
            in.n_f = n_q + (uint32_t)part;
            in.prev_dir = dir;
            in.m_f = (long long)(part >> 32);
            in.vis = (long long)(((unsigned long long)hi << 32) | lo);
        }
    }
    __syncthreads();
}

// One level of the direction-optimizing traversal: the workgroups agree on
// the direction from device counters, clear the bitmap two levels ahead and
// run a top-down or bottom-up step.  An empty frontier makes it a no-op, so
// the host can launch levels ahead of the termination check.
// grid_tier: a k_heavy launch follows; without one, top-down steps split
// their tiles over the workgroups instead.
__device__ void do_level_body(BfsArgs a, int ph, int slot, int grid_tier, DoShared& s) {
    do_level_in(a, ph, s.in);
    ph = s.in.ph;
    const uint32_t n_f = s.in.n_f, prev_dir = s.in.prev_dir;
    const long long m_f = s.in.m_f, vis = s.in.vis;
    if (blockIdx.x == 0 && threadIdx.x < SPREAD) *spread_at(a.spread, ph + 2, threadIdx.x) = 0ull;
    if (n_f == 0) {
        // Keep the slot rotation going so later no-op levels also read 0.
        phase_begin(a, ph, 0);
        return;
    }
    unsigned long long t0 = 0;
    stats_begin(t0, a);
    const uint32_t dir = do_direction(a, n_f, m_f, vis, prev_dir);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        a.ctr->dir[ph & 3] = dir;
        a.ctr->vis_edges[(ph + 1) & 3] = (unsigned long long)(vis + m_f);
    }
    uint32_t* clear = a.fbm[(ph + 2) % 3];
    for (int32_t w = blockIdx.x * BFS_THREADS + threadIdx.x; w < a.words; w += gridDim.x * BFS_THREADS) clear[w] = 0;
    if (dir == 0) {
        // Top-down steps use the first td_grid workgroups; the launch is
        // sized for the bottom-up step, which needs every wave slot.
        const uint32_t tdg = min(gridDim.x, (uint32_t)max(1, a.td_grid));
        if (blockIdx.x < tdg) {
            if (threadIdx.x == 0) s.td.qv.count = 0;
            __syncthreads();
            const int32_t th = grid_tier ? a.grid_th : INT_MAX;
            uint32_t* next_bm = a.by_label ? nullptr : a.fbm[(ph + 1) % 3];
            if (prev_dir == 0)
                td_phase<DO_GATHER_K>(a, ph, ph + 1, next_bm, true, s.td.qv, s.td.g, s.td.red, tdg, th, n_f, !grid_tier);
            else
                td_bitmap_phase<DO_GATHER_K>(a, ph, ph + 1, a.fbm[ph % 3], next_bm, s.td.qv, s.td.g, s.td.list, s.td.red, tdg, th,
                                n_f);
        }
    } else {
        phase_begin(a, ph, 0);
        if (blockIdx.x == 0 && threadIdx.x == 0) st_relaxed(a.max_depth, (uint32_t)ph);
        bu_waves(a, ph, ph + 1, a.fbm[ph % 3], a.fbm[(ph + 1) % 3], s.bu);
    }
    stats_end(t0, a, slot);
}

// Grid tier: the adjacency lists deferred by phase ph, cut into
// HEAVY_CHUNK-edge chunks; workgroups take chunks grid-stride and find each
// chunk's vertex through the chunk map.  Every chunk is checked against the
// entry it names, so stale map words can never index outside a list.
enum HeavyKind { HK_TD = 0, HK_TD_DO = 1, HK_PAIRS = 2 };

// Top-down grid-tier launches need a vertex queue, pair launches write in
// place; small LDS blocks keep them at full residency.
struct TdHeavyShared {
    LdsKeyQueue qv;
    ListSmem l;
    unsigned long long red[BFS_WAVES];
};
struct PairsHeavyShared {
    ListSmem l;
};
template <int KIND>
struct HeavySharedOf {
    typedef TdHeavyShared type;
};
template <>
struct HeavySharedOf<HK_PAIRS> {
    typedef PairsHeavyShared type;
};

// The grid tier's chunks [0, C) of H entries: chunk base + t * gridDim.x + b
// goes to thread t of workgroup b, which finds its piece of a list; the
// workgroup then gathers its 256 pieces positionally, as the level steps do
// with whole lists.
template <typename Sink>
__device__ __forceinline__ void gather_chunks(const BfsArgs& a, uint32_t H, uint32_t C, ListSmem& l, Sink& sink) {
    auto piece = [&](uint32_t c, int32_t& u, int32_t& start, int32_t& len) {
        const int32_t entry = coh_ld(&a.chunk_map[c], a.coh_out != 0);
        if ((uint32_t)entry >= H) return;
        const int2 eu = coh_ld2(&a.heavy[entry], a.coh_out != 0);
        if (!valid_vertex(a, eu.x) || (uint32_t)eu.y > c) return;
        const int32_t s0 = a.offs[eu.x], deg = a.offs[eu.x + 1] - s0;
        const long long off = (long long)(c - (uint32_t)eu.y) * HEAVY_CHUNK;
        if (off >= deg) return;
        u = eu.x;
        start = s0 + (int32_t)off;
        len = min((int32_t)HEAVY_CHUNK, deg - (int32_t)off);
    };
    for (uint64_t base = 0; base + blockIdx.x < C; base += (uint64_t)gridDim.x * BFS_THREADS) {
        int32_t u = -1, start = 0, len = 0;
        const uint64_t c = base + (uint64_t)threadIdx.x * gridDim.x + blockIdx.x;
        if (c < C) piece((uint32_t)c, u, start, len);
        positional_gather<GATHER_K>(a.cols, u, start, len, l, sink);
    }
}

template <int KIND>
__device__ void heavy_body(BfsArgs a, int ph, int32_t depth_next, int slot, typename HeavySharedOf<KIND>::type& s) {
    // Both slots are loaded beside the phase base, not after it.
    const unsigned long long alloc0 =
        __hip_atomic_load(&a.ctr->heavy_alloc[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned long long alloc1 =
        __hip_atomic_load(&a.ctr->heavy_alloc[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    resolve_phase(a, ph, depth_next);
    const unsigned long long alloc = (ph & 1) ? alloc1 : alloc0;
    const uint32_t H = min((uint32_t)(alloc >> 32), a.heavy_cap);
    const uint32_t C = min((uint32_t)alloc, a.chunk_cap);
    if (H == 0 || C == 0) return;
    unsigned long long t0 = 0;
    stats_begin(t0, a);
    if constexpr (KIND != HK_PAIRS) {
        if (threadIdx.x == 0) s.qv.count = 0;
        __syncthreads();
    }
    const GlobalQueue out = out_queue(a, ph);
    if constexpr (KIND == HK_PAIRS) {
        InPlaceSink sink{out, s.l};
        gather_chunks(a, H, C, s.l, sink);
    } else {
        TdSink<1> sink{a, s.qv, out, (KIND == HK_TD_DO && !a.by_label) ? a.fbm[(ph + 1) % 3] : nullptr, depth_next,
                       KIND == HK_TD_DO, 0ull};
        gather_chunks(a, H, C, s.l, sink);
        td_finish(a, ph, sink, s.red);
    }
    stats_end(t0, a, slot);
}

// Persistent kernels: all levels in one launch of a co-resident grid with a software
// grid barrier between phases (contract_expand_atomic::KernelGlobalBarrier,
// kernel.cuh:281-554; two_phase::Kernel, two_phase/kernel.cuh:60-313).
// The loop control (the input frontier's length) is read by one thread per
// workgroup and shared through LDS after each barrier; every workgroup reads
// the same value, so all leave the loop together.  With `sat_limit` set, the
// kernel quits when a frontier exceeds it (SATURATION_QUIT) and records
// where it stopped.
//
// Grid tier: a level's expansion defers lists of at least grid_th edges (as
// the level kernels do); after the level's barrier every workgroup reads the
// same deferral count, and when it is nonzero the whole grid splits those
// lists into chunks (heavy_body) before one more barrier.  Levels without
// hubs pay no extra barrier.  grid_th = INT_MAX turns the tier off.
enum FusedKind { FK_TD = 0, FK_CE = 1, FK_TP = 2 };

template <int KIND>
struct FusedHeavy {
    static constexpr int kind = (KIND == FK_TD) ? HK_TD : HK_PAIRS;
    typedef typename HeavySharedOf<kind>::type shared;
};

template <int KIND>
struct FusedShared {
    typedef LevelShared type;
};
template <>
struct FusedShared<FK_TP> {
    typedef PairLevelShared type;
};
template <>
struct FusedShared<FK_TD> {
    typedef TdLevelShared type;
};

template <int KIND, typename Shared>
__device__ void fused_body(const BfsArgs& a, int ph, int32_t depth, int max_levels, uint32_t sat_limit, Shared& s,
                           typename FusedHeavy<KIND>::shared& hs) {
    unsigned long long t0 = 0, busy = 0;
    if (a.wg_stats && threadIdx.x == 0) t0 = wg_clock();
    shared_init(s);
    // Every phase passes its frontier through agent-scope accesses (the
    // host sets a.persistent, a.coh_in and a.coh_out) and ends with the light
    // barrier.  `a` is read-only here: a kernel that writes into its argument
    // block gets a private copy of all of it, and every field read becomes a
    // scratch load (that cost each persistent strategy a quarter of its rate).
    const GridBarrier bar{a.bar_arrive, &a.ctr->bar_release, &a.ctr->bar_abort, 1u};
    uint32_t epoch = barrier_base_epoch(bar);
    if (blockIdx.x == 0 && threadIdx.x == 0) a.ctr->saturated = 0;
    // Barrier payload: the length of the frontier queue in counter slot
    // `slot` (clamped to 31 bits: a frontier never holds 2^31 entries, since
    // E < 2^31) with bit 31 set when the grid tier has lists deferred by
    // phase `heavy_ph` (heavy_ph < 0: not asked).  Workgroup 0 reads both
    // after every workgroup has arrived.
    auto payload_for = [&a](int slot, int heavy_ph) {
        return [&a, slot, heavy_ph]() -> uint32_t {
            uint32_t len = ld_relaxed(&a.ctr->qlen[slot & 3]);
            if (len > 0x7FFFFFFFu) len = 0x7FFFFFFFu;
            const bool deferred = heavy_ph >= 0 && __hip_atomic_load(&a.ctr->heavy_alloc[heavy_ph & 1], __ATOMIC_RELAXED,
                                                                     __HIP_MEMORY_SCOPE_AGENT) != 0ull;
            return len | (deferred ? 0x80000000u : 0u);
        };
    };
    const bool grid_tier = a.grid_th != INT_MAX;
    // Every thread reads the first level's length itself (written by the
    // launch before this one); later lengths come with the barriers.
    uint32_t n_in = ld_relaxed(&a.ctr->qlen[ph & 3]);
    int level = 0;
    for (; level < max_levels; ++level) {
        if (n_in == 0 || n_in > a.qcap[ph & 1]) break;
        if (sat_limit && n_in > sat_limit) {
            if (blockIdx.x == 0 && threadIdx.x == 0) a.ctr->saturated = 1;
            break;
        }
        unsigned long long tb = 0;
        if (a.wg_stats && threadIdx.x == 0) tb = wg_clock();
        int heavy_ph = ph;          // phase whose deferred lists the grid tier takes
        int32_t heavy_depth = depth;  // depth label of what it discovers (top-down)
        uint32_t word = 0;
        if constexpr (KIND == FK_TD) {
            td_phase<GATHER_K>(a, ph, depth + 1, nullptr, false, s.q, s.l, s.red, gridDim.x, a.grid_th, n_in);
            heavy_depth = depth + 1;
            ph += 1;
        } else if constexpr (KIND == FK_CE) {
            ce_phase<true>(a, ph, depth, s, n_in);
            ph += 1;
        } else if constexpr (KIND == FK_TP) {
            tp_contract_phase(a, ph, depth, s, n_in);
            if (a.wg_stats && threadIdx.x == 0) busy += wg_clock() - tb;
            if (!grid_sync(bar, ++epoch, payload_for(ph + 1, -1), &s.ctl, word)) break;
            if (a.wg_stats && threadIdx.x == 0) tb = wg_clock();
            // An overflowed vertex queue counts as empty (as phase_input_len
            // has it); the overflow flag ends the search.
            uint32_t n_mid = word & 0x7FFFFFFFu;
            if (n_mid > a.qcap[(ph + 1) & 1]) n_mid = 0;
            tp_expand_phase(a, ph + 1, depth, s.l, n_mid);
            heavy_ph = ph + 1;
            ph += 2;
        }
        depth += 1;
        if (a.wg_stats && threadIdx.x == 0) busy += wg_clock() - tb;
        if (!grid_sync(bar, ++epoch, payload_for(ph, grid_tier ? heavy_ph : -1), &s.ctl, word)) break;
        if (word & 0x80000000u) {
            // Lists this level deferred: the whole grid takes them in
            // chunks, appending to the same next frontier.
            heavy_body<FusedHeavy<KIND>::kind>(a, heavy_ph, heavy_depth, 0, hs);
            if (!grid_sync(bar, ++epoch, payload_for(ph, -1), &s.ctl, word)) break;
        }
        n_in = word & 0x7FFFFFFFu;
        // A nonempty next frontier tells that the level claimed vertices: those
        // on it (top-down, at `depth`), or those whose edges are on it.
        if (KIND != FK_TP && n_in != 0 && blockIdx.x == 0 && threadIdx.x == 0)
            atomic_max_u32(a.max_depth, (uint32_t)(KIND == FK_TD ? depth : depth - 1));
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        a.ctr->levels_run = (uint32_t)level;
        a.ctr->last_level = (uint32_t)ph;
    }
    if (a.wg_stats && threadIdx.x == 0) {
        atomic_add_u64(&a.wg_stats[0], busy);
        atomic_add_u64(&a.wg_stats[1], wg_clock() - t0);
    }
}

// Narrow persistent kernel: expand-contract for grids of at most kAllToAllMax
// workgroups, which high-diameter and small graphs use.  Their levels are a
// chain of dependent accesses, and the two longest links were the barrier
// (three hops through workgroup 0, 2.2 us) and the frontier queue's counter
// (every workgroup's reservation at one address, 11.4 ns each: 2.9 us for
// 256).  Here a workgroup writes what it finds to its own piece of the
// frontier as soon as it is claimed (no shared counter, no LDS queue), and the
// piece's length travels in its arrival word of the all-to-all barrier: every
// workgroup gets all the lengths with the barrier itself, and finds any entry
// by a search over their prefix sums.  What does not fit a piece goes to the
// shared queue as before and comes first in the next frontier.
struct NarrowShared {
    ListSmem l;
    uint32_t first[kAllToAllMax];  // entries before each workgroup's piece
    uint32_t count;                // entries found by this workgroup
    uint32_t spilled, deferred;
    int s_wave[BFS_WAVES];
};
static_assert(kAllToAllMax == BFS_THREADS, "one piece per thread");

constexpr uint32_t kNarrowSpilled = 0x40000000u, kNarrowDeferred = 0x80000000u, kNarrowCount = 0x3FFFFFFFu;

struct NarrowSink {
    const BfsArgs& a;
    NarrowShared& s;
    int32_t* piece;  // a.region entries
    const GlobalQueue& out;
    int32_t depth_next;
    __device__ __forceinline__ void reserve(uint32_t, ListSmem&) {}
    __device__ __forceinline__ void step_end() {}
    template <int K>
    __device__ __forceinline__ void step(uint32_t, const bool (&valid)[K], const int32_t (&v)[K],
                                         const int32_t (&src)[K]) {
        bool won[K];
        td_claim(a, valid, v, src, depth_next, won);
        uint64_t m[K];
        uint32_t cnt = 0;
#pragma unroll
        for (int r = 0; r < K; ++r) {
            m[r] = __ballot(won[r]);
            cnt += (uint32_t)__popcll(m[r]);
        }
        if (cnt == 0) return;
        uint32_t base = 0;
        if (lane_id() == 0) base = atomicAdd(&s.count, cnt);
        base = (uint32_t)wave_bcast((int)base, 0);
        const uint32_t spill_start = base > a.region ? base : a.region;
        uint32_t gb = 0;
        if (base + cnt > a.region) {
            if (lane_id() == 0) {
                gb = atomic_add_u32(out.len, base + cnt - spill_start);
                s.spilled = 1u;
            }
            gb = (uint32_t)wave_bcast((int)gb, 0);
        }
        uint32_t at = base;
#pragma unroll
        for (int r = 0; r < K; ++r) {
            const uint32_t pos = at + (uint32_t)lane_prefix(m[r]);
            at += (uint32_t)__popcll(m[r]);
            if (!won[r]) continue;
            if (pos < a.region) {
                coh_st(&piece[pos], v[r], true);
            } else if (gb + (pos - spill_start) < out.cap) {
                coh_st(&out.keys[gb + (pos - spill_start)], v[r], true);
            } else {
                st_relaxed(out.overflow, 1u);
            }
        }
    }
};

__device__ void fused_narrow_body(const BfsArgs& a, int ph, int32_t depth, NarrowShared& s) {
    unsigned long long t0 = 0, busy = 0;
    if (a.wg_stats && threadIdx.x == 0) t0 = wg_clock();
    const GridBarrier base_of{a.bar_arrive, &a.ctr->bar_release, &a.ctr->bar_abort, 1u};
    uint32_t epoch = barrier_base_epoch(base_of);
    const bool grid_tier = a.grid_th != INT_MAX;
    const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
    // The first frontier is the source, in the shared queue.
    uint32_t n_main = ld_relaxed(&a.ctr->qlen[ph & 3]), n_in = n_main;
    s.first[threadIdx.x] = 0u;
    int level = 0;
    for (;; ++level) {
        if (n_in == 0) break;
        if (n_in > a.qcap[ph & 1]) {
            // A frontier the queue could not hold is an overflow here too,
            // wherever its entries are.
            if (lead) st_relaxed(&a.ctr->overflow, 1u);
            break;
        }
        unsigned long long tb = 0;
        if (a.wg_stats && threadIdx.x == 0) tb = wg_clock();
        phase_begin(a, ph, n_in);
        if (threadIdx.x == 0) s.count = s.spilled = s.deferred = 0u;
        __syncthreads();  // also: `first` is complete
        const int32_t* qin = a.qk[ph & 1];
        const int32_t* pieces = a.regions + (size_t)(ph & 1) * kAllToAllMax * a.region;
        const GlobalQueue out = out_queue(a, ph);
        NarrowSink sink{a, s, a.regions + ((size_t)((ph + 1) & 1) * kAllToAllMax + blockIdx.x) * a.region, out,
                        depth + 1};
        const Deal deal = deal_out(n_in, gridDim.x, false);
        for (uint32_t base = 0; base < n_in; base += gridDim.x * BFS_THREADS) {
            const uint32_t i = deal.entry(base, blockIdx.x);
            int32_t u = -1, start = 0, deg = 0;
            if (i < n_in) {
                if (i < n_main) {
                    u = coh_ld(&qin[i], true);
                } else {
                    const uint32_t j = i - n_main;
                    uint32_t w = 0;  // last piece with first <= j
#pragma unroll
                    for (uint32_t h = kAllToAllMax / 2; h >= 1; h >>= 1)
                        if (s.first[w + h] <= j) w += h;
                    u = coh_ld(&pieces[w * a.region + (j - s.first[w])], true);
                }
                if (valid_vertex(a, u)) {
                    start = a.offs[u];
                    deg = a.offs[u + 1] - start;
                }
            }
            if (grid_tier) {
                if (deg >= a.grid_th) s.deferred = 1u;
                defer_heavy(a, ph, u, deg, a.grid_th);
            }
            positional_gather<GATHER_K>(a.cols, u, start, deg, s.l, sink);
        }
        depth += 1;
        ph += 1;
        __syncthreads();
        if (a.wg_stats && threadIdx.x == 0) busy += wg_clock() - tb;
        uint32_t word = 0;
        auto mine = [&] {
            return min(s.count, a.region) | (s.spilled ? kNarrowSpilled : 0u) |
                   (s.deferred ? kNarrowDeferred : 0u);
        };
        if (!grid_sync_words(a.bar_words, &a.ctr->bar_abort, ++epoch, mine(), word)) break;
        bool spilled = false;
        if (__syncthreads_or((word & ~kNarrowCount) != 0u)) {
            if (__syncthreads_or((word & kNarrowDeferred) != 0u)) {
                // Lists this level deferred: the whole grid takes them in
                // chunks, appending to the same pieces.
                const unsigned long long alloc = __hip_atomic_load(&a.ctr->heavy_alloc[(ph - 1) & 1], __ATOMIC_RELAXED,
                                                                   __HIP_MEMORY_SCOPE_AGENT);
                gather_chunks(a, min((uint32_t)(alloc >> 32), a.heavy_cap), min((uint32_t)alloc, a.chunk_cap), s.l,
                              sink);
                __syncthreads();
                if (!grid_sync_words(a.bar_words, &a.ctr->bar_abort, ++epoch, mine(), word)) break;
            }
            spilled = __syncthreads_or((word & kNarrowSpilled) != 0u) != 0;
        }
        n_main = spilled ? ld_relaxed(&a.ctr->qlen[ph & 3]) : 0u;
        int total;
        s.first[threadIdx.x] =
            (uint32_t)wg_exclusive_scan<BFS_THREADS>((int)(word & kNarrowCount), total, s.s_wave);
        n_in = n_main + (uint32_t)total;
        if (n_in != 0 && lead) atomic_max_u32(a.max_depth, (uint32_t)depth);
    }
    if (lead) {
        a.ctr->levels_run = (uint32_t)level;
        a.ctr->last_level = (uint32_t)ph;
        // Later launches continue the epochs.
        __hip_atomic_store(&a.ctr->bar_release, (unsigned long long)epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (a.wg_stats && threadIdx.x == 0) {
        atomic_add_u64(&a.wg_stats[0], busy);
        atomic_add_u64(&a.wg_stats[1], wg_clock() - t0);
    }
}

// Global-barrier benchmark (test/gbarrier/test_gbarrier.cu:43-50): the
// kernel does nothing but pass `iterations` barriers.
__device__ void gbarrier_bench_body(const GridBarrier& bar, int iterations, uint32_t* s_word) {
    uint32_t epoch = barrier_base_epoch(bar);
    for (int i = 0; i < iterations; ++i)
        if (!grid_sync(bar, ++epoch, s_word)) break;
}

// Cross-workgroup visibility check of the grid barrier: each workgroup writes
// a slab of words, passes the barrier, then compares three other
// workgroups' slabs with the expected pattern.  Every index is fixed by
// (block, lane) and in bounds; loaded values are only compared.
__device__ __forceinline__ uint32_t gb_pattern(uint32_t it, uint32_t b, uint32_t j) {
    uint32_t x = it * 0x9E3779B1u ^ (b * 0x85EBCA6Bu) ^ (j * 0xC2B2AE35u);
    x ^= x >> 15;
    x *= 0x2C1B3C6Du;
    x ^= x >> 12;
    return x | 1u;
}

__device__ void gbarrier_check_body(const GridBarrier& bar, uint32_t* data, int words, int iterations,
                                    unsigned long long* mismatches, uint32_t* s_word) {
    const uint32_t G = gridDim.x, b = blockIdx.x;
    uint32_t epoch = barrier_base_epoch(bar);
    unsigned long long bad = 0;
    const bool coh = bar.light != 0;  // light barrier: the slabs go through agent-scope accesses
    for (int it = 0; it < iterations; ++it) {
        for (int j = threadIdx.x; j < words; j += BFS_THREADS)
            coh_st((int32_t*)&data[(size_t)b * words + j], (int32_t)gb_pattern(it, b, j), coh);
        // The payload is the iteration number as workgroup 0 saw it in a
        // word every workgroup wrote before arriving: all must agree.
        uint32_t seen = 0;
        if (!grid_sync(bar, ++epoch,
                       [&] {
                           return (uint32_t)coh_ld((const int32_t*)&data[(size_t)(G - 1) * words], coh) ^
                                  gb_pattern(it, G - 1, 0) ^ (uint32_t)it;
                       },
                       s_word, seen))
            break;
        bad += (seen != (uint32_t)it) ? 1u : 0u;
        const uint32_t others[3] = {(b + 1) % G, (b + G / 2 + 1) % G, (b + G - 1) % G};
        for (int k = 0; k < 3; ++k) {
            const uint32_t o = others[k];
            for (int j = threadIdx.x; j < words; j += BFS_THREADS)
                bad += ((uint32_t)coh_ld((const int32_t*)&data[(size_t)o * words + j], coh) != gb_pattern(it, o, j))
                           ? 1u : 0u;
        }
        if (!grid_sync(bar, ++epoch, s_word)) break;
    }
    if (bad) atomic_add_u64(mismatches, bad);
}

}  // namespace b40c
