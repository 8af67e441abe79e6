// Single-pass kernels over blocks of consecutive input: each block publishes a
// sum and learns the sum of the blocks before it from a serving workgroup
// (prefix sum, run heads, sorted keys to CSR).
#pragma once
#include <algorithm>
#include <cstring>

#include "common.hpp"
#include "internal.hpp"

namespace b40c {
namespace {

constexpr int CHAIN_THREADS = 256;  // per workgroup of a chained kernel
constexpr int CHAIN_WAVES = CHAIN_THREADS / kWave;

// One 64-bit word per block: its own sum (CHAIN_SUM), which the serving
// workgroup replaces by the sum of all blocks before it (CHAIN_PREFIX).  Words
// are CHAIN_STRIDE apart, one per 64-byte line: stores to one line are
// serialised (33 ns each), and blocks in order store in order, so packed words
// limited a scan to one block per 55 ns (2^28 elements in 3.6 ms).
constexpr unsigned long long CHAIN_SUM = 1ull << 62, CHAIN_PREFIX = 2ull << 62, CHAIN_VALUE = CHAIN_SUM - 1;
constexpr int CHAIN_STRIDE = 8;

// No wait needs to end.  A chained kernel and a persistent one that are each
// partly resident keep the other's missing workgroups off the GPU (XCDs dispatch
// on their own, so even a block's predecessors may be missing).  The serving
// workgroup gives up after kChainSpins polls without a new sum, a block after a
// quarter of them without its prefix (about 11 and 3 ms; a poll is 0.7 us and a whole
// scan of 2^28 elements 0.5 ms).  Such blocks list themselves and leave, and the
// host finishes them when all sums are there.  (Blocks that also looked whether the
// server had given up made a scan of 2^26 elements 1 to 2 us slower.)
constexpr uint32_t kChainSpins = 1u << 14;

// Report of a chained call.
struct ChainReport {
    uint64_t total;
    uint32_t open;  // some blocks may be unfinished
};

// Device words of a chained call beside the blocks' words.
struct ChainMeta {
    uint64_t before;      // where the serving workgroup gave up: the sum,
    int32_t base;         // and the first block without its prefix
    uint32_t unfinished;  // blocks in the list
};

// What a chained kernel gets: one word per block (above), and in the second of a
// line's words entry i of the list of unfinished blocks.
struct Chain {
    unsigned long long* words;
    ChainMeta* meta;
    ChainReport* report;
    uint64_t before;  // what comes before the first block
    int32_t blocks;
};

// Chained kernels come in two forms: REST finishes the listed blocks, whose
// prefixes are all there.  (A flag among the arguments had to be loaded before
// anything else: 2 us of a scan of 2^26 elements.)
template <bool REST>
__device__ __forceinline__ bool chain_serves() {
    return !REST && blockIdx.x == 0;
}
template <bool REST>
__device__ __forceinline__ int chain_block(const Chain& c) {
    if (!REST) return (int)blockIdx.x - 1;
    return __builtin_amdgcn_readfirstlane((int)c.words[(size_t)blockIdx.x * CHAIN_STRIDE + 1]);
}

__device__ __forceinline__ unsigned long long chain_load(const Chain& c, int b) {
    return __hip_atomic_load(&c.words[(size_t)b * CHAIN_STRIDE], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void chain_store(const Chain& c, int b, unsigned long long w) {
    __hip_atomic_store(&c.words[(size_t)b * CHAIN_STRIDE], w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ __launch_bounds__(CHAIN_THREADS) void k_chain_init(Chain c) {
    for (int i = blockIdx.x * CHAIN_THREADS + threadIdx.x; i < c.blocks; i += gridDim.x * CHAIN_THREADS)
        c.words[(size_t)i * CHAIN_STRIDE] = 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) *c.meta = ChainMeta{c.before, 0, 0u};
}

struct ChainServeShared {
    uint64_t sum[CHAIN_WAVES];
    uint32_t ready[CHAIN_WAVES];
};

// Workgroup 0 of a chained kernel: turns the blocks' sums into prefixes, up to
// 256 of them per round trip (0.7 us), and reports the total.  The blocks poll one
// line each; when every block looked back over its predecessors' words itself,
// the polling alone took 20 to 45 us of a scan of 2^26 elements.  `before` comes
// before block `base`, the first to serve.
__device__ __forceinline__ void chain_serve(const Chain& c, ChainServeShared& s, uint64_t before, int base) {
    const int tid = threadIdx.x, lane = lane_id(), wid = tid / kWave;
    uint32_t spins = 0;
    while (base < c.blocks) {
        const int b = base + tid;
        const unsigned long long w = b < c.blocks ? chain_load(c, b) : 0ull;
        const uint64_t waiting = __ballot(w < CHAIN_SUM);
        const int ready = waiting ? __ffsll((unsigned long long)waiting) - 1 : kWave;
        const uint64_t v = lane < ready ? (w & CHAIN_VALUE) : 0ull;
        uint64_t incl = v;
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) {
            const uint64_t o = __shfl_up(incl, d, kWave);
            if (lane >= d) incl += o;
        }
        if (lane == kWave - 1) {
            s.sum[wid] = incl;
            s.ready[wid] = (uint32_t)ready;
        }
        __syncthreads();
        uint64_t mine = before;
        bool open = true;
        int taken = 0;
#pragma unroll
        for (int k = 0; k < CHAIN_WAVES; ++k) {
            if (k == wid && open && lane < ready) chain_store(c, b, CHAIN_PREFIX | (mine + incl - v));
            if (open) {
                mine += s.sum[k];
                taken += (int)s.ready[k];
                open = s.ready[k] == kWave;
            }
        }
        __syncthreads();
        before = mine;
        base += taken;
        if (taken) {
            spins = 0;
        } else {
            if (++spins > kChainSpins) break;
            __builtin_amdgcn_s_sleep(1);
        }
    }
    if (tid == 0) {
        if (base < c.blocks) {
            c.meta->before = before;
            c.meta->base = base;
            c.report->open = 1;
        } else {
            c.report->total = before;
        }
    }
}

// The word with the sum of the blocks before `block`, which publishes `mine`; one
// lane.  Zero: the block is listed and leaves without its output.
template <bool REST>
__device__ __forceinline__ unsigned long long chain_before(const Chain& c, int block, uint64_t mine) {
    if (REST) return chain_load(c, block);
    chain_store(c, block, CHAIN_SUM | mine);
    unsigned long long w;
    uint32_t spins = 0;
    while ((w = chain_load(c, block)) < CHAIN_PREFIX) {
        if (++spins > kChainSpins / 4) {
            c.report->open = 1;
            const uint32_t at = atomic_add_u32(&c.meta->unfinished, 1u);
            c.words[(size_t)at * CHAIN_STRIDE + 1] = (unsigned long long)block;
            return 0;
        }
        __builtin_amdgcn_s_sleep(1);
    }
    return w;
}

__global__ __launch_bounds__(CHAIN_THREADS) void k_chain_resume(Chain c) {
    __shared__ ChainServeShared s;
    if (chain_load(c, c.blocks - 1) >= CHAIN_PREFIX) return;  // only blocks gave up
    chain_serve(c, s, c.meta->before, c.meta->base);
}

// Chained calls: chain words, then the call's own, then a report for when there
// is no pinned slot.
inline size_t chain_bytes(int64_t blocks) {
    return (size_t)blocks * CHAIN_STRIDE * 8 + sizeof(ChainMeta) + sizeof(ChainReport);
}

// One chained call's scratch and report.
struct ChainCall {
    ReportSlot slot;
    DeviceBuffer mem;  // freed before the slot is given back
    Chain chain{};
    // `words`: chain_bytes(blocks) of the caller's device memory, or null to allocate them.
    b40c_status start(int64_t blocks, hipStream_t stream, void* words = nullptr) {
        if (!words) B40C_TRY(mem.alloc(chain_bytes(blocks)));
        chain.words = static_cast<unsigned long long*>(words ? words : mem.ptr);
        chain.meta = reinterpret_cast<ChainMeta*>(chain.words + (size_t)blocks * CHAIN_STRIDE);
        chain.report = reinterpret_cast<ChainReport*>(chain.meta + 1);
        if (slot.take()) chain.report = static_cast<ChainReport*>(slot.dev);
        return B40C_OK;
    }
    // One chained kernel over `blocks` blocks after `before`, to its end: launch(chain,
    // workgroups, rest) launches it, and its REST form for the blocks that gave up.
    // `total` is `before` and all the blocks' sums.
    template <typename Launch>
    b40c_status run(int64_t blocks, uint64_t before, uint64_t& total, hipStream_t stream, Launch launch) {
        chain.blocks = (int32_t)blocks;
        chain.before = before;
        if (slot.host)
            std::memset(slot.host, 0, sizeof(ChainReport));
        else
            B40C_TRY(fill_u32(reinterpret_cast<uint32_t*>(chain.report), 0, sizeof(ChainReport) / 4, stream));
        hipLaunchKernelGGL(k_chain_init, dim3((unsigned)std::min<int64_t>((blocks + CHAIN_THREADS - 1) / CHAIN_THREADS, 256)),
                           dim3(CHAIN_THREADS), 0, stream, chain);
        launch(chain, (unsigned)blocks + 1, false);
        ChainReport h;
        B40C_TRY(wait(h, stream));
        if (h.open) {
            hipLaunchKernelGGL(k_chain_resume, dim3(1), dim3(CHAIN_THREADS), 0, stream, chain);
            B40C_TRY(wait(h, stream));
            ChainMeta meta;
            B40C_HIP(hipMemcpyAsync(&meta, chain.meta, sizeof(meta), hipMemcpyDeviceToHost, stream));
            B40C_HIP(hipStreamSynchronize(stream));
            if (meta.unfinished) launch(chain, meta.unfinished, true);
            ChainReport done;
            B40C_TRY(wait(done, stream));
        }
        total = h.total;
        return B40C_OK;
    }

  private:
    b40c_status wait(ChainReport& h, hipStream_t stream) {
        const hipError_t launched = hipGetLastError();
        if (launched != hipSuccess) (void)hipStreamSynchronize(stream);  // the report and the words are in use until then
        B40C_HIP(launched);
        if (!slot.host) B40C_HIP(hipMemcpyAsync(&h, chain.report, sizeof(h), hipMemcpyDeviceToHost, stream));
        B40C_HIP(hipStreamSynchronize(stream));
        if (slot.host) std::memcpy(&h, slot.host, sizeof(h));
        return B40C_OK;
    }
};
static_assert(sizeof(ChainReport) <= ReportSlot::kBytes, "a report fits its slot");

}  // namespace
}  // namespace b40c
