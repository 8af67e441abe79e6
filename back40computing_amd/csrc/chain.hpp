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
constexpr uint32_t kChainSpins = 1u << 22;

// Report of a chained call.
struct ChainReport {
    uint64_t total;
    uint32_t failed;
};

__device__ __forceinline__ unsigned long long chain_load(const unsigned long long* chain, int b) {
    return __hip_atomic_load(&chain[(size_t)b * CHAIN_STRIDE], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void chain_store(unsigned long long* chain, int b, unsigned long long w) {
    __hip_atomic_store(&chain[(size_t)b * CHAIN_STRIDE], w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ __launch_bounds__(CHAIN_THREADS) void k_chain_init(unsigned long long* chain, int blocks) {
    for (int i = blockIdx.x * CHAIN_THREADS + threadIdx.x; i < blocks; i += gridDim.x * CHAIN_THREADS) chain[(size_t)i * CHAIN_STRIDE] = 0;
}

struct ChainServeShared {
    uint64_t sum[CHAIN_WAVES];
    uint32_t ready[CHAIN_WAVES];
};

// Workgroup 0 of a chained kernel: turns the blocks' sums into prefixes, up to
// 256 of them per round trip (0.7 us), and reports the total.  The blocks poll one
// line each; when every block looked back over its predecessors' words itself,
// the polling alone took 20 to 45 us of a scan of 2^26 elements.  Workgroups
// are dispatched in order, so the lowest block without a sum is running or
// next to run; should that fail, the bounded wait sets failed and the
// remaining blocks go on with what there is.
// `before` is what comes before the first block.
__device__ __forceinline__ void chain_serve(unsigned long long* chain, int blocks, ChainReport* report,
                                            ChainServeShared& s, uint64_t before = 0) {
    const int tid = threadIdx.x, lane = lane_id(), wid = tid / kWave;
    int base = 0;
    uint32_t spins = 0;
    while (base < blocks) {
        const int b = base + tid;
        const unsigned long long w = b < blocks ? chain_load(chain, b) : 0ull;
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
            if (k == wid && open && lane < ready) chain_store(chain, b, CHAIN_PREFIX | (mine + incl - v));
            if (open) {
                mine += s.sum[k];
                taken += (int)s.ready[k];
                open = s.ready[k] == kWave;
            }
        }
        __syncthreads();
        before = mine;
        base += taken;
        if (taken == 0 && base < blocks) {
            if (++spins > kChainSpins) {
                if (tid == 0) report->failed = 1;
                for (int i = base + tid; i < blocks; i += CHAIN_THREADS) chain_store(chain, i, CHAIN_PREFIX | before);
                return;
            }
            __builtin_amdgcn_s_sleep(1);
        }
    }
    if (tid == 0) report->total = before;
}

// Sum of the blocks before `block`, which publishes `mine`; one lane.
__device__ __forceinline__ uint64_t chain_before(unsigned long long* chain, int block, uint64_t mine,
                                                 ChainReport* report) {
    chain_store(chain, block, CHAIN_SUM | mine);
    unsigned long long w;
    uint32_t spins = 0;
    while ((w = chain_load(chain, block)) < CHAIN_PREFIX) {
        if (++spins > kChainSpins) {
            report->failed = 1;
            return 0;
        }
        __builtin_amdgcn_s_sleep(1);
    }
    return w & CHAIN_VALUE;
}

// Chained calls: chain words, then a report for when there is no pinned slot.
inline size_t chain_bytes(int64_t blocks) { return (size_t)blocks * CHAIN_STRIDE * 8 + sizeof(ChainReport); }

// One chained call's scratch and report.
struct ChainCall {
    ReportSlot slot;
    DeviceBuffer mem;  // freed before the slot is given back
    unsigned long long* chain = nullptr;
    ChainReport* report = nullptr;
    // `words`: chain_bytes(blocks) of the caller's device memory, or null to allocate them.
    b40c_status start(int64_t blocks, hipStream_t stream, void* words = nullptr) {
        if (!words) B40C_TRY(mem.alloc(chain_bytes(blocks)));
        chain = static_cast<unsigned long long*>(words ? words : mem.ptr);
        report = reinterpret_cast<ChainReport*>(chain + (size_t)blocks * CHAIN_STRIDE);
        if (slot.take())
            report = static_cast<ChainReport*>(slot.dev);
        else
            B40C_TRY(fill_u32(reinterpret_cast<uint32_t*>(report), 0, sizeof(ChainReport) / 4, stream));
        clear(blocks, stream);
        return B40C_OK;
    }
    // The words of a kernel's blocks; before every kernel of the call.
    void clear(int64_t blocks, hipStream_t stream) {
        hipLaunchKernelGGL(k_chain_init, dim3((unsigned)std::min<int64_t>((blocks + CHAIN_THREADS - 1) / CHAIN_THREADS, 256)), dim3(CHAIN_THREADS), 0,
                           stream, chain, (int)blocks);
    }
    b40c_status finish(const char* who, uint64_t& total, hipStream_t stream) {
        const hipError_t launched = hipGetLastError();
        if (launched != hipSuccess) (void)hipStreamSynchronize(stream);  // the report and `words` are in use until then
        B40C_HIP(launched);
        ChainReport h;
        if (!slot.host) B40C_HIP(hipMemcpyAsync(&h, report, sizeof(h), hipMemcpyDeviceToHost, stream));
        B40C_HIP(hipStreamSynchronize(stream));
        if (slot.host) std::memcpy(&h, slot.host, sizeof(h));
        if (h.failed) return fail(B40C_ERR_HIP, "%s: a block waited too long for the blocks before it", who);
        total = h.total;
        return B40C_OK;
    }
};
static_assert(sizeof(ChainReport) <= ReportSlot::kBytes, "a report fits its slot");

}  // namespace
}  // namespace b40c
