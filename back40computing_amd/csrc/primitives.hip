// Device primitives next to the CSR build:
//  * consecutive removal — consecutive_removal::Enactor::Trim
//    (b40c/consecutive_removal/enactor.cuh:119-126): the first element of
//    every run of equal keys (and its value), in input order;
//  * prefix sum — scan::Enactor::Scan (b40c/scan/enactor.cuh:122-136),
//    exclusive or inclusive, unsigned 32-bit arithmetic.
// Each is one kernel: a workgroup holds a block of the input in registers and
// waits for the sum of the blocks before it, which one workgroup keeps, so the
// input is read once.  Scans of arrays that are not 16-byte aligned or longer
// than the chain's words can sum (2^30 elements) take three passes over
// contiguous chunks instead: reduce per chunk, one-workgroup spine, ordered
// scan.
#include <climits>

#include "chain.hpp"

namespace b40c {
namespace {

constexpr int PT = CHAIN_THREADS;  // threads per workgroup = elements per tile
constexpr int PW = PT / kWave;

template <typename T>
__device__ __forceinline__ T wave_scan_incl(T x) {
    const int lane = lane_id();
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const T y = __shfl_up(x, d, kWave);
        if (lane >= d) x += y;
    }
    return x;
}

// Workgroup exclusive scan; `total` is the workgroup's sum.
template <typename T>
__device__ __forceinline__ T wg_scan_excl(T x, T& total, T* s_wave) {
    const int wid = threadIdx.x / kWave;
    const T incl = wave_scan_incl(x);
    if (lane_id() == kWave - 1) s_wave[wid] = incl;
    __syncthreads();
    T base = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < PW; ++w) {
        const T t = s_wave[w];
        base += (w < wid) ? t : T(0);
        tot += t;
    }
    __syncthreads();
    total = tot;
    return base + incl - x;
}

// Exclusive scan, in place, of the G per-chunk values (one workgroup);
// *total receives their sum.
__global__ __launch_bounds__(PT) void k_spine_u64(uint64_t* v, int G, uint64_t* total) {
    __shared__ uint64_t s_wave[PW];
    uint64_t carry = 0;
    for (int base = 0; base < G; base += PT) {
        const int i = base + threadIdx.x;
        const uint64_t x = (i < G) ? v[i] : 0;
        uint64_t tot;
        const uint64_t ex = wg_scan_excl<uint64_t>(x, tot, s_wave);
        if (i < G) v[i] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0) *total = carry;
}

__global__ __launch_bounds__(PT) void k_scan_reduce(const uint32_t* in, int64_t n, int64_t chunk, uint64_t* sums) {
    __shared__ uint64_t s_wave[PW];
    const int64_t begin = (int64_t)blockIdx.x * chunk, end = min(n, begin + chunk);
    uint64_t s = 0;
    for (int64_t i = begin + threadIdx.x; i < end; i += PT) s += in[i];
    uint64_t total;
    (void)wg_scan_excl<uint64_t>(s, total, s_wave);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// Each tile's values are in registers before the tile's first barrier, so
// `out` may alias `in`.
__global__ __launch_bounds__(PT) void k_scan_down(const uint32_t* in, uint32_t* out, int64_t n, int64_t chunk,
                                                  const uint64_t* offsets, int inclusive) {
    __shared__ uint32_t s_wave[PW];
    const int64_t begin = (int64_t)blockIdx.x * chunk, end = min(n, begin + chunk);
    uint32_t carry = (uint32_t)offsets[blockIdx.x];
    for (int64_t base = begin; base < end; base += PT) {
        const int64_t i = base + threadIdx.x;
        const uint32_t x = (i < end) ? in[i] : 0u;
        uint32_t tot;
        const uint32_t ex = wg_scan_excl<uint32_t>(x, tot, s_wave);
        if (i < end) out[i] = carry + ex + (inclusive ? x : 0u);
        carry += tot;
    }
}

// ---- vector paths: 16-byte loads, STEP elements per workgroup iteration ----
// A thread owns VEC consecutive elements of each of SUB sub-tiles, so every
// load instruction of a wave covers a contiguous 1 KiB and each thread has
// 64 bytes in flight per iteration; one workgroup scan per sub-tile.
constexpr int VEC32 = 4;                   // uint32 per uint4
constexpr int SUB32 = 4;
constexpr int64_t STEP32 = (int64_t)PT * VEC32 * SUB32;  // 4096 elements

__device__ __forceinline__ void load4_u32(const uint32_t* p, int64_t i, int64_t end, uint32_t (&x)[4]) {
    if (i + 4 <= end) {
        const uint4 q = *reinterpret_cast<const uint4*>(p + i);
        x[0] = q.x, x[1] = q.y, x[2] = q.z, x[3] = q.w;
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = (i + j < end) ? p[i + j] : 0u;
    }
}

__global__ __launch_bounds__(PT) void k_scan_reduce_v(const uint32_t* in, int64_t n, int64_t chunk, uint64_t* sums) {
    __shared__ uint64_t s_wave[PW];
    const int64_t begin = (int64_t)blockIdx.x * chunk, end = min(n, begin + chunk);
    uint64_t s = 0;
    for (int64_t base = begin; base < end; base += STEP32) {
        uint32_t x[SUB32][4];
#pragma unroll
        for (int k = 0; k < SUB32; ++k) load4_u32(in, base + (int64_t)k * PT * VEC32 + threadIdx.x * VEC32, end, x[k]);
#pragma unroll
        for (int k = 0; k < SUB32; ++k) s += (uint64_t)x[k][0] + x[k][1] + x[k][2] + x[k][3];
    }
    uint64_t total;
    (void)wg_scan_excl<uint64_t>(s, total, s_wave);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

__global__ __launch_bounds__(PT) void k_scan_down_v(const uint32_t* in, uint32_t* out, int64_t n, int64_t chunk,
                                                    const uint64_t* offsets, int inclusive) {
    __shared__ uint32_t s_wave[PW];
    const int64_t begin = (int64_t)blockIdx.x * chunk, end = min(n, begin + chunk);
    uint32_t carry = (uint32_t)offsets[blockIdx.x];
    for (int64_t base = begin; base < end; base += STEP32) {
        uint32_t x[SUB32][4];
#pragma unroll
        for (int k = 0; k < SUB32; ++k) load4_u32(in, base + (int64_t)k * PT * VEC32 + threadIdx.x * VEC32, end, x[k]);
#pragma unroll
        for (int k = 0; k < SUB32; ++k) {
            const int64_t i = base + (int64_t)k * PT * VEC32 + threadIdx.x * VEC32;
            uint32_t pre[4], run = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                pre[j] = run + (inclusive ? x[k][j] : 0u);
                run += x[k][j];
            }
            uint32_t tot;
            const uint32_t ex = carry + wg_scan_excl<uint32_t>(run, tot, s_wave);
            if (i + 4 <= end) {
                *reinterpret_cast<uint4*>(out + i) = make_uint4(ex + pre[0], ex + pre[1], ex + pre[2], ex + pre[3]);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (i + j < end) out[i + j] = ex + pre[j];
            }
            carry += tot;
        }
    }
}

// Prefix sum in one pass, bound by its read and its write: 2^26 elements in 113
// us (4.75 TB/s; a large copy reaches 5.3), where a reduce, a spine and a scan took 176.
// A workgroup holds SCAN_SUB sub-tiles of 1,024 elements (a thread four
// consecutive ones of each), so every load and store of a wave covers 1 KiB;
// 4, 12 or 16 sub-tiles measured 114, 117 and 144 us.  Each sub-tile is scanned
// per wave, and one wave scans the waves' totals while another waits for the
// blocks before.  Nothing here reads the output again, so its stores bypass the
// caches (with ordinary stores the reads lose 25 us).  `out` may equal `in`: a
// block is in registers before its first store, and blocks are disjoint.
constexpr int64_t kChainScanMax = 1ll << 30;  // sums of 32-bit values stay below 2^62
constexpr int SCAN_SUB = 8;
constexpr int64_t SCAN_BLOCK = (int64_t)PT * VEC32 * SCAN_SUB;

// Arrays are scanned in segments of at most kScanSegment elements, each after a wait
// for the one before: their chain words stay below 2 MB, which the runtime serves
// from chunks it keeps (8 us after an upload).  More are mapped anew on every call:
// 2^28 elements in place after an upload took 750 to 870 us, in segments 560 to 730,
// as three passes 650 to 730 (2^29 elements in a loop: 996 us in segments, 988 in one
// launch).
constexpr int64_t kScanSegment = (1ll << 28) - (1ll << 20);

template <bool REST>
__global__ __launch_bounds__(PT) void k_scan_chained(const uint32_t* in, uint32_t* out, int64_t n, int inclusive,
                                                     Chain chain) {
    static_assert(SCAN_SUB * PW <= kWave, "one wave scans the waves' totals");
    __shared__ uint32_t s_tot[SCAN_SUB * PW];
    __shared__ uint64_t s_sum[PW];
    __shared__ unsigned long long s_before;
    __shared__ ChainServeShared s_serve;
    if (chain_serves<REST>()) {
        chain_serve(chain, s_serve, chain.before, 0);
        return;
    }
    const int block = chain_block<REST>(chain);
    const int64_t begin = (int64_t)block * SCAN_BLOCK;
    const int tid = threadIdx.x, lane = lane_id(), wid = tid / kWave;
    uint32_t x[SCAN_SUB][4];
#pragma unroll
    for (int k = 0; k < SCAN_SUB; ++k) load4_u32(in, begin + (int64_t)k * PT * VEC32 + tid * VEC32, n, x[k]);
    uint64_t sum = 0;
    uint32_t ex[SCAN_SUB];
#pragma unroll
    for (int k = 0; k < SCAN_SUB; ++k) {
        sum += (uint64_t)x[k][0] + x[k][1] + x[k][2] + x[k][3];
        const uint32_t run = x[k][0] + x[k][1] + x[k][2] + x[k][3];
        const uint32_t incl = wave_scan_incl(run);
        ex[k] = incl - run;
        if (lane == kWave - 1) s_tot[k * PW + wid] = incl;
    }
#pragma unroll
    for (int d = kWave / 2; d >= 1; d >>= 1) sum += __shfl_xor(sum, d, kWave);
    if (lane == 0) s_sum[wid] = sum;
    __syncthreads();
    if (wid == 0) {
        uint64_t mine = 0;
#pragma unroll
        for (int w = 0; w < PW; ++w) mine += s_sum[w];
        if (lane == 0) s_before = chain_before<REST>(chain, block, mine);
    } else if (wid == 1) {
        const uint32_t t = lane < SCAN_SUB * PW ? s_tot[lane] : 0u;
        const uint32_t incl = wave_scan_incl(t);
        if (lane < SCAN_SUB * PW) s_tot[lane] = incl - t;
    }
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane((int)(s_before >> 32)) == 0) return;  // (a set word has its top bit)
    const uint32_t before = (uint32_t)s_before;
#pragma unroll
    for (int k = 0; k < SCAN_SUB; ++k) {
        const int64_t i = begin + (int64_t)k * PT * VEC32 + tid * VEC32;
        uint32_t run = before + s_tot[k * PW + wid] + ex[k];
        uint32_t y[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            y[j] = run + (inclusive ? x[k][j] : 0u);
            run += x[k][j];
        }
        if (i + 4 <= n) {
            typedef uint32_t vec4 __attribute__((ext_vector_type(4)));
            __builtin_nontemporal_store(vec4{y[0], y[1], y[2], y[3]}, reinterpret_cast<vec4*>(out + i));
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (i + j < n) out[i + j] = y[j];
        }
    }
}

// Run heads in one pass, bound by its reads and writes: 2^25 pairs, half of them
// kept, in 118 us (4.9 TB/s), where a count, a spine and a scatter took 235.  A
// wave holds TRIM_ITEMS rows of 64 consecutive keys (and values), so that every
// load, and every store of a row's kept entries, covers consecutive entries;
// four consecutive keys per thread scattered the stores (161 us).  8 or 32 rows
// measured 141 and 129 us.
constexpr int TRIM_ITEMS = 16;
constexpr int64_t TRIM_BLOCK = (int64_t)PT * TRIM_ITEMS;

template <bool VALS, bool REST>
__global__ __launch_bounds__(PT) void k_trim_chained(const uint64_t* keys, const uint32_t* vals, int64_t n,
                                                     uint64_t* keys_out, uint32_t* vals_out,
                                                     Chain chain) {
    __shared__ uint32_t s_tot[PW];
    __shared__ unsigned long long s_before;
    __shared__ ChainServeShared s_serve;
    if (chain_serves<REST>()) {
        chain_serve(chain, s_serve, chain.before, 0);
        return;
    }
    const int block = chain_block<REST>(chain);
    const int lane = lane_id(), wid = threadIdx.x / kWave;
    const int64_t begin = (int64_t)block * TRIM_BLOCK + (int64_t)wid * kWave * TRIM_ITEMS;
    uint64_t x[TRIM_ITEMS];
    uint32_t v[TRIM_ITEMS];
    uint64_t last = 0;  // the key before the row; lane 0
    if (lane == 0 && begin > 0 && begin < n) last = keys[begin - 1];
#pragma unroll
    for (int k = 0; k < TRIM_ITEMS; ++k) {
        const int64_t i = begin + k * kWave + lane;
        x[k] = i < n ? keys[i] : 0ull;
        if (VALS) v[k] = i < n ? vals[i] : 0u;
    }
    uint64_t heads[TRIM_ITEMS];
    uint32_t count = 0;
#pragma unroll
    for (int k = 0; k < TRIM_ITEMS; ++k) {
        const int64_t i = begin + k * kWave + lane;
        const uint64_t left = __shfl_up(x[k], 1, kWave);
        const uint64_t prev = lane == 0 ? last : left;
        heads[k] = __ballot(i < n && (i == 0 || x[k] != prev));
        count += (uint32_t)__popcll(heads[k]);
        last = __shfl(x[k], kWave - 1, kWave);
    }
    if (lane == 0) s_tot[wid] = count;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint64_t mine = 0;
#pragma unroll
        for (int w = 0; w < PW; ++w) {
            const uint32_t t = s_tot[w];
            s_tot[w] = (uint32_t)mine;
            mine += t;
        }
        s_before = chain_before<REST>(chain, block, mine);
    }
    __syncthreads();
    if (!s_before) return;
    uint64_t pos = (s_before & CHAIN_VALUE) + s_tot[wid];
#pragma unroll
    for (int k = 0; k < TRIM_ITEMS; ++k) {
        if ((heads[k] >> lane) & 1u) {
            const uint64_t at = pos + __popcll(heads[k] & ((1ull << lane) - 1));
            keys_out[at] = x[k];
            if (VALS) vals_out[at] = v[k];
        }
        pos += (uint64_t)__popcll(heads[k]);
    }
}

inline bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

// Contiguous chunks of whole `step`-element iterations, at most 8 per CU.
void chunking(int64_t n, int64_t step, int64_t& chunk, int& G) {
    DeviceInfo info;
    const int cus = (device_info(info) == B40C_OK) ? info.num_cus : 256;
    const int64_t steps = (n + step - 1) / step;
    const int64_t g = std::max<int64_t>(1, std::min<int64_t>(steps, (int64_t)cus * 8));
    chunk = (steps + g - 1) / g * step;
    G = (int)((n + chunk - 1) / chunk);
    if (G < 1) G = 1;
}


}  // namespace

int scan_u32_max_partials() {
    DeviceInfo info;
    const int cus = (device_info(info) == B40C_OK) ? info.num_cus : 256;
    return cus * 8;
}

b40c_status scan_u32_async(const uint32_t* in, uint32_t* out, int64_t n, bool exclusive, uint64_t* partials,
                           uint64_t* total, hipStream_t stream) {
    if (n <= 0) return B40C_OK;
    const bool vec = aligned16(in) && aligned16(out);
    int64_t chunk;
    int G;
    chunking(n, vec ? STEP32 : PT, chunk, G);
    if (vec)
        hipLaunchKernelGGL(k_scan_reduce_v, dim3(G), dim3(PT), 0, stream, in, n, chunk, partials);
    else
        hipLaunchKernelGGL(k_scan_reduce, dim3(G), dim3(PT), 0, stream, in, n, chunk, partials);
    hipLaunchKernelGGL(k_spine_u64, dim3(1), dim3(PT), 0, stream, partials, G, total);
    if (vec)
        hipLaunchKernelGGL(k_scan_down_v, dim3(G), dim3(PT), 0, stream, in, out, n, chunk, partials,
                           exclusive ? 0 : 1);
    else
        hipLaunchKernelGGL(k_scan_down, dim3(G), dim3(PT), 0, stream, in, out, n, chunk, partials,
                           exclusive ? 0 : 1);
    B40C_HIP(hipGetLastError());
    return B40C_OK;
}

}  // namespace b40c

using b40c::fail;

extern "C" {

b40c_status b40c_consecutive_removal_u64(const uint64_t* d_keys_in, const uint32_t* d_values_in,
                                         uint64_t* d_keys_out, uint32_t* d_values_out, int64_t n,
                                         int64_t* num_compacted) {
    using namespace b40c;
    if (n < 0 || !num_compacted || (n > 0 && (!d_keys_in || !d_keys_out)) || (!d_values_in != !d_values_out))
        return fail(B40C_ERR_INVALID_ARG, "b40c_consecutive_removal_u64: bad arguments");
    if (n > 0 && (d_keys_in == d_keys_out || (d_values_in && d_values_in == d_values_out)))
        return fail(B40C_ERR_INVALID_ARG, "b40c_consecutive_removal_u64: output must not alias input");
    *num_compacted = 0;
    if (n == 0) return B40C_OK;
    const int64_t blocks = (n + TRIM_BLOCK - 1) / TRIM_BLOCK;
    if (blocks >= INT32_MAX) return fail(B40C_ERR_INVALID_ARG, "b40c_consecutive_removal_u64: n out of range");
    ChainCall call;
    B40C_TRY(call.start(blocks, nullptr));
    uint64_t total = 0;
    B40C_TRY(call.run(blocks, 0, total, nullptr, [&](const Chain& chain, unsigned wgs, bool rest) {
        auto* kernel = d_values_in ? (rest ? k_trim_chained<true, true> : k_trim_chained<true, false>)
                                   : (rest ? k_trim_chained<false, true> : k_trim_chained<false, false>);
        hipLaunchKernelGGL(kernel, dim3(wgs), dim3(PT), 0, nullptr, d_keys_in, d_values_in, n, d_keys_out,
                           d_values_out, chain);
    }));
    *num_compacted = (int64_t)total;
    return B40C_OK;
}

b40c_status b40c_scan_u32(const uint32_t* d_in, uint32_t* d_out, int64_t n, int32_t exclusive, uint64_t* total) {
    using namespace b40c;
    if (n < 0 || (n > 0 && (!d_in || !d_out)))
        return fail(B40C_ERR_INVALID_ARG, "b40c_scan_u32: bad arguments");
    if (total) *total = 0;
    if (n == 0) return B40C_OK;
    if (aligned16(d_in) && aligned16(d_out) && n <= kChainScanMax) {
        ChainCall call;
        B40C_TRY(call.start((std::min<int64_t>(n, kScanSegment) + SCAN_BLOCK - 1) / SCAN_BLOCK, nullptr));
        uint64_t sum = 0;
        for (int64_t at = 0; at < n; at += kScanSegment) {
            const int64_t len = std::min<int64_t>(n - at, kScanSegment);
            B40C_TRY(call.run((len + SCAN_BLOCK - 1) / SCAN_BLOCK, sum, sum, nullptr,
                              [&](const Chain& chain, unsigned wgs, bool rest) {
                                  hipLaunchKernelGGL(rest ? k_scan_chained<true> : k_scan_chained<false>, dim3(wgs),
                                                     dim3(PT), 0, nullptr, d_in + at, d_out + at, len,
                                                     exclusive ? 0 : 1, chain);
                              }));
        }
        if (total) *total = sum;
        return B40C_OK;
    }
    DeviceBuffer sums, tot;
    B40C_TRY(sums.alloc((size_t)scan_u32_max_partials() * 8));
    B40C_TRY(tot.alloc(8));
    B40C_TRY(scan_u32_async(d_in, d_out, n, exclusive != 0, sums.as<uint64_t>(), tot.as<uint64_t>(), nullptr));
    uint64_t h = 0;
    B40C_HIP(hipMemcpy(&h, tot.ptr, 8, hipMemcpyDeviceToHost));
    if (total) *total = h;
    return B40C_OK;
}

}  // extern "C"
