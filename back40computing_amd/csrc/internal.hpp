// Internal host-side declarations shared by the library's translation units.
#pragma once

#include <atomic>

#include "common.hpp"

namespace b40c {

// Owning device allocation (hipMalloc / hipFree).
struct DeviceBuffer {
    void* ptr = nullptr;
    size_t bytes = 0;
    DeviceBuffer() = default;
    DeviceBuffer(const DeviceBuffer&) = delete;
    DeviceBuffer& operator=(const DeviceBuffer&) = delete;
    ~DeviceBuffer() { release(); }
    b40c_status alloc(size_t n) {
        release();
        if (n == 0) n = 1;
        hipError_t e = hipMalloc(&ptr, n);
        if (e != hipSuccess) {
            ptr = nullptr;
            return fail(e == hipErrorOutOfMemory ? B40C_ERR_OOM : B40C_ERR_HIP, "hipMalloc(%zu) failed: %s", n,
                        hipGetErrorString(e));
        }
        bytes = n;
        return B40C_OK;
    }
    // Grow-only reallocation (contents are not preserved).
    b40c_status reserve(size_t n) { return (n <= bytes && ptr) ? B40C_OK : alloc(n); }
    void release() {
        if (ptr) (void)hipFree(ptr);
        ptr = nullptr;
        bytes = 0;
    }
    template <typename T>
    T* as() const { return static_cast<T*>(ptr); }
};

// runtime.hip.  A call's report: a few pinned host words that its kernels
// write and the host reads after one stream synchronization, in place of a copy
// (about 10 us).  One page of slots per process, held until it ends; take()
// is false when the page could not be had or every slot is in use.
struct ReportSlot {
    void* host = nullptr;  // kBytes bytes, zeroed by take()
    void* dev = nullptr;   // the same words as kernels address them
    static constexpr size_t kBytes = 64;
    ReportSlot() = default;
    ReportSlot(const ReportSlot&) = delete;
    ReportSlot& operator=(const ReportSlot&) = delete;
    ~ReportSlot();
    bool take();
};

// radix_sort.hip.  A sort's device scratch: one block of `words` uint32 words.
struct SortScratch {
    uint32_t* base = nullptr;
    size_t words = 0;
};
// A sort's launch policy (the reference's per-architecture KernelPolicy /
// AutotunedPolicy, radix_sort/autotuned_policy.cuh:190-230, chosen at run
// time): keys per thread of a tile (8 or 16; a tile is 512 x that) and
// workgroups per CU (1-8).  Zero fields take the size-based default.
struct SortPolicy {
    int items = 0;
    int wgs_per_cu = 0;
};
// Policy with its zero fields filled in for n keys (with their values
// pair_bytes bytes each).
SortPolicy resolve_sort_policy(SortPolicy p, int64_t n, int pair_bytes, int num_cus);
// Words of scratch a sort of n keys wants.
size_t sort_scratch_words(int64_t n);
// With `scratch` null, or less than sort_scratch_words(n), it is allocated for the call.
b40c_status radix_sort_u64(uint64_t* k0, uint64_t* k1, int64_t n, int begin_bit, int end_bit, int32_t* selector,
                           hipStream_t stream, uint32_t* scratch = nullptr, size_t scratch_words = 0);
b40c_status radix_sort_pairs_u32(uint32_t* k0, uint32_t* k1, uint32_t* v0, uint32_t* v1, int64_t n, int begin_bit,
                                 int end_bit, int32_t* selector, hipStream_t stream);

// primitives.hip: prefix scan of uint32 on `stream` with caller-provided
// scratch (`partials`: scan_u32_max_partials() entries; `total`: the exact sum).
int scan_u32_max_partials();
b40c_status scan_u32_async(const uint32_t* in, uint32_t* out, int64_t n, bool exclusive, uint64_t* partials,
                           uint64_t* total, hipStream_t stream);

}  // namespace b40c

// Device-resident CSR graph (reference counted).
struct b40c_graph {
    int32_t nodes = 0;
    int64_t edges = 0;
    b40c::DeviceBuffer offsets;  // int32[nodes + 1]
    b40c::DeviceBuffer cols;     // int32[edges]
    std::atomic<int> refs{1};
    // 1: every edge (u,v) has its reverse (v,u); 0: not (or not provable);
    // -1: not yet checked.  Bottom-up BFS steps are only valid when 1.
    std::atomic<int> symmetric{-1};
    // Largest out-degree, or -1 while not yet computed (graph_max_degree).
    std::atomic<int> max_degree{-1};
    const int32_t* d_offsets() const { return offsets.as<int32_t>(); }
    const int32_t* d_cols() const { return cols.as<int32_t>(); }
};

namespace b40c {
void graph_retain(b40c_graph* g);
void graph_release(b40c_graph* g);
// Resolves g->symmetric (runs a GPU check the first time it is unknown).
b40c_status graph_symmetric(b40c_graph* g, bool& symmetric);
b40c_status graph_max_degree(b40c_graph* g, int32_t& max_degree);
}  // namespace b40c
