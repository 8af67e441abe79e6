// Host build of the library (test infrastructure only).
//
// Stands in for <hip/hip_runtime.h> when the library's sources (csrc/*.hip) are
// compiled for the host: kernels, launches, streams, captured graphs and
// allocations all run on the CPU, so the library's own C entry points can be
// driven end to end under AddressSanitizer.
//
//  * A workgroup is one host thread and its lanes are fibers on it, switched
//    at every wave collective, workgroup barrier and s_sleep; between those a
//    wave is not in lockstep.  __shared__ is
//    `static thread_local`: one copy per workgroup, and the host threads are
//    kept, so LDS starts with what an earlier kernel left there.
//  * Workgroups start in order, at most emu::dev().resident at a time.
//  * Device allocations are host allocations of exactly the asked size, filled
//    with garbage.
//  * Launches run at once, or, with emu::dev().lazy, when something waits for
//    them.  A memset in a captured graph ends the program: the library keeps
//    those out of its graphs.
//  * Tests set the device's size, occupancies, limits and errors in emu::dev().
#pragma once

#include <sched.h>
#include <sys/mman.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <tuple>
#include <type_traits>
#include <utility>
#include <vector>

#include <sanitizer/asan_interface.h>
#include <sanitizer/common_interface_defs.h>

#define __device__
#define __host__
#define __global__
#define __shared__ static thread_local
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __align__(n) __attribute__((aligned(n)))

struct int2 {
    int x, y;
};
inline int2 make_int2(int x, int y) { return int2{x, y}; }
struct alignas(16) uint4 {
    uint32_t x, y, z, w;
};
inline uint4 make_uint4(uint32_t x, uint32_t y, uint32_t z, uint32_t w) { return uint4{x, y, z, w}; }
struct alignas(16) int4 {
    int32_t x, y, z, w;
};
inline int4 make_int4(int32_t x, int32_t y, int32_t z, int32_t w) { return int4{x, y, z, w}; }
struct alignas(8) uint2 {
    uint32_t x, y;
};
struct alignas(16) ulonglong2 {
    unsigned long long x, y;
};
struct dim3 {
    uint32_t x, y, z;
    dim3(uint32_t a = 1, uint32_t b = 1, uint32_t c = 1) : x(a), y(b), z(c) {}
};

template <class A, class B>
inline typename std::common_type<A, B>::type min(A a, B b) {
    return a < b ? a : b;
}
template <class A, class B>
inline typename std::common_type<A, B>::type max(A a, B b) {
    return a > b ? a : b;
}

typedef int hipError_t;
enum { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };

// ---------------------------------------------------------------------------
// Lanes, waves, workgroups.
// ---------------------------------------------------------------------------
extern "C" void emu_switch(void** save, void* load);

namespace emu {

struct Device {
    int cus = 4;
    unsigned resident = 64;             // workgroups running at a time
    int occupancy = 8;                  // workgroups per CU of a kernel not named below
    std::map<std::string, int> occupancies;
    size_t largest_alloc = ~(size_t)0;  // larger device allocations fail
    bool lazy = false;
    unsigned chain_spins = 1u << 14;    // polls of a bounded wait
    int label_claim_nodes = 1 << 20;
    long long scan_segment = 1 << 27;   // elements of a scan's launch
    // Called as a workgroup starts (kernel's name, workgroup); may wait.
    std::function<void(const std::string&, unsigned)> on_start;
    std::function<void(const std::string&, unsigned)> on_end;
    std::vector<std::pair<std::string, unsigned>> launches;  // persistent launches: kernel, grid
};
inline Device& dev() {
    static Device d;
    return d;
}

enum State { RUN, WAIT_WAVE, WAIT_MEET, WAIT_BLOCK, YIELD, DONE };
struct Block;
struct Wave {
    uint64_t x[2][64];
    uint64_t mask[2] = {0, 0};
    int live = 0, arrived = 0;
    int met = 0;  // lanes at the wave barrier
    uint64_t gen = 0;
};
struct Lane {
    dim3 tid, bid, bdim, gdim;
    int lane = 0;
    Wave* wave = nullptr;
    Block* block = nullptr;
    State state = RUN;
    void* sp = nullptr;
    char* stack = nullptr;
};
struct Block {
    std::vector<Lane> lanes;
    std::vector<Wave> waves;
    int live = 0, arrived = 0;
    int acc[2] = {0, 0};
    uint64_t gen = 0;
    void* sched_sp = nullptr;
    const void* sched_bottom = nullptr;
    size_t sched_size = 0;
    const std::function<void()>* body = nullptr;
};
inline thread_local Lane* cur = nullptr;
constexpr size_t kStack = 96 << 10;

// Out of the current lane, back to its workgroup's scheduler.
inline void leave(bool last = false) {
    Lane& l = *cur;
    Block& b = *l.block;
    void* fake = nullptr;
    __sanitizer_start_switch_fiber(last ? nullptr : &fake, b.sched_bottom, b.sched_size);
    emu_switch(&l.sp, b.sched_sp);
    __sanitizer_finish_switch_fiber(fake, nullptr, nullptr);
}
inline void enter(Block& b, Lane& l) {
    cur = &l;
    void* fake = nullptr;
    __sanitizer_start_switch_fiber(&fake, l.stack, kStack);
    emu_switch(&b.sched_sp, l.sp);
    __sanitizer_finish_switch_fiber(fake, nullptr, nullptr);
    cur = nullptr;
}
inline void let_go(Block& b, Wave& w, State from) {
    const size_t first = (size_t)(&w - b.waves.data()) * 64;
    for (size_t i = first; i < first + 64 && i < b.lanes.size(); ++i)
        if (b.lanes[i].state == from) b.lanes[i].state = RUN;
}
inline void release_wave(Block& b, Wave& w) {
    w.arrived = 0;
    ++w.gen;
    w.mask[w.gen & 1] = 0;
    let_go(b, w, WAIT_WAVE);
}
inline void release_meeting(Block& b, Wave& w) {
    w.met = 0;
    let_go(b, w, WAIT_MEET);
}
inline void release_block(Block& b) {
    b.arrived = 0;
    ++b.gen;
    b.acc[b.gen & 1] = 0;
    for (Lane& l : b.lanes)
        if (l.state == WAIT_BLOCK) l.state = RUN;
}
// Every lane of the wave that has not ended publishes a value; returns the
// wave's values and which lanes took part.
inline const uint64_t* wave_exchange(uint64_t v, uint64_t* mask = nullptr) {
    Lane& l = *cur;
    Wave& w = *l.wave;
    const int k = (int)(w.gen & 1);
    w.x[k][l.lane] = v;
    w.mask[k] |= 1ull << l.lane;
    if (++w.arrived == w.live) {
        release_wave(*l.block, w);
    } else {
        l.state = WAIT_WAVE;
        leave();
    }
    if (mask) *mask = w.mask[k];
    return w.x[k];
}
// Wave barrier: where the groups of a wave meet again.
inline void wave_meet() {
    Lane& l = *cur;
    Wave& w = *l.wave;
    if (++w.met == w.live) {
        release_meeting(*l.block, w);
    } else {
        l.state = WAIT_MEET;
        leave();
    }
}
inline int block_op(int v) {
    Lane& l = *cur;
    Block& b = *l.block;
    const int k = (int)(b.gen & 1);
    if (v) b.acc[k] = 1;
    if (++b.arrived == b.live) {
        release_block(b);
    } else {
        l.state = WAIT_BLOCK;
        leave();
    }
    return b.acc[k];
}
inline void yield() {
    cur->state = YIELD;
    leave();
}

inline void lane_main() {
    __sanitizer_finish_switch_fiber(nullptr, &cur->block->sched_bottom, &cur->block->sched_size);
    (*cur->block->body)();
    Lane& l = *cur;
    l.state = DONE;
    Wave& w = *l.wave;
    Block& b = *l.block;
    --w.live;
    --b.live;
    if (w.arrived && w.arrived == w.live) release_wave(b, w);
    if (w.met && w.met == w.live) release_meeting(b, w);
    if (b.arrived && b.arrived == b.live) release_block(b);
    leave(true);
    std::abort();
}

template <class T>
inline uint64_t bits_of(T v) {
    static_assert(sizeof(T) <= 8, "shuffle of a wide type");
    uint64_t u = 0;
    std::memcpy(&u, &v, sizeof(T));
    return u;
}
template <class T>
inline T from_bits(uint64_t u) {
    T v;
    std::memcpy(&v, &u, sizeof(T));
    return v;
}

// A host thread that runs workgroups; keeps its lanes' stacks and its LDS.
struct Stacks {
    char* mem = nullptr;
    size_t lanes = 0;
    char* at(size_t i, size_t want) {
        if (want > lanes) {
            if (mem) munmap(mem, lanes * kStack);
            mem = (char*)mmap(nullptr, want * kStack, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
            if (mem == MAP_FAILED) std::abort();
            lanes = want;
        }
        return mem + i * kStack;
    }
    ~Stacks() {
        if (mem) munmap(mem, lanes * kStack);
    }
};

struct Launch {
    std::string name;
    dim3 grid, block;
    std::function<void()> body;
};

inline void run_block(const Launch& job, unsigned id) {
    static thread_local Stacks stacks;
    static thread_local Block b;
    const unsigned threads = job.block.x;
    if (threads % 64) {
        std::fprintf(stderr, "host build: %s: %u threads is not a whole number of waves\n", job.name.c_str(), threads);
        std::abort();
    }
    b.lanes.assign(threads, Lane());
    b.waves.assign(threads / 64, Wave());
    b.live = (int)threads;
    b.arrived = 0;
    b.gen = 0;
    b.acc[0] = b.acc[1] = 0;
    b.body = &job.body;
    for (Wave& w : b.waves) w.live = 64;
    for (unsigned t = 0; t < threads; ++t) {
        Lane& l = b.lanes[t];
        l.tid = dim3(t, 0, 0);
        l.bid = dim3(id % job.grid.x, id / job.grid.x, 0);
        l.bdim = job.block;
        l.gdim = job.grid;
        l.lane = (int)(t % 64);
        l.wave = &b.waves[t / 64];
        l.block = &b;
        l.stack = stacks.at(t, threads);
        // An ended lane left lane_main's frame behind.
        __asan_unpoison_memory_region(l.stack + kStack - 4096, 4096);
        // The frame emu_switch pops: six registers, then its return address.
        // At lane_main's entry the stack must be 8 past a multiple of 16.
        void** top = (void**)(l.stack + kStack - 64);
        *--top = nullptr;
        *--top = (void*)&lane_main;
        for (int r = 0; r < 6; ++r) *--top = nullptr;
        l.sp = top;
    }
    if (dev().on_start) dev().on_start(job.name, id);
    auto since = std::chrono::steady_clock::now();
    while (b.live > 0) {
        bool ran = false, progress = false;
        for (Lane& l : b.lanes) {
            if (l.state != RUN && l.state != YIELD) continue;
            l.state = RUN;
            enter(b, l);
            ran = true;
            progress |= l.state != YIELD;
        }
        if (progress) {
            since = std::chrono::steady_clock::now();
            continue;
        }
        // Groups of a wave's lanes may leave a loop of collectives early and
        // wait at a barrier: the others go on without them.
        for (Wave& w : b.waves)
            if (!ran && w.arrived) {
                release_wave(b, w);
                progress = true;
            }
        if (progress) continue;
        if (!ran) {
            std::fprintf(stderr, "host build: %s: workgroup %u: no lane can go on (a collective reached by part of a wave or workgroup)\n",
                         job.name.c_str(), id);
            std::abort();
        }
        sched_yield();
        if (std::chrono::steady_clock::now() - since > std::chrono::seconds(60)) {
            std::fprintf(stderr, "host build: %s: workgroup %u waits for ever\n", job.name.c_str(), id);
            std::abort();
        }
    }
    if (dev().on_end) dev().on_end(job.name, id);
}

class Pool {
  public:
    static Pool& get() {
        static Pool* p = new Pool();  // never destroyed: its threads outlive main's statics
        return *p;
    }
    void run(const Launch& job) {
        std::lock_guard<std::mutex> one(run_mu_);
        const unsigned total = job.grid.x * job.grid.y;
        const unsigned want = std::min(std::max(1u, dev().resident), total);
        std::unique_lock<std::mutex> lk(mu_);
        while (threads_.size() < want) {
            const unsigned me = (unsigned)threads_.size();
            threads_.emplace_back([this, me] { work(me); });
        }
        job_ = &job;
        next_ = 0;
        total_ = total;
        active_ = want;
        busy_ = want;
        ++gen_;
        wake_.notify_all();
        done_.wait(lk, [&] { return busy_ == 0; });
        job_ = nullptr;
    }

  private:
    void work(unsigned me) {
        uint64_t seen = 0;
        std::unique_lock<std::mutex> lk(mu_);
        while (true) {
            wake_.wait(lk, [&] { return gen_ != seen && me < active_ && job_; });
            seen = gen_;
            const Launch* job = job_;
            while (next_ < total_) {
                const unsigned id = next_++;
                lk.unlock();
                run_block(*job, id);
                lk.lock();
            }
            if (--busy_ == 0) done_.notify_all();
        }
    }
    std::mutex run_mu_, mu_;
    std::condition_variable wake_, done_;
    std::vector<std::thread> threads_;
    const Launch* job_ = nullptr;
    unsigned next_ = 0, total_ = 0, active_ = 0, busy_ = 0;
    uint64_t gen_ = 0;
};

// ---------------------------------------------------------------------------
// Streams, captured graphs, errors.
// ---------------------------------------------------------------------------
struct Stream {
    bool capturing = false;
    std::vector<std::function<void()>> recorded;
    std::deque<std::function<void()>> pending;
};
struct Graph {
    std::vector<std::function<void()>> nodes;
};
inline Stream& null_stream() {
    static Stream s;
    return s;
}
inline std::recursive_mutex& api_mu() {
    static std::recursive_mutex m;
    return m;
}
inline std::vector<Stream*>& streams() {
    static std::vector<Stream*> v{&null_stream()};
    return v;
}
inline void drain(Stream* s) {
    std::lock_guard<std::recursive_mutex> lk(api_mu());
    while (!s->pending.empty()) {
        auto f = std::move(s->pending.front());
        s->pending.pop_front();
        f();
    }
}
// What a wait on `first` lets run: its work, then everybody else's.
inline void drain_all(Stream* first = nullptr) {
    std::lock_guard<std::recursive_mutex> lk(api_mu());
    if (first) drain(first);
    for (Stream* s : streams()) drain(s);
}
inline void enqueue(Stream* s, std::function<void()> f) {
    std::lock_guard<std::recursive_mutex> lk(api_mu());
    if (!s) s = &null_stream();
    if (s->capturing)
        s->recorded.push_back(std::move(f));
    else if (dev().lazy)
        s->pending.push_back(std::move(f));
    else
        f();
}
inline thread_local hipError_t last_error = hipSuccess;
inline hipError_t set(hipError_t e) {
    if (e != hipSuccess) last_error = e;
    return e;
}

// Kernels launched through hipLaunchKernel, or that a test names.
struct Kernel {
    std::string name;
    std::function<std::function<void()>(void**)> bind;
};
inline std::map<const void*, Kernel>& kernels() {
    static std::map<const void*, Kernel> m;
    return m;
}
template <class... P, size_t... I>
std::function<void()> bind_args(void (*k)(P...), void** a, std::index_sequence<I...>) {
    std::tuple<std::decay_t<P>...> t{*static_cast<std::decay_t<P>*>(a[I])...};
    return [k, t] { std::apply(k, t); };
}
template <class... P>
bool name_kernel(const char* name, void (*k)(P...)) {
    kernels()[(const void*)k] =
        Kernel{name, [k](void** a) { return bind_args(k, a, std::index_sequence_for<P...>{}); }};
    return true;
}
inline std::string name_of(const void* k) {
    auto it = kernels().find(k);
    return it == kernels().end() ? std::string("kernel") : it->second.name;
}
inline int occupancy_of(const void* k) {
    auto it = dev().occupancies.find(name_of(k));
    return it == dev().occupancies.end() ? dev().occupancy : it->second;
}
template <class... P, class... A>
void launch(const char* text, void (*k)(P...), dim3 grid, dim3 block, Stream* s, A&&... a) {
    std::tuple<std::decay_t<P>...> t{static_cast<std::decay_t<P>>(a)...};
    auto named = kernels().find((const void*)k);
    Launch job{named == kernels().end() ? text : named->second.name, grid, block, [k, t] { std::apply(k, t); }};
    enqueue(s, [job] { Pool::get().run(job); });
}

template <class T>
inline T fetch_max(T* p, T v) {
    T c = __atomic_load_n(p, __ATOMIC_SEQ_CST);
    while (c < v && !__atomic_compare_exchange_n(p, &c, v, false, __ATOMIC_SEQ_CST, __ATOMIC_SEQ_CST)) {
    }
    return c;
}
template <class T>
inline T fetch_min(T* p, T v) {
    T c = __atomic_load_n(p, __ATOMIC_SEQ_CST);
    while (c > v && !__atomic_compare_exchange_n(p, &c, v, false, __ATOMIC_SEQ_CST, __ATOMIC_SEQ_CST)) {
    }
    return c;
}

}  // namespace emu

#define threadIdx (emu::cur->tid)
#define blockIdx (emu::cur->bid)
#define blockDim (emu::cur->bdim)
#define gridDim (emu::cur->gdim)

// ---------------------------------------------------------------------------
// Device functions.
// ---------------------------------------------------------------------------
inline int __lane_id() { return emu::cur->lane; }
inline void __syncthreads() { emu::block_op(0); }
inline int __syncthreads_or(int v) { return emu::block_op(v); }
inline void __threadfence() { __atomic_thread_fence(__ATOMIC_SEQ_CST); }

inline unsigned long long __ballot(int pred) {
    uint64_t mask = 0;
    const uint64_t* x = emu::wave_exchange(pred ? 1u : 0u, &mask);
    unsigned long long m = 0;
    for (int l = 0; l < 64; ++l)
        if (((mask >> l) & 1) && x[l]) m |= 1ull << l;
    return m;
}
template <class T>
inline T __shfl(T v, int src, int width = 64) {
    (void)width;
    const uint64_t* x = emu::wave_exchange(emu::bits_of(v));
    return emu::from_bits<T>(x[src & 63]);
}
template <class T>
inline T __shfl_up(T v, unsigned delta, int width = 64) {
    (void)width;
    const uint64_t* x = emu::wave_exchange(emu::bits_of(v));
    const int l = emu::cur->lane;
    return l >= (int)delta ? emu::from_bits<T>(x[l - (int)delta]) : v;
}
template <class T>
inline T __shfl_xor(T v, int mask, int width = 64) {
    (void)width;
    const uint64_t* x = emu::wave_exchange(emu::bits_of(v));
    return emu::from_bits<T>(x[(emu::cur->lane ^ mask) & 63]);
}
#define __builtin_amdgcn_wave_barrier() emu::wave_meet()
#define __builtin_amdgcn_readfirstlane(v) (v)
inline int emu_readlane(int v, int l) { return __shfl(v, l); }
#define __builtin_amdgcn_readlane(v, l) emu_readlane((v), (l))

inline int __popc(unsigned x) { return __builtin_popcount(x); }
inline int __popcll(unsigned long long x) { return __builtin_popcountll(x); }
inline int __ffs(int x) { return __builtin_ffs(x); }
inline int __ffsll(unsigned long long x) { return __builtin_ffsll((long long)x); }
inline int __clz(int x) { return x ? __builtin_clz((unsigned)x) : 32; }
inline int __clzll(long long x) { return x ? __builtin_clzll((unsigned long long)x) : 64; }

inline uint32_t emu_mbcnt_lo(uint32_t mask, uint32_t add) {
    const int l = emu::cur->lane;
    const uint32_t below = l >= 32 ? 0xFFFFFFFFu : ((1u << l) - 1u);
    return add + (uint32_t)__builtin_popcount(mask & below);
}
inline uint32_t emu_mbcnt_hi(uint32_t mask, uint32_t add) {
    const int l = emu::cur->lane - 32;
    const uint32_t below = l <= 0 ? 0u : ((1u << l) - 1u);
    return add + (uint32_t)__builtin_popcount(mask & below);
}
#define __builtin_amdgcn_mbcnt_lo(m, a) emu_mbcnt_lo((m), (a))
#define __builtin_amdgcn_mbcnt_hi(m, a) emu_mbcnt_hi((m), (a))

#define __HIP_MEMORY_SCOPE_SINGLETHREAD 1
#define __HIP_MEMORY_SCOPE_WAVEFRONT 2
#define __HIP_MEMORY_SCOPE_WORKGROUP 3
#define __HIP_MEMORY_SCOPE_AGENT 4
#define __HIP_MEMORY_SCOPE_SYSTEM 5
#define __hip_atomic_load(p, order, scope) __atomic_load_n((p), __ATOMIC_SEQ_CST)
#define __hip_atomic_store(p, v, order, scope) __atomic_store_n((p), (v), __ATOMIC_SEQ_CST)
#define __hip_atomic_fetch_add(p, v, order, scope) __atomic_fetch_add((p), (v), __ATOMIC_SEQ_CST)
#define __hip_atomic_fetch_or(p, v, order, scope) __atomic_fetch_or((p), (v), __ATOMIC_SEQ_CST)
#define __hip_atomic_fetch_and(p, v, order, scope) __atomic_fetch_and((p), (v), __ATOMIC_SEQ_CST)
#define __hip_atomic_fetch_max(p, v, order, scope) emu::fetch_max((p), (v))
#define __hip_atomic_fetch_min(p, v, order, scope) emu::fetch_min((p), (v))
#define __builtin_amdgcn_fence(order, scope) __atomic_thread_fence(__ATOMIC_SEQ_CST)
#define __builtin_amdgcn_s_waitcnt(n) __atomic_thread_fence(__ATOMIC_SEQ_CST)
#define __builtin_amdgcn_s_sleep(n) emu::yield()

template <class T>
inline T atomicAdd(T* p, typename std::common_type<T>::type v) {
    return __atomic_fetch_add(p, v, __ATOMIC_SEQ_CST);
}
template <class T>
inline T atomicOr(T* p, typename std::common_type<T>::type v) {
    return __atomic_fetch_or(p, v, __ATOMIC_SEQ_CST);
}
template <class T>
inline T atomicAnd(T* p, typename std::common_type<T>::type v) {
    return __atomic_fetch_and(p, v, __ATOMIC_SEQ_CST);
}
template <class T>
inline T atomicExch(T* p, typename std::common_type<T>::type v) {
    return __atomic_exchange_n(p, v, __ATOMIC_SEQ_CST);
}
template <class T>
inline T atomicMax(T* p, typename std::common_type<T>::type v) {
    return emu::fetch_max(p, v);
}
template <class T>
inline T atomicMin(T* p, typename std::common_type<T>::type v) {
    return emu::fetch_min(p, v);
}
template <class T>
inline T atomicCAS(T* p, typename std::common_type<T>::type expect, typename std::common_type<T>::type v) {
    __atomic_compare_exchange_n(p, &expect, v, false, __ATOMIC_SEQ_CST, __ATOMIC_SEQ_CST);
    return expect;
}
inline unsigned long long wall_clock64() {
    return (unsigned long long)std::chrono::steady_clock::now().time_since_epoch().count();
}

// ---------------------------------------------------------------------------
// Runtime calls.
// ---------------------------------------------------------------------------
typedef emu::Stream* hipStream_t;
typedef emu::Graph* hipGraph_t;
typedef emu::Graph* hipGraphExec_t;
struct emuEvent {
    std::chrono::steady_clock::time_point t;
};
typedef emuEvent* hipEvent_t;
enum hipMemcpyKind { hipMemcpyHostToHost, hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipMemcpyDeviceToDevice, hipMemcpyDefault };
enum hipStreamCaptureMode { hipStreamCaptureModeGlobal, hipStreamCaptureModeThreadLocal, hipStreamCaptureModeRelaxed };
enum { hipStreamNonBlocking = 1, hipHostMallocCoherent = 1, hipHostMallocPortable = 2, hipHostMallocMapped = 4, hipHostMallocDefault = 0 };
enum hipDeviceAttribute_t { hipDeviceAttributeMultiprocessorCount };
struct hipDeviceProp_t {
    int multiProcessorCount;
    char gcnArchName[64];
};

inline const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "host build"; }
inline hipError_t hipGetLastError() {
    const hipError_t e = emu::last_error;
    emu::last_error = hipSuccess;
    return e;
}
inline hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
inline hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
    p->multiProcessorCount = emu::dev().cus;
    std::strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
inline hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
    *v = emu::dev().cus;
    return hipSuccess;
}
template <class T>
inline hipError_t hipMalloc(T** out, size_t n) {
    if (n > emu::dev().largest_alloc) return emu::set(hipErrorOutOfMemory);
    void* p = nullptr;
    if (posix_memalign(&p, 256, n)) return emu::set(hipErrorOutOfMemory);
    std::memset(p, 0xA5, n);
    *out = (T*)p;
    return hipSuccess;
}
inline hipError_t hipFree(void* p) {
    emu::drain_all();
    std::free(p);
    return hipSuccess;
}
template <class T>
inline hipError_t hipHostMalloc(T** out, size_t n, unsigned = 0) {
    void* p = nullptr;
    if (posix_memalign(&p, 256, n)) return emu::set(hipErrorOutOfMemory);
    std::memset(p, 0xA5, n);
    *out = (T*)p;
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
    emu::drain_all();
    std::free(p);
    return hipSuccess;
}
template <class T>
inline hipError_t hipHostGetDevicePointer(T** out, void* h, unsigned) {
    *out = (T*)h;
    return hipSuccess;
}
inline hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    emu::drain_all();
    std::memcpy(d, s, n);
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st = nullptr) {
    emu::enqueue(st, [=] { std::memcpy(d, s, n); });
    return hipSuccess;
}
inline hipError_t hipMemset(void* d, int v, size_t n) {
    emu::drain_all();
    std::memset(d, v, n);
    return hipSuccess;
}
inline hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t st = nullptr) {
    if (st && st->capturing) {
        std::fprintf(stderr, "host build: memset in a captured graph\n");
        std::abort();
    }
    emu::enqueue(st, [=] { std::memset(d, v, n); });
    return hipSuccess;
}
inline hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    std::lock_guard<std::recursive_mutex> lk(emu::api_mu());
    *s = new emu::Stream();
    emu::streams().push_back(*s);
    return hipSuccess;
}
inline hipError_t hipStreamCreate(hipStream_t* s) { return hipStreamCreateWithFlags(s, 0); }
inline hipError_t hipStreamSynchronize(hipStream_t s) {
    emu::drain_all(s ? s : &emu::null_stream());
    return hipSuccess;
}
inline hipError_t hipStreamDestroy(hipStream_t s) {
    std::lock_guard<std::recursive_mutex> lk(emu::api_mu());
    emu::drain_all();
    auto& v = emu::streams();
    for (size_t i = 0; i < v.size(); ++i)
        if (v[i] == s) {
            v.erase(v.begin() + (long)i);
            break;
        }
    delete s;
    return hipSuccess;
}
inline hipError_t hipDeviceSynchronize() {
    emu::drain_all();
    return hipSuccess;
}
inline hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
    s->capturing = true;
    s->recorded.clear();
    return hipSuccess;
}
inline hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) {
    s->capturing = false;
    *g = new emu::Graph{std::move(s->recorded)};
    s->recorded.clear();
    return hipSuccess;
}
inline hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, void*, void*, size_t) {
    *e = new emu::Graph(*g);
    return hipSuccess;
}
inline hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s) {
    for (auto& f : e->nodes) emu::enqueue(s, f);
    return hipSuccess;
}
inline hipError_t hipGraphDestroy(hipGraph_t g) {
    delete g;
    return hipSuccess;
}
inline hipError_t hipGraphExecDestroy(hipGraphExec_t g) {
    delete g;
    return hipSuccess;
}
inline hipError_t hipEventCreate(hipEvent_t* e) {
    *e = new emuEvent();
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s = nullptr) {
    emu::enqueue(s, [=] { e->t = std::chrono::steady_clock::now(); });
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t) {
    emu::drain_all();
    return hipSuccess;
}
inline hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) {
    *ms = std::chrono::duration<float, std::milli>(b->t - a->t).count();
    return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
    delete e;
    return hipSuccess;
}
inline hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* fn, int, size_t) {
    *n = emu::occupancy_of(fn);
    return hipSuccess;
}
#define HIP_SYMBOL(x) (&(x))
template <class T>
inline hipError_t hipGetSymbolAddress(void** p, T* sym) {
    *p = (void*)sym;
    return hipSuccess;
}

// Persistent kernels: every workgroup has to be resident.
inline hipError_t hipLaunchKernel(const void* fn, dim3 grid, dim3 block, void** args, size_t, hipStream_t s) {
    auto it = emu::kernels().find(fn);
    if (it == emu::kernels().end()) {
        std::fprintf(stderr, "host build: hipLaunchKernel of a kernel that is not named\n");
        std::abort();
    }
    emu::Device& d = emu::dev();
    d.launches.emplace_back(it->second.name, grid.x);
    if (grid.x > (unsigned)(emu::occupancy_of(fn) * d.cus) || grid.x > d.resident) {
        std::fprintf(stderr, "host build: %s: %u workgroups, of which %d are resident\n", it->second.name.c_str(), grid.x,
                     emu::occupancy_of(fn) * d.cus);
        std::abort();
    }
    emu::Launch job{it->second.name, grid, block, it->second.bind(args)};
    emu::enqueue(s, [job] { emu::Pool::get().run(job); });
    return hipSuccess;
}
#define hipLaunchKernelGGL(kernel, grid, block, shmem, stream, ...) \
    emu::launch(#kernel, kernel, grid, block, stream, ##__VA_ARGS__)
