// Stable LSD radix sort for gfx950, one kernel per 8-bit digit place, in the
// place of b40c's radix_sort enactor (b40c/radix_sort/enactor.cuh:520-622) and
// its upsweep/spine/downsweep kernels (radix_sort/upsweep/kernel.cuh:90,
// scan/spine/kernel.cuh:92, radix_sort/downsweep/kernel.cuh:236).
//
// Design (MI355X-first rather than a translation):
//  * 8-bit digits (256 bins) instead of the reference's 4-bit digits: half the
//    passes, and 160 KB of LDS per CU easily holds the per-wave histograms.
//  * The digit totals of every place do not change while keys are permuted, so
//    one kernel (k_histogram) counts them all in one read of the keys.
//  * A place is then one kernel (k_place).  A workgroup owns a tile of
//    consecutive keys: it ranks them, publishes its digit counts, learns where
//    its digits start in the output, and scatters, so HBM moves each key once in
//    and once out per place.  Sixteen more workgroups chain the tiles: they turn
//    the published counts into starts, each for 16 digits.  Workgroups that
//    look back over their predecessors' words by themselves (Merrill and Garland
//    2016) poll 256 words of each and spend more on that than on the keys (2^26
//    64-bit keys: 4.4 ms a sort; with blocks of four tiles, which read their keys
//    twice, 3.5 ms; served, 2.75 ms).
//  * Stable local ranking uses wave64 "match" masks built from 8 ballots (one
//    per digit bit) and per-wave running digit counters in LDS; keys are
//    processed in (wave, round, lane) order which equals index order inside a
//    tile, so ranks are stable.  The tile is exchanged through LDS into digit
//    order and written out as contiguous per-digit runs (two-phase scatter,
//    partition/downsweep/tile.cuh:779-1030).
//  * Sorts of at most SMALL_KEYS keys run every place in one workgroup and one
//    launch (k_small_sort).
//  * Signed and floating-point keys (KeyTraits, radix_sort/sort_utils.cuh:
//    87-183) are ordered by the reference's bit twiddles, applied in
//    registers whenever a digit is extracted: memory always holds the
//    caller's keys, so no pass rewrites them and the trivial-pass skip stays
//    valid for every key type.
//  * The trivial-pass early exit (downsweep/kernel.cuh DownsweepPass) is
//    decided on the device: k_plan flags places whose keys all share one digit;
//    they move nothing, and which buffer a place reads follows from the number
//    of places before it that did (DoubleBuffer::selector).
//  * Scratch comes from the caller as one array of words: a per-call
//    allocation for the stateless entry points, the sort enactor's own buffer,
//    or a fixed device array for the allocation-free entry point; the block
//    size grows until the chain words fit it.  Launching a sort allocates
//    nothing and does not synchronize; only waiting for the selector does.
#include <cstring>
#include <mutex>

#include "common.hpp"
#include "internal.hpp"

namespace b40c {
namespace {

constexpr int RS_BINS = 256;
constexpr int RS_MAX_WGS_PER_CU = 8;
// Most blocks of a place: 64 MB of chain words (128 MB from 2^30 keys on).
constexpr int64_t kMaxBlocks = 1 << 15;

// Order-preserving views of the key bits (sort_utils.cuh:87-183):
// CONV 0 unsigned (as is), 1 signed (flip the sign bit), 2 IEEE float
// (negative: flip all bits; positive: flip the sign bit).
enum KeyConv { KC_UNSIGNED = 0, KC_SIGNED = 1, KC_FLOAT = 2 };

template <typename K, int CONV>
__device__ __forceinline__ K ordered_bits(K k) {
    constexpr K HIGH = (K)1 << (8 * sizeof(K) - 1);
    if (CONV == KC_SIGNED) return k ^ HIGH;
    if (CONV == KC_FLOAT) return k ^ ((k & HIGH) ? (K)~(K)0 : HIGH);
    return k;
}

template <typename K, int CONV>
__device__ __forceinline__ uint32_t digit_of(K key, int shift, uint32_t mask) {
    return (uint32_t)(ordered_bits<K, CONV>(key) >> shift) & mask;
}

// A value the compiler knows nothing about: what is computed from it inside a
// loop stays there.  Otherwise the dozens of offsets and masks that depend on
// the lane alone are kept in registers across the whole tile loop (162 instead
// of 97 VGPRs for 64-bit keys, one workgroup less per CU).
__device__ __forceinline__ int opaque(int x) {
    asm volatile("" : "+v"(x));
    return x;
}

// Ranks of a tile's keys within (wave, digit), in index order; hist (this
// wave's, zeroed) receives the wave's digit counts.  Keys past tile_n get
// 0xFFFFFFFF.  Key j of a lane is tile element wid * 64 * ITEMS + j * 64 + lane.
template <typename K, int CONV, int ITEMS>
__device__ __forceinline__ void rank_tile(const K (&key)[ITEMS], uint32_t (&rank)[ITEMS], uint32_t* hist, int wid,
                                          int tile_n, int shift, uint32_t mask) {
    const int lane = opaque(lane_id());
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const bool valid = wid * (kWave * ITEMS) + j * kWave + lane < tile_n;
        const uint32_t d = digit_of<K, CONV>(key[j], shift, mask);
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const bool bit = (d >> b) & 1u;
            const uint64_t bal = __ballot(bit);
            peers &= bit ? bal : ~bal;
        }
        const uint32_t before = hist[d];
        rank[j] = before + (uint32_t)lane_prefix(peers);
        const bool leader = valid && lane_prefix(peers) == 0;
        if (leader) hist[d] = before + (uint32_t)__popcll(peers);
        if (!valid) rank[j] = 0xFFFFFFFFu;
    }
}

constexpr int OS_THREADS = 512;
constexpr int OS_WAVES = OS_THREADS / kWave;
constexpr int MAX_PLACES = 8;
constexpr int HIST_COPIES = 8;
constexpr int SMALL_THREADS = 1024;
constexpr int SMALL_ITEMS = 8;
constexpr int SMALL_KEYS = SMALL_THREADS * SMALL_ITEMS;

// Device state of one sort, carved out of its scratch words.
struct SortState {
    uint32_t* copies;   // [HIST_COPIES][MAX_PLACES][RS_BINS] digit totals, spread over copies
    uint32_t* base;     // [MAX_PLACES][RS_BINS] first output position of each digit
    uint32_t* trivial;  // [MAX_PLACES] place whose keys all share one digit
    uint32_t* failed;   // beside `trivial`: a place with unfinished blocks (place + 1), and how many it has
    uint32_t* served;   // where a serving workgroup gave up: blocks served, and each digit's next start
    uint32_t* status;   // [2][blocks][RS_BINS] chain words (by place parity), 32 or 64 bits each
    int32_t* out;       // report: selector, unfinished place + 1
    int32_t blocks;
    int32_t wide;       // 64-bit chain words (n >= 2^30)
    int32_t grouped;    // blocks in the order of place_block, else in the workgroups'
    int32_t places;
};
constexpr size_t kReportWords = 16;  // the report, where it is in the scratch (first words)
constexpr size_t kStateWords = kReportWords + (size_t)(HIST_COPIES + 1) * MAX_PLACES * RS_BINS + RS_BINS + 64;
// The unfinished blocks of a place are listed where the totals were, 16 bits each.
static_assert(kMaxBlocks * 2 <= (int64_t)HIST_COPIES * MAX_PLACES * RS_BINS * 4 && kMaxBlocks <= 1 << 16,
              "every block fits the list");

// Clears the totals and the first place's chain words.
__global__ __launch_bounds__(256) void k_sort_init(SortState st) {
    const int64_t step = (int64_t)gridDim.x * 256;
    const int64_t i0 = (int64_t)blockIdx.x * 256 + threadIdx.x;
    for (int64_t i = i0; i < HIST_COPIES * MAX_PLACES * RS_BINS; i += step) st.copies[i] = 0;
    const int64_t words = (int64_t)st.blocks * RS_BINS * (st.wide ? 2 : 1);
    for (int64_t i = i0; i < words; i += step) st.status[i] = 0;
    if (i0 < 2) st.out[i0] = 0;
    if (i0 < 2) st.failed[i0] = 0;
}

// Digit totals of every place in one read, eight keys per thread at a time.
// Where a wave's keys of such a step all share a place's digit (high bits,
// mostly), the place is added once: same-address LDS atomics would cost 64
// times that.  The test is one XOR per key and one ballot per place and step;
// a test per key and place made the kernel issue-bound (300 us instead of
// 125 us for 2^26 64-bit keys).  The workgroups' totals go to HIST_COPIES
// copies: same-line atomics are serialised (11.4 ns).
template <typename K, int CONV>
__global__ __launch_bounds__(OS_THREADS) void k_histogram(const K* keys, int64_t n, int begin_bit, int end_bit,
                                                          SortState st) {
    __shared__ uint32_t hist[2][MAX_PLACES][RS_BINS];
    const int tid = threadIdx.x, lane = lane_id();
    uint32_t(&mine)[MAX_PLACES][RS_BINS] = hist[(tid / kWave) & 1];
    for (int i = tid; i < 2 * MAX_PLACES * RS_BINS; i += OS_THREADS) (&hist[0][0][0])[i] = 0;
    __syncthreads();
    constexpr int R = 8;
    const int64_t step = (int64_t)gridDim.x * OS_THREADS * R;
    for (int64_t base = (int64_t)blockIdx.x * OS_THREADS * R; base < n; base += step) {
        const K* kt = keys + base;
        const uint32_t tn = (uint32_t)min((int64_t)(OS_THREADS * R), n - base);
        K k[R];
#pragma unroll
        for (int j = 0; j < R; ++j) k[j] = kt[min((uint32_t)(j * OS_THREADS + tid), tn - 1u)];
        K differ = 0;
#pragma unroll
        for (int j = 0; j < R; ++j) {
            k[j] = ordered_bits<K, CONV>(k[j]);
            differ |= k[j] ^ k[0];
        }
        const bool whole = tn == (uint32_t)(OS_THREADS * R);
        const K k0 = __shfl(k[0], 0, kWave);
        differ |= k[0] ^ k0;
#pragma unroll
        for (int p = 0; p < (int)sizeof(K); ++p) {
            const int shift = begin_bit + 8 * p;
            if (shift >= end_bit) break;
            const uint32_t mask = (1u << min(8, end_bit - shift)) - 1u;
            if (whole && __ballot(((uint32_t)(differ >> shift) & mask) != 0u) == 0ull) {
                if (lane == 0) atomicAdd(&mine[p][(uint32_t)(k0 >> shift) & mask], (uint32_t)(R * kWave));
                continue;
            }
#pragma unroll
            for (int j = 0; j < R; ++j)
                if (whole || (uint32_t)(j * OS_THREADS + tid) < tn)
                    atomicAdd(&mine[p][(uint32_t)(k[j] >> shift) & mask], 1u);
        }
    }
    __syncthreads();
    uint32_t* out = st.copies + (size_t)(blockIdx.x % HIST_COPIES) * MAX_PLACES * RS_BINS;
    for (int i = tid; i < st.places * RS_BINS; i += OS_THREADS) {
        const uint32_t c = (&hist[0][0][0])[i] + (&hist[1][0][0])[i];
        if (c) atomic_add_u32(&out[i], c);
    }
}

// One workgroup per place: the digits' first output positions, and whether
// the place is trivial.
__global__ __launch_bounds__(RS_BINS) void k_plan(SortState st, int64_t n) {
    __shared__ int s_wave[RS_BINS / kWave];
    const int p = blockIdx.x, d = threadIdx.x;
    uint32_t c = 0;
#pragma unroll
    for (int k = 0; k < HIST_COPIES; ++k) c += st.copies[((size_t)k * MAX_PLACES + p) * RS_BINS + d];
    int total;
    const int excl = wg_exclusive_scan<RS_BINS>((int)c, total, s_wave);
    st.base[p * RS_BINS + d] = (uint32_t)excl;
    const int triv = __syncthreads_or((int64_t)c == n);
    if (d == 0) st.trivial[p] = triv ? 1u : 0u;
}

// Chain of the blocks of a place: one word per block and digit, the block's
// count first (COUNT), then the digit's next output position where the block
// starts (START), which a serving workgroup puts in its place.
//
// No wait needs to end.  A place and a persistent kernel of another stream that
// are each partly resident keep the other's missing workgroups off the GPU (XCDs
// dispatch on their own, so even a block's predecessors may be missing).  A
// serving workgroup gives up after kChainSpins polls without new counts (about 50
// ms; a place of 2^26 keys takes 0.3, and the long blocks of 2^32 keys should publish
// 15 apart at most); blocks without their starts then list themselves and leave
// their keys where they are, later places move nothing, and the host finishes the
// place (no block waits any more: all counts are there) and the places after it.
constexpr uint32_t kChainSpins = 1u << 16;
__device__ __forceinline__ void place_failed(const SortState& st, int place) {
    st.out[1] = place + 1;
    st_relaxed(st.failed, (uint32_t)place + 1);
}
__device__ __forceinline__ uint16_t* unfinished_blocks(const SortState& st) { return (uint16_t*)st.copies; }
template <typename W>
struct ChainWord {
    static constexpr W COUNT = (W)1 << (8 * sizeof(W) - 2);
    static constexpr W START = (W)2 << (8 * sizeof(W) - 2);
    static constexpr W VALUE = COUNT - 1;
};
template <typename W>
__device__ __forceinline__ W chain_load(const W* status, int block, int d) {
    return __hip_atomic_load(&status[(size_t)block * RS_BINS + d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename W>
__device__ __forceinline__ void chain_store(W* status, int block, int d, W w) {
    __hip_atomic_store(&status[(size_t)block * RS_BINS + d], w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Workgroups 0 .. SERVERS - 1 of a place each serve SERVE_DIGITS digits: they turn
// the blocks' counts into starts, a window of OS_WAVES * SERVE_SUBS * ROW blocks
// per round trip past the caches (0.7 us).  A thread has ROW consecutive blocks of
// one digit.  Workgroups are dispatched in order, so the servers run, and the
// lowest block without counts runs, or will as soon as there is room for it beside
// the workgroups dispatched before it that wait for it (none in plain order, up to
// GROUPED_AHEAD in that of place_block); other kernels may leave less room (above).
constexpr int SERVE_DIGITS = 16;  // one 64-byte line of 32-bit words
constexpr int SERVERS = RS_BINS / SERVE_DIGITS;
constexpr int SERVE_SUBS = kWave / SERVE_DIGITS;
// Blocks per thread.  Of few blocks most publish their counts at the same time
// and a wide window takes them in one step (1.3 M 64-bit keys, 318 blocks, 44
// bits: 132 us with 8, 146 with 4); many come a few at a time and a short step
// answers sooner (2^26 keys: 2.92 and 2.75 ms; 4 M 12-byte pairs, 977 blocks:
// 336 and 314 us).
constexpr int SERVE_FEW_BLOCKS = 512;
constexpr int SERVE_ROW_FEW = 8;
constexpr int SERVE_ROW_MANY = 4;

struct ServeShared {
    unsigned long long sum[OS_WAVES][SERVE_DIGITS];
    int lead[OS_WAVES];
};

// RESUME: goes on where the serving workgroup of the place stopped.
template <typename W, int ROW, bool RESUME>
__device__ __forceinline__ void serve_place(W* status, const SortState& st, int place, ServeShared& s) {
    constexpr int WAVE_BLOCKS = SERVE_SUBS * ROW;
    const int tid = threadIdx.x, lane = lane_id(), wid = tid / kWave;
    const int col = lane % SERVE_DIGITS, sub = lane / SERVE_DIGITS;
    const int d = (int)blockIdx.x * SERVE_DIGITS + col;
    const int blocks = st.blocks;
    W start = (W)(RESUME ? st.served[SERVERS + d] : st.base[place * RS_BINS + d]);
    uint32_t spins = 0;
    int first = RESUME ? (int)st.served[blockIdx.x] : 0;
    if (RESUME && chain_load(status, blocks - 1, d) >= ChainWord<W>::START) return;  // served all
    while (first < blocks) {
        const int mine = first + wid * WAVE_BLOCKS + sub * ROW;
        W w[ROW];
#pragma unroll
        for (int r = 0; r < ROW; ++r) w[r] = chain_load(status, min(mine + r, blocks - 1), d);
        int lead = 0;  // leading blocks of the row whose counts are there, for all the digits
#pragma unroll
        for (int r = 0; r < ROW; ++r)
            if (lead == r && mine + r < blocks && w[r] >= ChainWord<W>::COUNT) ++lead;
#pragma unroll
        for (int m = 1; m < SERVE_DIGITS; m <<= 1) lead = min(lead, __shfl_xor(lead, m, kWave));
        int wave_lead = 0;
        bool open = true;
#pragma unroll
        for (int k = 0; k < SERVE_SUBS; ++k) {
            const int l = __shfl(lead, k * SERVE_DIGITS, kWave);
            if (k == sub && !open) lead = 0;
            if (open) wave_lead += l;
            open = open && l == ROW;
        }
        W row = 0, excl[ROW];
#pragma unroll
        for (int r = 0; r < ROW; ++r) {
            excl[r] = row;
            if (r < lead) row += w[r] & ChainWord<W>::VALUE;
        }
        W incl = row;
#pragma unroll
        for (int m = SERVE_DIGITS; m < kWave; m <<= 1) {
            const W o = __shfl_up(incl, m, kWave);
            if (lane >= m) incl += o;
        }
        if (sub == SERVE_SUBS - 1) s.sum[wid][col] = incl;
        if (lane == 0) s.lead[wid] = wave_lead;
        __syncthreads();
        int taken = 0;
        open = true;
        W next = start;
#pragma unroll
        for (int k = 0; k < OS_WAVES; ++k) {
            if (k == wid && open) {
                const W at = next + incl - row;
#pragma unroll
                for (int r = 0; r < ROW; ++r)
                    if (r < lead) chain_store(status, mine + r, d, (W)(ChainWord<W>::START | (at + excl[r])));
            }
            if (open) {
                taken += s.lead[k];
                next += (W)s.sum[k][col];
            }
            open = open && s.lead[k] == WAVE_BLOCKS;
        }
        __syncthreads();
        start = next;
        first += taken;
        if (taken) {
            spins = 0;
        } else {
            if (++spins > kChainSpins) {
                if (tid < SERVE_DIGITS) st.served[SERVERS + d] = (uint32_t)start;
                if (tid == 0) {
                    st.served[blockIdx.x] = (uint32_t)first;
                    place_failed(st, place);
                }
                return;
            }
            __builtin_amdgcn_s_sleep(1);
        }
    }
}

template <bool RESUME>
__device__ __forceinline__ void serve_place(uint32_t* status, const SortState& st, int place, ServeShared& s) {
    if (st.wide)
        serve_place<unsigned long long, SERVE_ROW_MANY, RESUME>((unsigned long long*)status, st, place, s);
    else if (st.blocks <= SERVE_FEW_BLOCKS)
        serve_place<uint32_t, SERVE_ROW_FEW, RESUME>(status, st, place, s);
    else
        serve_place<uint32_t, SERVE_ROW_MANY, RESUME>(status, st, place, s);
}

// The word with the start of a block's digit d, from its server.  Zero: gave up.
template <typename W>
__device__ __forceinline__ W await_start(const W* status, int block, int d, const SortState& st, int place) {
    W w;
    uint32_t spins = 0;
    while ((w = chain_load(status, block, d)) < ChainWord<W>::START) {
        if (++spins % 256 == 0 && (ld_relaxed(st.failed) || spins > 4 * kChainSpins)) {
            place_failed(st, place);
            return 0;
        }
        __builtin_amdgcn_s_sleep(2);
    }
    return w;
}

// Block of the i-th working workgroup.  Workgroups go to the XCDs in turn; of
// every XCD_RUN * 8 blocks each XCD takes XCD_RUN consecutive ones, whose runs
// of a digit meet in the middle of a line: its L2 then writes the line once.
// Blocks then wait for others that are dispatched after them: before block 7 of a
// group, 49 later ones are (7 of each other XCD).  A device that may not hold
// those, the servers and the block itself, at one workgroup per CU, keeps plain
// order.
constexpr int XCDS = 8;
constexpr int XCD_RUN = 8;
constexpr int GROUPED_AHEAD = (XCDS - 1) * (XCD_RUN - 1);
constexpr int GROUPED_CUS = SERVERS + GROUPED_AHEAD + 1;
__device__ __forceinline__ int place_block(int i, int blocks, bool grouped) {
    constexpr int GROUP = XCDS * XCD_RUN;
    if (i < 0 || !grouped || i / GROUP * GROUP + GROUP > blocks) return i;
    return i / GROUP * GROUP + i % XCDS * XCD_RUN + i % GROUP / XCDS;
}

// One digit place.  ITEMS keys per thread: a tile of OS_THREADS * ITEMS keys
// is ranked and staged in LDS at once.  Bound by memory and by waiting for the
// starts: 2^26 64-bit keys take 320 us (1.07 GB of keys in and out, 3.4 TB/s; 295
// us with the wait left out), where counting and scattering kernels took 590.
// The order of the XCDs (place_block) gives 20 to 30 us of that.
// REST: the listed blocks of a place, whose starts are all there.
template <typename K, int CONV, bool VALS, int ITEMS, bool REST>
__global__ __launch_bounds__(OS_THREADS) void k_place(K* k0, K* k1, uint32_t* v0, uint32_t* v1, int64_t n, int place,
                                                      int shift, uint32_t mask, int64_t block_keys, SortState st) {
    constexpr int TILE = OS_THREADS * ITEMS;
    __shared__ K stage_k[TILE];
    __shared__ uint32_t stage_v[VALS ? TILE : 1];
    __shared__ uint32_t wave_hist[OS_WAVES][RS_BINS];
    __shared__ uint32_t next_out[RS_BINS];   // next output position of each digit
    __shared__ uint32_t out_shift[RS_BINS];  // output position minus tile position
    __shared__ uint32_t tile_excl[RS_BINS];
    __shared__ int s_wave[OS_WAVES];
    __shared__ ServeShared s_serve;
    __shared__ uint32_t s_gave_up;

    const int tid = threadIdx.x, lane = lane_id(), wid = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int block = REST ? (int)unfinished_blocks(st)[blockIdx.x]
                           : place_block((int)blockIdx.x - SERVERS, st.blocks, st.grouped != 0);
    const size_t words = (size_t)st.blocks * RS_BINS * (st.wide ? 2 : 1);
    uint32_t* status = st.status + (place & 1) * words;
    int moved = 0;  // places before this one that moved the keys
    for (int p = 0; p < place; ++p) moved += st.trivial[p] ? 0 : 1;
    // The other parity's words of this block, for the next place (its last user, the
    // place before this one, has finished); while the starts are on their way, where
    // the keys' loads need not wait for it (2^25 64-bit keys: 709 us, 720 at the head).
    auto clear_next = [&] {
        uint32_t* next_status = st.status + ((place + 1) & 1) * words;
        for (int i = tid; i < RS_BINS * (st.wide ? 2 : 1); i += OS_THREADS)
            next_status[(size_t)block * RS_BINS * (st.wide ? 2 : 1) + i] = 0;
    };
    if (!REST) {
        const bool skip = st.trivial[place] != 0;
        const uint32_t failed = st.failed[0];
        if (place == st.places - 1 && block == 0 && tid == 0) st.out[0] = (moved + (skip ? 0 : 1)) & 1;
        if (failed && failed <= (uint32_t)place) return;  // (failed == place + 1: in this launch, go on)
        if (skip) {
            if (block >= 0) clear_next();
            return;
        }
        if (block < 0) {
            serve_place<false>(status, st, place, s_serve);
            return;
        }
    }
    const K* kin = (moved & 1) ? k1 : k0;
    K* kout = (moved & 1) ? k0 : k1;
    const uint32_t* vin = VALS ? ((moved & 1) ? v1 : v0) : nullptr;
    uint32_t* vout = VALS ? ((moved & 1) ? v0 : v1) : nullptr;
    const int64_t begin = (int64_t)block * block_keys;
    const int64_t end = min(n, begin + block_keys);
    const bool one_tile = end - begin <= TILE;

    auto announce = [&](uint32_t count) {  // threads 0 .. RS_BINS - 1
        if (st.wide)
            chain_store((unsigned long long*)status, block, tid, ChainWord<unsigned long long>::COUNT | count);
        else
            chain_store(status, block, tid, ChainWord<uint32_t>::COUNT | count);
    };
    if (!REST && !one_tile) {
        for (int i = lane; i < RS_BINS; i += kWave) wave_hist[wid][i] = 0;
        __syncthreads();
        for (int64_t tb = begin; tb < end; tb += TILE) {
            const uint32_t tn = (uint32_t)min((int64_t)TILE, end - tb);
            const K* kt = kin + tb;
            K key[ITEMS];
#pragma unroll
            for (int j = 0; j < ITEMS; ++j) key[j] = kt[min((uint32_t)(j * OS_THREADS + tid), tn - 1u)];
#pragma unroll
            for (int j = 0; j < ITEMS; ++j)
                if ((uint32_t)(j * OS_THREADS + tid) < tn)
                    atomicAdd(&wave_hist[wid][digit_of<K, CONV>(key[j], shift, mask)], 1u);
        }
        __syncthreads();
        if (tid < RS_BINS) {
            uint32_t count = 0;
#pragma unroll
            for (int w = 0; w < OS_WAVES; ++w) count += wave_hist[w][tid];
            announce(count);
        }
        clear_next();
        __syncthreads();
    }
    for (int64_t tile_base = begin; tile_base < end; tile_base += TILE) {
        const int tile_n = (int)min((int64_t)TILE, end - tile_base);
        const int tid = opaque((int)threadIdx.x);
        const int lane = tid % kWave;
        // Positions past the end read the last key instead: no branch per load.
        K key[ITEMS];
        uint32_t val[ITEMS];
        uint32_t rank[ITEMS];
        const K* kt = kin + tile_base;
        const uint32_t* vt = VALS ? vin + tile_base : nullptr;
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            const uint32_t idx = min((uint32_t)(wid * (kWave * ITEMS) + j * kWave + lane), (uint32_t)tile_n - 1u);
            key[j] = kt[idx];
            if (VALS) val[j] = vt[idx];
        }
        for (int i = lane; i < RS_BINS; i += kWave) wave_hist[wid][i] = 0;
        if (!REST && tid == 0) s_gave_up = 0;
        __syncthreads();
        rank_tile<K, CONV, ITEMS>(key, rank, wave_hist[wid], wid, tile_n, shift, mask);
        __syncthreads();
        // Per digit: offsets of each wave inside the digit, and tile totals.
        uint32_t cnt = 0;
        if (tid < RS_BINS) {
#pragma unroll
            for (int w = 0; w < OS_WAVES; ++w) {
                const uint32_t c = wave_hist[w][tid];
                wave_hist[w][tid] = cnt;
                cnt += c;
            }
            if (!REST && one_tile) announce(cnt);
        }
        if (!REST && one_tile) clear_next();
        int tot;
        const int excl = wg_exclusive_scan<OS_THREADS>((int)cnt, tot, s_wave);
        if (tid < RS_BINS) tile_excl[tid] = (uint32_t)excl;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            if (rank[j] != 0xFFFFFFFFu) {
                const uint32_t d = digit_of<K, CONV>(key[j], shift, mask);
                const uint32_t pos = tile_excl[d] + wave_hist[wid][d] + rank[j];
                stage_k[pos] = key[j];
                if (VALS) stage_v[pos] = val[j];
            }
        }
        if (tid < RS_BINS) {
            uint32_t at;
            if (tile_base != begin) {
                at = next_out[tid];
            } else if (st.wide) {
                const unsigned long long w = await_start((const unsigned long long*)status, block, tid, st, place);
                if (w == 0) s_gave_up = 1;
                at = (uint32_t)(w & ChainWord<unsigned long long>::VALUE);
            } else {
                const uint32_t w = await_start((const uint32_t*)status, block, tid, st, place);
                if (w == 0) s_gave_up = 1;
                at = w & ChainWord<uint32_t>::VALUE;
            }
            out_shift[tid] = at - (uint32_t)excl;
            next_out[tid] = at + cnt;
        }
        __syncthreads();
        if (!REST && s_gave_up) {
            if (tid == 0) unfinished_blocks(st)[atomic_add_u32(&st.failed[1], 1u)] = (uint16_t)block;
            return;
        }
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            const int k = j * OS_THREADS + tid;
            if (k < tile_n) {
                const K kk = stage_k[k];
                const uint32_t out = out_shift[digit_of<K, CONV>(kk, shift, mask)] + (uint32_t)k;
                kout[out] = kk;
                if (VALS) vout[out] = stage_v[k];
            }
        }
        __syncthreads();
    }
}

// A place with unfinished blocks: serves all of them (their counts are there).
__global__ __launch_bounds__(OS_THREADS) void k_place_resume(SortState st, int place) {
    __shared__ ServeShared s_serve;
    serve_place<true>(st.status + (place & 1) * (size_t)st.blocks * RS_BINS * (st.wide ? 2 : 1), st, place, s_serve);
}
// ... and it is finished.
__global__ __launch_bounds__(kWave) void k_place_finished(SortState st) {
    if (threadIdx.x < 2) st.failed[threadIdx.x] = 0;
    if (threadIdx.x == 0) st.out[1] = 0;
}

// Every place of a small sort in one workgroup: the keys stay in registers
// and LDS between the places.  A launch costs 2.5 us or more and a place of a
// few thousand keys about as much, so the launches of the large form would be
// most of such a sort (6,001 32-bit pairs: 31 us against 100 us in 17
// launches).
template <typename K, int CONV, bool VALS>
__global__ __launch_bounds__(SMALL_THREADS) void k_small_sort(K* k0, K* k1, uint32_t* v0, uint32_t* v1, int n,
                                                              int begin_bit, int end_bit, int32_t* out) {
    constexpr int WAVES = SMALL_THREADS / kWave;
    __shared__ K stage_k[SMALL_KEYS];
    __shared__ uint32_t stage_v[VALS ? SMALL_KEYS : 1];
    __shared__ uint32_t wave_hist[WAVES][RS_BINS];
    __shared__ uint32_t tile_excl[RS_BINS];
    __shared__ int s_wave[WAVES];
    const int tid = threadIdx.x, lane = lane_id(), wid = tid / kWave;
    K key[SMALL_ITEMS];
    uint32_t val[SMALL_ITEMS], rank[SMALL_ITEMS];
#pragma unroll
    for (int j = 0; j < SMALL_ITEMS; ++j) {
        const int idx = wid * (kWave * SMALL_ITEMS) + j * kWave + lane;
        key[j] = idx < n ? k0[idx] : (K)0;
        if (VALS) val[j] = idx < n ? v0[idx] : 0u;
    }
    int moved = 0;
    for (int shift = begin_bit; shift < end_bit; shift += 8) {
        const uint32_t mask = (1u << min(8, end_bit - shift)) - 1u;
        for (int i = lane; i < RS_BINS; i += kWave) wave_hist[wid][i] = 0;
        __syncthreads();
        rank_tile<K, CONV, SMALL_ITEMS>(key, rank, wave_hist[wid], wid, n, shift, mask);
        __syncthreads();
        uint32_t cnt = 0;
        if (tid < RS_BINS) {
#pragma unroll
            for (int w = 0; w < WAVES; ++w) {
                const uint32_t c = wave_hist[w][tid];
                wave_hist[w][tid] = cnt;
                cnt += c;
            }
        }
        int tot;
        const int excl = wg_exclusive_scan<SMALL_THREADS>((int)cnt, tot, s_wave);
        if (tid < RS_BINS) tile_excl[tid] = (uint32_t)excl;
        if (__syncthreads_or(tid < RS_BINS && cnt == (uint32_t)n)) continue;  // all keys share one digit
        ++moved;
#pragma unroll
        for (int j = 0; j < SMALL_ITEMS; ++j) {
            if (rank[j] != 0xFFFFFFFFu) {
                const uint32_t d = digit_of<K, CONV>(key[j], shift, mask);
                const uint32_t pos = tile_excl[d] + wave_hist[wid][d] + rank[j];
                stage_k[pos] = key[j];
                if (VALS) stage_v[pos] = val[j];
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < SMALL_ITEMS; ++j) {
            const int idx = wid * (kWave * SMALL_ITEMS) + j * kWave + lane;
            if (idx < n) {
                key[j] = stage_k[idx];
                if (VALS) val[j] = stage_v[idx];
            }
        }
    }
    if (moved) {
        K* ko = (moved & 1) ? k1 : k0;
        uint32_t* vo = (moved & 1) ? v1 : v0;
#pragma unroll
        for (int j = 0; j < SMALL_ITEMS; ++j) {
            const int idx = wid * (kWave * SMALL_ITEMS) + j * kWave + lane;
            if (idx < n) {
                ko[idx] = key[j];
                if (VALS) vo[idx] = val[j];
            }
        }
    }
    if (tid == 0) {
        out[0] = moved & 1;
        out[1] = 0;
    }
}

// Block size and count for n keys: whole tiles, at most `max_blocks` blocks.
struct SortPlan {
    int64_t block_keys = 1;
    int blocks = 1;
    int items = 8;
    bool wide = false;
    bool grouped = false;
    int hist_wgs = 1;
};

bool wide_words(int64_t n) { return n >= (1ll << 30); }
size_t look_words(int64_t blocks, bool wide) { return (size_t)2 * blocks * RS_BINS * (wide ? 2 : 1); }

// Blocks of one tile: longer ones read their keys twice, and are for sorts
// whose chain words would exceed the scratch or kMaxBlocks, and for a policy
// that names a number of workgroups.
SortPlan sort_plan(int64_t n, int num_cus, const SortPolicy& pol, size_t max_words) {
    SortPlan p;
    p.items = pol.items;
    p.wide = wide_words(n);
    p.grouped = num_cus >= GROUPED_CUS;
    const int64_t tile = (int64_t)OS_THREADS * pol.items;
    const int64_t tiles = std::max<int64_t>(1, (n + tile - 1) / tile);
    int64_t most = kMaxBlocks;
    if (pol.wgs_per_cu > 0) most = (int64_t)num_cus * pol.wgs_per_cu;
    if (n > SMALL_KEYS) most = std::min<int64_t>(most, (max_words - kStateWords) / look_words(1, p.wide));
    const int64_t per = (tiles + most - 1) / most;
    p.block_keys = per * tile;
    p.blocks = (int)((tiles + per - 1) / per);
    p.hist_wgs = (int)std::min<int64_t>((n + OS_THREADS * 8 - 1) / (OS_THREADS * 8), (int64_t)num_cus * 2);
    return p;
}

SortState sort_state(const SortScratch& sc, const SortPlan& plan, int places, int32_t* out) {
    SortState st;
    st.copies = sc.base + kReportWords;
    st.base = st.copies + (size_t)HIST_COPIES * MAX_PLACES * RS_BINS;
    st.trivial = st.base + (size_t)MAX_PLACES * RS_BINS;
    st.failed = st.trivial + MAX_PLACES;
    st.served = st.failed + 2;
    st.status = sc.base + kStateWords;
    st.out = out;
    st.blocks = plan.blocks;
    st.wide = plan.wide ? 1 : 0;
    st.grouped = plan.grouped ? 1 : 0;
    st.places = places;
    return st;
}

// Places of a sort that stopped at `place`, `blocks` of whose blocks are unfinished.
struct SortRest {
    int place = -1;
    uint32_t blocks = 0;
};

template <typename K, int CONV, bool VALS, int ITEMS>
void launch_places(K* k0, K* k1, uint32_t* v0, uint32_t* v1, int64_t n, int begin_bit, int end_bit,
                   const SortPlan& plan, const SortState& st, const SortRest& rest, hipStream_t stream) {
    auto mask_of = [&](int shift) { return (1u << std::min(8, end_bit - shift)) - 1u; };
    if (rest.place < 0) {
        const int64_t clear = (int64_t)HIST_COPIES * MAX_PLACES * RS_BINS + (int64_t)look_words(plan.blocks, plan.wide) / 2;
        hipLaunchKernelGGL(k_sort_init, dim3((unsigned)std::min<int64_t>((clear + 1023) / 1024, 512)), dim3(256), 0,
                           stream, st);
        hipLaunchKernelGGL((k_histogram<K, CONV>), dim3(plan.hist_wgs), dim3(OS_THREADS), 0, stream, (const K*)k0, n,
                           begin_bit, end_bit, st);
        hipLaunchKernelGGL(k_plan, dim3(st.places), dim3(RS_BINS), 0, stream, st, n);
    } else {
        const int shift = begin_bit + 8 * rest.place;
        hipLaunchKernelGGL(k_place_resume, dim3(SERVERS), dim3(OS_THREADS), 0, stream, st, rest.place);
        if (rest.blocks)
            hipLaunchKernelGGL((k_place<K, CONV, VALS, ITEMS, true>), dim3(rest.blocks), dim3(OS_THREADS), 0, stream,
                               k0, k1, v0, v1, n, rest.place, shift, mask_of(shift), plan.block_keys, st);
        hipLaunchKernelGGL(k_place_finished, dim3(1), dim3(kWave), 0, stream, st);
    }
    for (int place = rest.place + 1; place < st.places; ++place) {
        const int shift = begin_bit + 8 * place;
        hipLaunchKernelGGL((k_place<K, CONV, VALS, ITEMS, false>), dim3(plan.blocks + SERVERS), dim3(OS_THREADS), 0,
                           stream, k0, k1, v0, v1, n, place, shift, mask_of(shift), plan.block_keys, st);
    }
}

template <typename K, int CONV>
void launch_typed(void* k0, void* k1, uint32_t* v0, uint32_t* v1, int64_t n, int begin_bit, int end_bit,
                  const SortPlan& plan, const SortScratch& sc, int32_t* out, const SortRest& rest, hipStream_t stream) {
    if (n <= SMALL_KEYS) {
        if (v0)
            hipLaunchKernelGGL((k_small_sort<K, CONV, true>), dim3(1), dim3(SMALL_THREADS), 0, stream, (K*)k0, (K*)k1,
                               v0, v1, (int)n, begin_bit, end_bit, out);
        else
            hipLaunchKernelGGL((k_small_sort<K, CONV, false>), dim3(1), dim3(SMALL_THREADS), 0, stream, (K*)k0, (K*)k1,
                               v0, v1, (int)n, begin_bit, end_bit, out);
        return;
    }
    const SortState st = sort_state(sc, plan, (end_bit - begin_bit + 7) / 8, out);
    auto launch = v0 ? (plan.items == 16 ? launch_places<K, CONV, true, 16> : launch_places<K, CONV, true, 8>)
                     : (plan.items == 16 ? launch_places<K, CONV, false, 16> : launch_places<K, CONV, false, 8>);
    launch((K*)k0, (K*)k1, v0, v1, n, begin_bit, end_bit, plan, st, rest, stream);
}

int key_bits(int32_t key_type) {
    switch (key_type) {
        case B40C_KEY_U32:
        case B40C_KEY_I32:
        case B40C_KEY_F32:
            return 32;
        case B40C_KEY_U64:
        case B40C_KEY_I64:
        case B40C_KEY_F64:
            return 64;
    }
    return 0;
}

b40c_status validate(const char* who, int32_t key_type, const void* k0, const void* k1, const uint32_t* v0,
                     const uint32_t* v1, int64_t n, int begin_bit, int end_bit, const int32_t* selector) {
    const int kb = key_bits(key_type);
    if (!kb) return fail(B40C_ERR_INVALID_ARG, "%s: unknown key type %d", who, key_type);
    if (!selector || (n > 0 && (!k0 || !k1)) || ((v0 == nullptr) != (v1 == nullptr)))
        return fail(B40C_ERR_INVALID_ARG, "%s: null pointer", who);
    if (n < 0 || begin_bit < 0 || end_bit > kb || begin_bit > end_bit)
        return fail(B40C_ERR_INVALID_ARG, "%s: bad arguments (n=%lld bits=[%d,%d))", who, (long long)n, begin_bit,
                    end_bit);
    if (n > 0xFFFFFFFFll) return fail(B40C_ERR_UNSUPPORTED, "%s: n=%lld exceeds 2^32-1", who, (long long)n);
    return B40C_OK;
}

}  // namespace

// Default keys per thread: 16 where key and value are at most 8 bytes (the tile
// is 64 KB of LDS, two workgroups per CU) and the sort gives the CUs almost two
// (1.75) of these workgroups each; else 8.  Longer runs of a digit waste fewer
// partial lines (16 against 8, 2^26 64-bit keys: 2.91 and 3.15 ms; 32-bit pairs
// 1.58 and 1.70; 4 M 64-bit keys 230 and 246 us), but shorter sorts lack
// workgroups (3 M 64-bit keys: 216 and 208 us; 1.3 M 32-bit pairs 80 and 74) and
// 12-byte pairs the LDS (4 M pairs: 413 and 336 us).
SortPolicy resolve_sort_policy(SortPolicy p, int64_t n, int pair_bytes, int num_cus) {
    if (p.items != 8 && p.items != 16)
        p.items = pair_bytes <= 8 && 4 * n >= 7 * (int64_t)num_cus * OS_THREADS * 16 ? 16 : 8;
    if (p.wgs_per_cu < 0 || p.wgs_per_cu > RS_MAX_WGS_PER_CU) p.wgs_per_cu = 0;
    return p;
}

// Never less for more keys, whatever the policy: an enactor's scratch serves
// every sort of at most as many keys as the one that sized it.
size_t sort_scratch_words(int64_t n) {
    if (n <= SMALL_KEYS) return kReportWords;
    const int64_t blocks = std::min<int64_t>((n + OS_THREADS * 8 - 1) / (OS_THREADS * 8), kMaxBlocks);
    return kStateWords + look_words(blocks, wide_words(n));
}

namespace {
// Scratch that any sort can do with, in fewer and longer blocks: that of the
// allocation-free entry point.
constexpr size_t kNoAllocWords = (size_t)RS_BINS * 2048 + 2 * RS_BINS + 64;
static_assert((kNoAllocWords - kStateWords) / (2 * RS_BINS) == 988 && (kNoAllocWords - kStateWords) / (4 * RS_BINS) == 494,
              "the blocks that its comment names");

// A sort's scratch in device memory of at least `words` words, or what there is room for.
b40c_status reserve_scratch(DeviceBuffer& mem, size_t words) {
    const b40c_status s = mem.reserve(words * sizeof(uint32_t));
    if (s != B40C_ERR_OOM || words <= kNoAllocWords) return s;
    (void)hipGetLastError();
    return mem.reserve(kNoAllocWords * sizeof(uint32_t));
}

// One sort's report words (selector, unfinished place + 1): a pinned slot, or, without one,
// the first words of the scratch, copied back after the sort.
struct SortReport {
    ReportSlot slot;
    int32_t* dev = nullptr;
    void take(const SortScratch& sc, bool pinned) {
        dev = static_cast<int32_t*>(pinned && slot.take() ? slot.dev : sc.base);
    }
    b40c_status wait(int32_t (&words)[2], hipStream_t stream) {
        if (!slot.host) B40C_HIP(hipMemcpyAsync(words, dev, sizeof(words), hipMemcpyDeviceToHost, stream));
        B40C_HIP(hipStreamSynchronize(stream));
        if (slot.host) std::memcpy(words, slot.host, sizeof(words));
        return B40C_OK;
    }
};
}  // namespace

// Launches the sort, or what is left of it (no allocation, no synchronization).
static b40c_status radix_sort_launch(int32_t key_type, void* k0, void* k1, uint32_t* v0, uint32_t* v1, int64_t n,
                                     int begin_bit, int end_bit, int num_cus, const SortPolicy& pol,
                                     const SortScratch& sc, int32_t* report, const SortRest& rest,
                                     hipStream_t stream) {
    const SortPlan plan = sort_plan(n, num_cus, pol, sc.words);
    switch (key_type) {
        case B40C_KEY_U32: launch_typed<uint32_t, KC_UNSIGNED>(k0, k1, v0, v1, n, begin_bit, end_bit, plan, sc, report, rest, stream); break;
        case B40C_KEY_I32: launch_typed<uint32_t, KC_SIGNED>(k0, k1, v0, v1, n, begin_bit, end_bit, plan, sc, report, rest, stream); break;
        case B40C_KEY_F32: launch_typed<uint32_t, KC_FLOAT>(k0, k1, v0, v1, n, begin_bit, end_bit, plan, sc, report, rest, stream); break;
        case B40C_KEY_U64: launch_typed<uint64_t, KC_UNSIGNED>(k0, k1, v0, v1, n, begin_bit, end_bit, plan, sc, report, rest, stream); break;
        case B40C_KEY_I64: launch_typed<uint64_t, KC_SIGNED>(k0, k1, v0, v1, n, begin_bit, end_bit, plan, sc, report, rest, stream); break;
        case B40C_KEY_F64: launch_typed<uint64_t, KC_FLOAT>(k0, k1, v0, v1, n, begin_bit, end_bit, plan, sc, report, rest, stream); break;
        default: return fail(B40C_ERR_INVALID_ARG, "radix sort: unknown key type %d", key_type);
    }
    B40C_HIP(hipGetLastError());
    return B40C_OK;
}

// Runs a sort with its scratch and waits for the selector (one stream
// synchronization).  `pinned` false: nothing is allocated, not even the
// report page of the process's first sort.
static b40c_status radix_sort_sync(int32_t key_type, void* k0, void* k1, uint32_t* v0, uint32_t* v1, int64_t n,
                                   int begin_bit, int end_bit, int num_cus, const SortPolicy& pol,
                                   const SortScratch& sc, int32_t* selector, hipStream_t stream, bool pinned = true) {
    SortReport report;
    report.take(sc, pinned);
    SortRest rest;
    int32_t words[2] = {0, 0};
    do {
        const b40c_status launched = radix_sort_launch(key_type, k0, k1, v0, v1, n, begin_bit, end_bit, num_cus, pol,
                                                       sc, report.dev, rest, stream);
        if (launched != B40C_OK) {
            // Some kernels may be on their way: the report is theirs until they end.
            (void)hipStreamSynchronize(stream);
            return launched;
        }
        B40C_TRY(report.wait(words, stream));
        if (words[1]) {  // a place later each time
            rest.place = words[1] - 1;
            const uint32_t* unfinished = sort_state(sc, SortPlan{}, 0, nullptr).failed + 1;
            B40C_HIP(hipMemcpyAsync(&rest.blocks, unfinished, sizeof(rest.blocks), hipMemcpyDeviceToHost, stream));
            B40C_HIP(hipStreamSynchronize(stream));
        }
    } while (words[1]);
    *selector = words[0];
    return B40C_OK;
}

// Stateless form: with the caller's scratch if it is large enough, else
// allocated for this call.
b40c_status radix_sort_once(int32_t key_type, void* k0, void* k1, uint32_t* v0, uint32_t* v1, int64_t n, int begin_bit,
                            int end_bit, int32_t* selector, hipStream_t stream, uint32_t* scratch = nullptr,
                            size_t scratch_words = 0) {
    *selector = 0;
    if (n <= 1 || begin_bit == end_bit) return B40C_OK;
    DeviceInfo info;
    B40C_TRY(device_info(info));
    DeviceBuffer mem;
    const SortPolicy pol = resolve_sort_policy(SortPolicy{}, n, key_bits(key_type) / 8 + (v0 ? 4 : 0), info.num_cus);
    const size_t words = sort_scratch_words(n);
    if (!scratch || scratch_words < words) {
        B40C_TRY(reserve_scratch(mem, words));
        scratch = mem.as<uint32_t>();
        scratch_words = mem.bytes / sizeof(uint32_t);
    }
    return radix_sort_sync(key_type, k0, k1, v0, v1, n, begin_bit, end_bit, info.num_cus, pol,
                           SortScratch{scratch, scratch_words}, selector, stream);
}

b40c_status radix_sort_u64(uint64_t* k0, uint64_t* k1, int64_t n, int begin_bit, int end_bit, int32_t* selector,
                           hipStream_t stream, uint32_t* scratch_mem, size_t scratch_words) {
    B40C_TRY(validate("radix sort", B40C_KEY_U64, k0, k1, nullptr, nullptr, n, begin_bit, end_bit, selector));
    return radix_sort_once(B40C_KEY_U64, k0, k1, nullptr, nullptr, n, begin_bit, end_bit, selector, stream, scratch_mem,
                           scratch_words);
}

b40c_status radix_sort_pairs_u32(uint32_t* k0, uint32_t* k1, uint32_t* v0, uint32_t* v1, int64_t n, int begin_bit,
                                 int end_bit, int32_t* selector, hipStream_t stream) {
    B40C_TRY(validate("radix sort", B40C_KEY_U32, k0, k1, v0, v1, n, begin_bit, end_bit, selector));
    return radix_sort_once(B40C_KEY_U32, k0, k1, v0, v1, n, begin_bit, end_bit, selector, stream);
}

}  // namespace b40c

// ---------------------------------------------------------------------------
// Allocation-free sort (no counterpart in the reference): its scratch is this
// fixed device array, one copy per GPU, which the GPU keeps until the
// process ends: 2 MiB + 2 KiB, enough for the chain words of 988 blocks
// (494 from 2^30 keys on); blocks are as large as n <= 2^32 - 1 keys then need.
// In host code `scratch` is only a stand-in for the device array; its device
// address comes from hipGetSymbolAddress, once per device, and only that address
// is used.
// ---------------------------------------------------------------------------
static __device__ __align__(256) uint32_t scratch[b40c::kNoAllocWords];

namespace b40c {
namespace {
constexpr int kNoAllocMaxDevices = 64;
struct NoAllocSlot {
    std::once_flag once;
    hipError_t err = hipSuccess;
    uint32_t* ptr = nullptr;  // device address of `scratch` on this device
    int num_cus = 0;
};
NoAllocSlot g_noalloc[kNoAllocMaxDevices];

// Resolves the calling thread's current device's copy of `scratch` (first
// call on a device only).
b40c_status noalloc_slot(NoAllocSlot*& out) {
    int dev = 0;
    B40C_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= kNoAllocMaxDevices)
        return fail(B40C_ERR_UNSUPPORTED, "allocation-free sort: device %d beyond the %d supported", dev,
                    kNoAllocMaxDevices);
    NoAllocSlot& slot = g_noalloc[dev];
    std::call_once(slot.once, [&] {
        slot.err = hipGetSymbolAddress((void**)&slot.ptr, HIP_SYMBOL(scratch));
        if (slot.err == hipSuccess) slot.err = hipDeviceGetAttribute(&slot.num_cus, hipDeviceAttributeMultiprocessorCount, dev);
    });
    if (slot.err != hipSuccess)
        return fail(B40C_ERR_HIP, "allocation-free sort: resolving the scratch array failed: %s",
                    hipGetErrorString(slot.err));
    out = &slot;
    return B40C_OK;
}
}  // namespace
}  // namespace b40c

// Sort enactor: owns its scratch across calls, like the reference Enactor's
// spine storage (radix_sort/enactor.cuh:96-140).  One stream per enactor.
struct b40c_sort_enactor {
    b40c::DeviceBuffer scratch;
    hipStream_t stream = nullptr;
    b40c::SortPolicy policy;  // zero fields: the size-based default
};

using namespace b40c;

extern "C" {

b40c_status b40c_radix_sort_u64(uint64_t* d_keys0, uint64_t* d_keys1, int64_t n, int32_t begin_bit, int32_t end_bit,
                                int32_t* selector) {
    B40C_TRY(validate("b40c_radix_sort_u64", B40C_KEY_U64, d_keys0, d_keys1, nullptr, nullptr, n, begin_bit, end_bit,
                      selector));
    return radix_sort_once(B40C_KEY_U64, d_keys0, d_keys1, nullptr, nullptr, n, begin_bit, end_bit, selector, nullptr);
}

b40c_status b40c_radix_sort_pairs_u32(uint32_t* d_keys0, uint32_t* d_keys1, uint32_t* d_vals0, uint32_t* d_vals1,
                                      int64_t n, int32_t begin_bit, int32_t end_bit, int32_t* selector) {
    if (n > 0 && (!d_vals0 || !d_vals1))
        return fail(B40C_ERR_INVALID_ARG, "b40c_radix_sort_pairs_u32: null pointer");
    B40C_TRY(validate("b40c_radix_sort_pairs_u32", B40C_KEY_U32, d_keys0, d_keys1, d_vals0, d_vals1, n, begin_bit,
                      end_bit, selector));
    return radix_sort_once(B40C_KEY_U32, d_keys0, d_keys1, d_vals0, d_vals1, n, begin_bit, end_bit, selector, nullptr);
}

b40c_status b40c_radix_sort(int32_t key_type, void* d_keys0, void* d_keys1, uint32_t* d_vals0, uint32_t* d_vals1,
                            int64_t n, int32_t begin_bit, int32_t end_bit, int32_t* selector) {
    B40C_TRY(validate("b40c_radix_sort", key_type, d_keys0, d_keys1, d_vals0, d_vals1, n, begin_bit, end_bit, selector));
    return radix_sort_once(key_type, d_keys0, d_keys1, d_vals0, d_vals1, n, begin_bit, end_bit, selector, nullptr);
}

b40c_status b40c_radix_sort_u64_noalloc(uint64_t* d_keys0, uint64_t* d_keys1, int64_t n, int32_t begin_bit,
                                        int32_t end_bit, int32_t* selector) {
    B40C_TRY(validate("b40c_radix_sort_u64_noalloc", B40C_KEY_U64, d_keys0, d_keys1, nullptr, nullptr, n, begin_bit,
                      end_bit, selector));
    *selector = 0;
    if (n <= 1 || begin_bit == end_bit) return B40C_OK;
    NoAllocSlot* slot = nullptr;
    B40C_TRY(noalloc_slot(slot));
    const SortPolicy pol = resolve_sort_policy(SortPolicy{}, n, 8, slot->num_cus);
    return radix_sort_sync(B40C_KEY_U64, d_keys0, d_keys1, nullptr, nullptr, n, begin_bit, end_bit, slot->num_cus,
                           pol, SortScratch{slot->ptr, kNoAllocWords}, selector, nullptr, false);
}

b40c_status b40c_sort_enactor_create(b40c_sort_enactor** out) {
    if (!out) return fail(B40C_ERR_INVALID_ARG, "b40c_sort_enactor_create: null out");
    b40c_sort_enactor* e = new b40c_sort_enactor();
    const hipError_t err = hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking);
    if (err != hipSuccess) {
        delete e;
        return fail(B40C_ERR_HIP, "b40c_sort_enactor_create: %s", hipGetErrorString(err));
    }
    *out = e;
    return B40C_OK;
}

b40c_status b40c_sort_enactor_sort(b40c_sort_enactor* e, int32_t key_type, void* d_keys0, void* d_keys1,
                                   uint32_t* d_vals0, uint32_t* d_vals1, int64_t n, int32_t begin_bit, int32_t end_bit,
                                   int32_t* selector) {
    if (!e) return fail(B40C_ERR_INVALID_ARG, "b40c_sort_enactor_sort: null enactor");
    B40C_TRY(validate("b40c_sort_enactor_sort", key_type, d_keys0, d_keys1, d_vals0, d_vals1, n, begin_bit, end_bit,
                      selector));
    *selector = 0;
    if (n <= 1 || begin_bit == end_bit) return B40C_OK;
    DeviceInfo info;
    B40C_TRY(device_info(info));
    const SortPolicy pol = resolve_sort_policy(e->policy, n, key_bits(key_type) / 8 + (d_vals0 ? 4 : 0), info.num_cus);
    const size_t words = sort_scratch_words(n);
    // Grow-only: later sorts of at most this size allocate nothing.
    B40C_TRY(reserve_scratch(e->scratch, words));
    return radix_sort_sync(key_type, d_keys0, d_keys1, d_vals0, d_vals1, n, begin_bit, end_bit, info.num_cus, pol,
                           SortScratch{e->scratch.as<uint32_t>(), e->scratch.bytes / sizeof(uint32_t)}, selector,
                           e->stream);
}

b40c_status b40c_sort_enactor_set_policy(b40c_sort_enactor* e, int32_t items_per_thread, int32_t wgs_per_cu) {
    if (!e) return fail(B40C_ERR_INVALID_ARG, "b40c_sort_enactor_set_policy: null enactor");
    if ((items_per_thread != 0 && items_per_thread != 8 && items_per_thread != 16) || wgs_per_cu < 0 ||
        wgs_per_cu > RS_MAX_WGS_PER_CU)
        return fail(B40C_ERR_INVALID_ARG,
                    "b40c_sort_enactor_set_policy: items_per_thread must be 0, 8 or 16 and wgs_per_cu 0-%d (got %d, %d)",
                    RS_MAX_WGS_PER_CU, items_per_thread, wgs_per_cu);
    e->policy.items = items_per_thread;
    e->policy.wgs_per_cu = wgs_per_cu;
    return B40C_OK;
}

void b40c_sort_enactor_destroy(b40c_sort_enactor* e) {
    if (!e) return;
    if (e->stream) {
        (void)hipStreamSynchronize(e->stream);
        (void)hipStreamDestroy(e->stream);
    }
    delete e;
}

}  // extern "C"
