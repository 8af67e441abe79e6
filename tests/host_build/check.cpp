// Checks of the library's own entry points on the host build (test
// infrastructure only): check CASE [ARGUMENT...].  Each case prints what it runs
// and exits 0 if everything held; results are compared with the serial
// references below.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdarg>
#include <random>
#include <set>

#include "b40c_mi355x.h"

namespace {

[[noreturn]] void die(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    std::fprintf(stderr, "check failed: ");
    std::vfprintf(stderr, fmt, ap);
    std::fprintf(stderr, " [last error: %s]\n", b40c_last_error_string());
    va_end(ap);
    std::fflush(nullptr);
    _Exit(1);
}
#define REQUIRE(cond, ...)                                        \
    do {                                                          \
        if (!(cond)) {                                            \
            std::fprintf(stderr, "%s:%d: ", __FILE__, __LINE__);  \
            die(__VA_ARGS__);                                     \
        }                                                         \
    } while (0)
#define OK(expr)                                                                \
    do {                                                                        \
        const b40c_status s_ = (expr);                                          \
        REQUIRE(s_ == B40C_OK, "%s returned %d", #expr, (int)s_);               \
    } while (0)

// ---- graphs -----------------------------------------------------------------

struct HostGraph {
    std::string name;
    int32_t n = 0;
    std::vector<int32_t> off, cols;
    int64_t m() const { return (int64_t)cols.size(); }
};

HostGraph make_graph(const std::string& name, int32_t n, std::vector<std::pair<int32_t, int32_t>> edges, bool undirected) {
    if (undirected) {
        const size_t k = edges.size();
        for (size_t i = 0; i < k; ++i) edges.emplace_back(edges[i].second, edges[i].first);
    }
    std::sort(edges.begin(), edges.end());
    edges.erase(std::unique(edges.begin(), edges.end()), edges.end());
    HostGraph g;
    g.name = name;
    g.n = n;
    g.off.assign((size_t)n + 1, 0);
    for (auto& e : edges) ++g.off[(size_t)e.first + 1];
    for (int32_t v = 0; v < n; ++v) g.off[(size_t)v + 1] += g.off[(size_t)v];
    for (auto& e : edges) g.cols.push_back(e.second);
    return g;
}

HostGraph path_graph(int32_t n) {
    std::vector<std::pair<int32_t, int32_t>> e;
    for (int32_t v = 0; v + 1 < n; ++v) e.emplace_back(v, v + 1);
    return make_graph("path" + std::to_string(n), n, e, true);
}
HostGraph star_graph(int32_t leaves) {
    std::vector<std::pair<int32_t, int32_t>> e;
    for (int32_t v = 1; v <= leaves; ++v) e.emplace_back(0, v);
    return make_graph("star" + std::to_string(leaves), leaves + 1, e, true);
}
// A skewed graph of 2^scale vertices: ids drawn bit by bit with P(0) = 0.7.
HostGraph skewed_graph(int scale, int factor, bool undirected, unsigned seed) {
    std::mt19937 rng(seed);
    std::bernoulli_distribution one(0.3);
    std::vector<std::pair<int32_t, int32_t>> e;
    for (int i = 0; i < factor << scale; ++i) {
        int32_t a = 0, b = 0;
        for (int k = 0; k < scale; ++k) {
            a = a * 2 + (one(rng) ? 1 : 0);
            b = b * 2 + (one(rng) ? 1 : 0);
        }
        if (a != b) e.emplace_back(a, b);
    }
    return make_graph((undirected ? "skewed" : "directed") + std::to_string(scale), 1 << scale, e, undirected);
}
HostGraph grid_graph(int32_t w) {
    std::vector<std::pair<int32_t, int32_t>> e;
    auto id = [&](int x, int y, int z) { return (int32_t)(((z * w + y) * w + x) * 2654435761ull % (uint64_t)(w * w * w)); };
    std::set<int32_t> seen;
    for (int z = 0; z < w; ++z)
        for (int y = 0; y < w; ++y)
            for (int x = 0; x < w; ++x) {
                seen.insert(id(x, y, z));
                if (x + 1 < w) e.emplace_back(id(x, y, z), id(x + 1, y, z));
                if (y + 1 < w) e.emplace_back(id(x, y, z), id(x, y + 1, z));
                if (z + 1 < w) e.emplace_back(id(x, y, z), id(x, y, z + 1));
            }
    REQUIRE((int32_t)seen.size() == w * w * w, "grid ids collide");
    return make_graph("grid" + std::to_string(w), w * w * w, e, true);
}

std::vector<int32_t> serial_bfs(const HostGraph& g, int32_t src) {
    std::vector<int32_t> d((size_t)g.n, -1), q{src};
    d[(size_t)src] = 0;
    for (size_t h = 0; h < q.size(); ++h)
        for (int32_t i = g.off[(size_t)q[h]]; i < g.off[(size_t)q[h] + 1]; ++i)
            if (d[(size_t)g.cols[(size_t)i]] < 0) {
                d[(size_t)g.cols[(size_t)i]] = d[(size_t)q[h]] + 1;
                q.push_back(g.cols[(size_t)i]);
            }
    return d;
}

struct DeviceGraph {
    b40c_graph* g = nullptr;
    explicit DeviceGraph(const HostGraph& h) { OK(b40c_graph_from_host_csr(h.n, h.m(), h.off.data(), h.cols.data(), &g)); }
    ~DeviceGraph() { b40c_graph_destroy(g); }
};
struct Problem {
    b40c_problem* p = nullptr;
    explicit Problem(b40c_graph* g) { OK(b40c_problem_create_from_graph(g, 0, &p)); }
    ~Problem() { b40c_problem_destroy(p); }
};
struct Enactor {
    b40c_enactor* e = nullptr;
    explicit Enactor(int32_t strategy, const b40c_tuning* t = nullptr, int32_t instrument = 0) {
        OK(b40c_enactor_create(strategy, instrument, &e));
        if (t) OK(b40c_enactor_set_tuning(e, t));
    }
    ~Enactor() { b40c_enactor_destroy(e); }
};

const char* kStrategies[] = {"expand-contract", "contract-expand", "two-phase", "hybrid", "persistent", "direction-optimizing"};

// Reset and search; labels, predecessors and search depth against the serial search.
void search(const HostGraph& h, b40c_problem* p, b40c_enactor* e, int32_t src, int32_t mode) {
    OK(b40c_problem_reset(p, b40c_enactor_frontier_type(e), 1.3));
    OK(b40c_enact_search(e, p, src, 0, mode));
    std::vector<int32_t> depth((size_t)h.n), pred((size_t)h.n);
    OK(b40c_problem_extract(p, depth.data(), pred.data()));
    const std::vector<int32_t> want = serial_bfs(h, src);
    int32_t deepest = 0;
    for (int32_t v = 0; v < h.n; ++v) {
        REQUIRE(depth[(size_t)v] == want[(size_t)v], "%s source %d: depth[%d] is %d, not %d", h.name.c_str(), src, v,
                depth[(size_t)v], want[(size_t)v]);
        deepest = std::max(deepest, want[(size_t)v]);
        const int32_t u = pred[(size_t)v];
        if (v == src || want[(size_t)v] < 0) {
            REQUIRE(u == (v == src ? -2 : -1), "%s: pred[%d] is %d", h.name.c_str(), v, u);
            continue;
        }
        REQUIRE(u >= 0 && u < h.n && want[(size_t)u] == want[(size_t)v] - 1 &&
                    std::binary_search(h.cols.begin() + h.off[(size_t)u], h.cols.begin() + h.off[(size_t)u + 1], v),
                "%s: pred[%d] is %d", h.name.c_str(), v, u);
    }
    int32_t sd = 0;
    OK(b40c_get_statistics(e, nullptr, &sd, nullptr));
    REQUIRE(sd == deepest + 1, "%s source %d: search depth %d, not %d", h.name.c_str(), src, sd, deepest + 1);
}

std::vector<HostGraph> search_graphs() {
    return {path_graph(1), path_graph(7), star_graph(3000), skewed_graph(9, 8, true, 1), skewed_graph(9, 6, false, 2), grid_graph(7)};
}

// Every strategy and mode on every graph: claims on labels (marks 1) or on the
// bitmask (marks 0), `wgs` persistent workgroups per CU, grid tier from `tier`.
void case_searches(int marks, int wgs, int tier) {
    emu::dev().label_claim_nodes = marks ? 1 << 20 : 0;
    for (const HostGraph& h : search_graphs()) {
        DeviceGraph g(h);
        for (int32_t strategy = 0; strategy < 6; ++strategy)
            for (int32_t mode = 0; mode < 3; ++mode) {
                std::printf("%s %s mode %d\n", h.name.c_str(), kStrategies[strategy], mode);
                std::fflush(stdout);
                Problem p(g.g);
                b40c_tuning t{};
                t.persistent_wgs_per_cu = wgs;
                t.grid_gather_threshold = tier;
                t.saturation_quit = 8;
                t.levels_per_sync = 1 + strategy % 3;
                Enactor e(strategy, &t);
                for (int32_t src : {0, h.n / 2, h.n - 1}) search(h, p.p, e.e, src, mode);
            }
    }
}

// A grid of more than 256 workgroups: the persistent kernel with the shared queue.
void case_wide_persistent() {
    emu::dev().cus = 260;
    emu::dev().resident = 300;
    for (const HostGraph& h : {star_graph(3000), skewed_graph(9, 8, true, 1)}) {
        DeviceGraph g(h);
        Problem p(g.g);
        Enactor e(B40C_EXPAND_CONTRACT);
        search(h, p.p, e.e, 0, B40C_MODE_FUSED);
        const auto& last = emu::dev().launches.back();
        REQUIRE(last.first == "k_fused<FK_TD>" && last.second == 260, "%s with %u workgroups was launched", last.first.c_str(),
                last.second);
    }
}

// Instrumented enactors: the average duty is a share of the workgroups' time,
// whatever launches a search is made of.
void case_duty() {
    for (const HostGraph& h : {skewed_graph(9, 8, true, 1), grid_graph(7), star_graph(3000)}) {
        DeviceGraph g(h);
        for (int32_t strategy = 0; strategy < 6; ++strategy)
            for (int32_t mode = 0; mode < 3; ++mode) {
                Problem p(g.g);
                b40c_tuning t{};
                t.saturation_quit = 4;
                t.grid_gather_threshold = 64;
                Enactor e(strategy, &t, 1);
                search(h, p.p, e.e, 0, mode);
                double duty = 0;
                OK(b40c_get_statistics(e.e, nullptr, nullptr, &duty));
                std::printf("%s %s mode %d: duty %.3f\n", h.name.c_str(), kStrategies[strategy], mode, duty);
                std::fflush(stdout);
                REQUIRE(duty > 0 && duty <= 1, "a duty of %.3f", duty);
            }
    }
}

// Several strategies in turn on one problem: what one leaves behind is not the
// next one's input.  `first_sync` levels per host check for direction-optimizing.
void case_shared_problem(int first_sync) {
    for (const HostGraph& h : {path_graph(5), path_graph(9), skewed_graph(9, 8, true, 1)}) {
        DeviceGraph g(h);
        Problem p(g.g);
        b40c_tuning t{};
        t.levels_per_sync = first_sync;
        Enactor dir(B40C_DIRECTION_OPTIMIZING, &t);
        t.levels_per_sync = 4;
        for (int32_t src : {0, h.n / 2, h.n - 1})
            for (int32_t strategy = 0; strategy < 6; ++strategy)
                for (int32_t mode : {B40C_MODE_ITERATIVE, B40C_MODE_DEFAULT}) {
                    std::printf("%s source %d: direction-optimizing, then %s mode %d\n", h.name.c_str(), src,
                                kStrategies[strategy], mode);
                    std::fflush(stdout);
                    search(h, p.p, dir.e, src, B40C_MODE_DEFAULT);
                    Enactor e(strategy, &t);
                    search(h, p.p, e.e, src, mode);
                }
    }
}

// Contract-expand launches whose first workgroup starts when all the others have
// ended: the search depth does not depend on it.  Vertices 1 and 2 list the same
// 448 sinks, the latter after 128 vertices of its own level, so the last level's
// 1,024 pairs are four tiles and all of the first one's are culled.
void case_late_first_workgroup() {
    std::vector<std::pair<int32_t, int32_t>> e;
    for (int32_t v = 1; v < 131; ++v) e.emplace_back(0, v);
    for (int32_t v = 3; v < 579; ++v) {
        if (v >= 131) e.emplace_back(1, v);
        e.emplace_back(2, v);
    }
    const HostGraph h = make_graph("sinks", 579, e, false);
    std::atomic<int> ended{0};
    b40c_tuning t{};
    t.grid_size = 8;
    emu::dev().on_start = [&](const std::string& k, unsigned id) {
        if (k != "k_phase<PK_CE>" || id != 0) return;
        while (ended.load() < 7) sched_yield();
        ended = 0;
    };
    emu::dev().on_end = [&](const std::string& k, unsigned id) {
        if (k == "k_phase<PK_CE>" && id != 0) ++ended;
    };
    DeviceGraph g(h);
    Problem p(g.g);
    Enactor x(B40C_CONTRACT_EXPAND, &t);
    search(h, p.p, x.e, 0, B40C_MODE_ITERATIVE);
}

// Fewer of the narrow persistent kernel's workgroups fit a CU than of the general
// one's: the grid is sized by the kernel that is launched.
void case_narrow_occupancy() {
    emu::dev().occupancies["k_fused_narrow"] = 1;
    const HostGraph h = skewed_graph(9, 8, true, 1);
    DeviceGraph g(h);
    Problem p(g.g);
    b40c_tuning t{};
    t.persistent_wgs_per_cu = 8;
    for (int grid : {0, 7, 1}) {
        t.grid_size = grid;
        Enactor e(B40C_EXPAND_CONTRACT, &t);
        search(h, p.p, e.e, 0, B40C_MODE_FUSED);
        const auto& last = emu::dev().launches.back();
        REQUIRE(last.first == "k_fused_narrow" && last.second == (grid == 1 ? 1u : 4u), "%s with %u workgroups was launched",
                last.first.c_str(), last.second);
    }
}

// A tuning that is read and set again changes nothing: fields that the caller left
// open, which the library chooses per graph, stay open.
void case_tuning_round_trip() {
    const HostGraph h = grid_graph(7);
    DeviceGraph g(h);
    Problem p(g.g);
    for (int32_t strategy = 0; strategy < 6; ++strategy) {
        Enactor fresh(strategy);
        b40c_tuning t{}, again{};
        OK(b40c_enactor_get_tuning(fresh.e, &t));
        Enactor copy(strategy, &t);
        OK(b40c_enactor_get_tuning(copy.e, &again));
        REQUIRE(std::memcmp(&t, &again, sizeof(t)) == 0, "%s: the tuning read back differs", kStrategies[strategy]);
        const int32_t mode = strategy == B40C_HYBRID ? B40C_MODE_DEFAULT : B40C_MODE_FUSED;
        emu::dev().launches.clear();
        search(h, p.p, fresh.e, 0, mode);
        const auto want = emu::dev().launches;
        emu::dev().launches.clear();
        search(h, p.p, copy.e, 0, mode);
        REQUIRE(emu::dev().launches == want, "%s: other persistent launches", kStrategies[strategy]);
        t = b40c_tuning{};
        t.persistent_wgs_per_cu = 3;
        t.grid_gather_threshold = 100;
        OK(b40c_enactor_set_tuning(copy.e, &t));
        OK(b40c_enactor_get_tuning(copy.e, &again));
        REQUIRE(again.persistent_wgs_per_cu == 3 && again.grid_gather_threshold == 100, "%s: what was set is not reported",
                kStrategies[strategy]);
    }
}

// Queues of less than one entry by the sizing factor: every strategy ends with an
// overflow or, where no frontier is longer than one, with the right labels.
void case_tiny_queues() {
    for (const HostGraph& h : {path_graph(2), path_graph(7), star_graph(20)}) {
        DeviceGraph g(h);
        for (int32_t strategy = 0; strategy < 6; ++strategy)
            for (int32_t mode = 0; mode < 3; ++mode) {
                std::printf("%s %s mode %d\n", h.name.c_str(), kStrategies[strategy], mode);
                std::fflush(stdout);
                Problem p(g.g);
                Enactor e(strategy);
                OK(b40c_problem_reset(p.p, b40c_enactor_frontier_type(e.e), 0.01));
                const b40c_status s = b40c_enact_search(e.e, p.p, 0, 0, mode);
                REQUIRE(s == B40C_OK || s == B40C_ERR_QUEUE_OVERFLOW, "the search returned %d", (int)s);
                if (s != B40C_OK) continue;
                std::vector<int32_t> depth((size_t)h.n);
                OK(b40c_problem_extract(p.p, depth.data(), nullptr));
                REQUIRE(depth == serial_bfs(h, 0), "wrong labels and no overflow");
            }
    }
}

// No memory for the narrow persistent kernel's frontier pieces: the search runs
// the general form.
void case_no_frontier_pieces() {
    const HostGraph h = skewed_graph(9, 8, true, 1);
    DeviceGraph g(h);
    Problem p(g.g);
    Enactor e(B40C_EXPAND_CONTRACT);
    search(h, p.p, e.e, 0, B40C_MODE_ITERATIVE);  // the queues are allocated
    emu::dev().largest_alloc = 200000;
    for (int k = 0; k < 2; ++k) {
        search(h, p.p, e.e, 1, B40C_MODE_FUSED);
        REQUIRE(emu::dev().launches.back().first == "k_fused<FK_TD>", "%s was launched", emu::dev().launches.back().first.c_str());
    }
    emu::dev().largest_alloc = ~(size_t)0;
    search(h, p.p, e.e, 1, B40C_MODE_FUSED);
    REQUIRE(emu::dev().launches.back().first == "k_fused_narrow", "%s was launched", emu::dev().launches.back().first.c_str());
}

// ---- sort, scan, removal, CSR builds -------------------------------------------

template <class T>
struct DeviceArray {
    void* p = nullptr;
    size_t n;
    explicit DeviceArray(size_t k) : n(k) { OK(b40c_device_alloc(&p, (int64_t)(k * sizeof(T)))); }
    explicit DeviceArray(const std::vector<T>& h) : DeviceArray(h.size()) { put(h); }
    DeviceArray(const DeviceArray&) = delete;
    ~DeviceArray() { b40c_device_free(p); }
    void put(const std::vector<T>& h) { OK(b40c_memcpy_h2d(p, h.data(), (int64_t)(h.size() * sizeof(T)))); }
    std::vector<T> get(size_t k) const {
        std::vector<T> h(k);
        OK(b40c_memcpy_d2h(h.data(), p, (int64_t)(k * sizeof(T))));
        return h;
    }
    T* ptr() const { return static_cast<T*>(p); }
};

// Keys whose bits [0, bits) are random; every fifth equals its neighbour.
std::vector<uint64_t> random_keys(size_t n, int bits, unsigned seed) {
    std::mt19937_64 rng(seed);
    std::vector<uint64_t> k(n);
    for (size_t i = 0; i < n; ++i) k[i] = i % 5 == 1 ? k[i - 1] : rng() & (bits == 64 ? ~0ull : (1ull << bits) - 1);
    return k;
}

void sort_u64(size_t n, int bits, b40c_sort_enactor* e = nullptr) {
    std::printf("sort %zu keys of %d bits\n", n, bits);
    std::fflush(stdout);
    std::vector<uint64_t> k = random_keys(n, bits, (unsigned)n);
    DeviceArray<uint64_t> a(k), b(n);
    int32_t sel = -1;
    if (e)
        OK(b40c_sort_enactor_sort(e, B40C_KEY_U64, a.ptr(), b.ptr(), nullptr, nullptr, (int64_t)n, 0, 64, &sel));
    else
        OK(b40c_radix_sort_u64(a.ptr(), b.ptr(), (int64_t)n, 0, 64, &sel));
    std::sort(k.begin(), k.end());
    REQUIRE((sel ? b : a).get(n) == k, "%zu keys are not in order", n);
}

void sort_pairs(size_t n, int bits) {
    std::printf("sort %zu pairs of %d bits\n", n, bits);
    std::fflush(stdout);
    const std::vector<uint64_t> k = random_keys(n, bits, (unsigned)n + 1);
    std::vector<uint32_t> key(k.begin(), k.end()), val(n);
    for (size_t i = 0; i < n; ++i) val[i] = (uint32_t)i;
    DeviceArray<uint32_t> a(key), b(n), va(val), vb(n);
    int32_t sel = -1;
    OK(b40c_radix_sort_pairs_u32(a.ptr(), b.ptr(), va.ptr(), vb.ptr(), (int64_t)n, 0, 32, &sel));
    std::stable_sort(val.begin(), val.end(), [&](uint32_t x, uint32_t y) { return key[x] < key[y]; });
    const std::vector<uint32_t> gk = (sel ? b : a).get(n), gv = (sel ? vb : va).get(n);
    for (size_t i = 0; i < n; ++i)
        REQUIRE(gv[i] == val[i] && gk[i] == key[val[i]], "pair %zu of %zu is wrong", i, n);
}

void case_sorts() {
    for (size_t n : {2, 63, 8192, 8193, 40000}) sort_u64(n, 64);
    for (size_t n : {1000, 9000, 30001}) sort_pairs(n, 20);
}

// A small device that runs 20 workgroups at a time: every block of a place whose
// turn has come can start, whatever the others wait for.
void case_sort_few_resident() {
    emu::dev().resident = 20;
    emu::dev().chain_spins = 30000;
    sort_u64(70 * 4096 + 17, 16);
    sort_pairs(66 * 4096, 8);
}
// The fewest workgroups at a time with which blocks are grouped by XCD.
void case_sort_grouped() {
    emu::dev().cus = 66;
    emu::dev().resident = 66;
    emu::dev().chain_spins = 30000;
    sort_u64(140 * 4096 + 17, 16);
}

// A sort that returns an error after its kernels were launched, then another one:
// the second one's report is its own, though the first one's kernels run late.
void case_sort_after_error() {
    emu::dev().lazy = true;
    b40c_sort_enactor *e = nullptr, *f = nullptr;
    OK(b40c_sort_enactor_create(&e));
    OK(b40c_sort_enactor_create(&f));
    const size_t n = 500;
    const std::vector<uint64_t> one = random_keys(n, 8, 1), two = random_keys(n, 16, 2);
    DeviceArray<uint64_t> a(one), b(n), c(two), d(n);
    int32_t sel = -1;
    sort_u64(n, 8, e);  // the scratch is allocated
    sort_u64(n, 8, f);
    emu::last_error = hipErrorUnknown;
    REQUIRE(b40c_sort_enactor_sort(e, B40C_KEY_U64, a.ptr(), b.ptr(), nullptr, nullptr, (int64_t)n, 0, 64, &sel) == B40C_ERR_HIP,
            "the planted error was not returned");
    OK(b40c_sort_enactor_sort(f, B40C_KEY_U64, c.ptr(), d.ptr(), nullptr, nullptr, (int64_t)n, 0, 64, &sel));
    std::vector<uint64_t> want = two;
    std::sort(want.begin(), want.end());
    REQUIRE((sel ? d : c).get(n) == want, "selector %d is not this sort's", sel);
    b40c_sort_enactor_destroy(e);
    b40c_sort_enactor_destroy(f);
}

// Device memory too short for the scratch that a sort or a build wants: they make
// do with less.
void case_short_of_memory() {
    const size_t n = 1100 * 4096;
    {
        std::vector<uint64_t> k = random_keys(n, 8, 3);
        DeviceArray<uint64_t> a(k), b(n);
        b40c_sort_enactor* e = nullptr;
        OK(b40c_sort_enactor_create(&e));
        emu::dev().largest_alloc = 2200000;
        int32_t sel = -1;
        OK(b40c_radix_sort_u64(a.ptr(), b.ptr(), (int64_t)n, 0, 8, &sel));
        std::vector<uint64_t> want = k;
        std::sort(want.begin(), want.end());
        REQUIRE((sel ? b : a).get(n) == want, "the keys are not in order");
        a.put(k);
        OK(b40c_sort_enactor_sort(e, B40C_KEY_U64, a.ptr(), b.ptr(), nullptr, nullptr, (int64_t)n, 0, 8, &sel));
        REQUIRE((sel ? b : a).get(n) == want, "the enactor's keys are not in order");
        b40c_sort_enactor_destroy(e);
    }
    // A build whose arrays fit but not with the sort's scratch beside them.
    const int32_t m = 140000;
    std::vector<int32_t> r((size_t)m), c((size_t)m);
    for (int32_t i = 0; i < m; ++i) {
        r[(size_t)i] = i / 8;
        c[(size_t)i] = i % 8;
    }
    emu::dev().largest_alloc = (size_t)m * (2 * 8 + 8) + 50000;
    b40c_graph* g = nullptr;
    OK(b40c_graph_from_coo_unique(m / 8, m, r.data(), c.data(), 0, &g));
    int64_t edges = 0;
    OK(b40c_graph_info(g, nullptr, &edges));
    REQUIRE(edges == m, "%lld edges", (long long)edges);
    b40c_graph_destroy(g);
}

void case_primitives() {
    for (size_t n : {1, 1023, 8192, 8193, 50001}) {
        std::printf("scan and removal %zu\n", n);
        std::fflush(stdout);
        const std::vector<uint64_t> k = random_keys(n, 40, (unsigned)n);
        std::vector<uint32_t> x(k.begin(), k.end()), y(n);
        uint64_t sum = 0, total = 0;
        for (size_t i = 0; i < n; ++i) {
            y[i] = (uint32_t)sum;
            sum += x[i];
        }
        DeviceArray<uint32_t> in(x), out(n);
        OK(b40c_scan_u32(in.ptr(), out.ptr(), (int64_t)n, 1, &total));
        REQUIRE(out.get(n) == y && total == sum, "scan of %zu", n);
        DeviceArray<uint64_t> ka(k), kb(n);
        DeviceArray<uint32_t> vb(n);
        int64_t kept = 0;
        OK(b40c_consecutive_removal_u64(ka.ptr(), in.ptr(), kb.ptr(), vb.ptr(), (int64_t)n, &kept));
        std::vector<uint64_t> wk;
        std::vector<uint32_t> wv;
        for (size_t i = 0; i < n; ++i)
            if (i == 0 || k[i] != k[i - 1]) {
                wk.push_back(k[i]);
                wv.push_back(x[i]);
            }
        REQUIRE(kept == (int64_t)wk.size() && kb.get(wk.size()) == wk && vb.get(wk.size()) == wv, "removal of %zu", n);
    }
}

// Calls `f` while the workgroup `late` of every kernel whose name holds `kernel`
// (in the first launch only, or in every one) starts only when a workgroup that
// depends on it has ended, which it does only by giving up waiting: one of the
// serving ones (below `servers`) if `late` is a block, a block if it serves.
// Returns how often that happened.
int with_late_workgroup(const char* kernel, unsigned late, unsigned servers, bool every, const std::function<void()>& f) {
    std::atomic<unsigned> ended{0}, highest{0};
    std::atomic<int> launches{0};
    emu::dev().chain_spins = 50;
    emu::dev().on_start = [&](const std::string& k, unsigned id) {
        if (k.find(kernel) == std::string::npos || id != late) return;
        const unsigned before = (unsigned)launches++;
        if (before && !every) return;
        const unsigned each = late < servers ? highest.load() + 1 - servers : servers;
        while (ended.load() <= before * each) sched_yield();
    };
    emu::dev().on_end = [&](const std::string& k, unsigned id) {
        if (k.find(kernel) == std::string::npos) return;
        for (unsigned h = highest; h < id && !highest.compare_exchange_weak(h, id);) {
        }
        if ((id < servers) != (late < servers)) ++ended;
    };
    f();
    emu::dev().chain_spins = 1u << 14;
    emu::dev().on_start = nullptr;
    emu::dev().on_end = nullptr;
    return launches.load();
}

// Chained calls one of whose blocks starts after the serving workgroup has given
// up: what the others then leave undone is finished.
void case_late_blocks() {
    const size_t n = 9 * 8192 + 77;
    const std::vector<uint64_t> k = random_keys(n, 40, 9);
    std::vector<uint32_t> x(k.begin(), k.end()), y(n);
    uint64_t sum = 0;
    for (size_t i = 0; i < n; ++i) {
        y[i] = (uint32_t)sum;
        sum += x[i];
    }
    std::vector<uint64_t> wk;
    for (size_t i = 0; i < n; ++i)
        if (i == 0 || k[i] != k[i - 1]) wk.push_back(k[i]);
    for (unsigned late : {1u, 2u, 8u}) {
        std::printf("workgroup %u late\n", late);
        std::fflush(stdout);
        DeviceArray<uint32_t> in(x);
        const int scans = with_late_workgroup("k_scan_chained", late, 1, false, [&] {
            uint64_t total = 0;
            OK(b40c_scan_u32(in.ptr(), in.ptr(), (int64_t)n, 1, &total));
            REQUIRE(total == sum, "the total");
        });
        REQUIRE(scans > 0 && in.get(n) == y, "the scan");
        DeviceArray<uint64_t> ka(k), kb(n);
        const int trims = with_late_workgroup("k_trim_chained", late, 1, false, [&] {
            int64_t kept = 0;
            OK(b40c_consecutive_removal_u64(ka.ptr(), nullptr, kb.ptr(), nullptr, (int64_t)n, &kept));
            REQUIRE(kept == (int64_t)wk.size(), "%lld kept", (long long)kept);
        });
        REQUIRE(trims > 0 && kb.get(wk.size()) == wk, "the removal");
        const HostGraph h = skewed_graph(12, 12, false, 3);
        std::vector<int32_t> r, off((size_t)h.n + 1), cols((size_t)h.m());
        for (int32_t v = 0; v < h.n; ++v) r.insert(r.end(), (size_t)(h.off[(size_t)v + 1] - h.off[(size_t)v]), v);
        b40c_graph* g = nullptr;
        const int builds = with_late_workgroup("k_csr_chained", late, 1, false, [&] {
            OK(b40c_graph_from_coo_unique(h.n, h.m(), r.data(), h.cols.data(), 0, &g));
        });
        OK(b40c_graph_copy_to_host(g, off.data(), cols.data()));
        REQUIRE(builds > 0 && off == h.off && cols == h.cols, "the CSR");
        b40c_graph_destroy(g);
    }
}

// Sorts one of whose workgroups starts in each place only after those that need it
// have given up: a block or a serving workgroup, with blocks of one tile and of
// several, with values, and in the fixed scratch.
void case_late_sorts() {
    const char* place = "k_place<K, CONV, VALS, ITEMS, false>";
    for (unsigned late : {16u, 17u, 19u, 3u}) {
        std::printf("workgroup %u late\n", late);
        std::fflush(stdout);
        const int places = with_late_workgroup(place, late, 16, true, [] { sort_u64(20000, 64); });
        REQUIRE(places > 8, "%d launches of places", places);
        REQUIRE(with_late_workgroup(place, late, 16, true, [] { sort_pairs(20000, 20); }) > 3, "no place was late");
        b40c_sort_enactor* e = nullptr;
        OK(b40c_sort_enactor_create(&e));
        OK(b40c_sort_enactor_set_policy(e, 8, 1));
        REQUIRE(with_late_workgroup(place, late, 16, true, [&] { sort_u64(70000, 40, e); }) > 5, "no place was late");
        sort_u64(70000, 40, e);
        b40c_sort_enactor_destroy(e);
        const size_t n = 30011;
        std::vector<uint64_t> k = random_keys(n, 12, 3);
        DeviceArray<uint64_t> a(k), b(n);
        int32_t sel = -1;
        with_late_workgroup(place, late, 16, true,
                            [&] { OK(b40c_radix_sort_u64_noalloc(a.ptr(), b.ptr(), (int64_t)n, 0, 12, &sel)); });
        std::sort(k.begin(), k.end());
        REQUIRE((sel ? b : a).get(n) == k, "the sort in the fixed scratch");
    }
}

// Scans of several launches: whole and partial last blocks and segments.
void case_scan_segments() {
    const size_t block = 8192;
    for (size_t blocks : {1, 3}) {
        emu::dev().scan_segment = (long long)(blocks * block);
        for (size_t n : {block, blocks * block, blocks * block + 1, 2 * blocks * block - 1, 2 * blocks * block, 7 * block + 5}) {
            std::printf("scan %zu in segments of %zu blocks\n", n, blocks);
            std::fflush(stdout);
            const std::vector<uint64_t> k = random_keys(n, 32, (unsigned)n);
            std::vector<uint32_t> x(k.begin(), k.end()), excl(n), incl(n);
            uint64_t sum = 0, total = 0;
            for (size_t i = 0; i < n; ++i) {
                excl[i] = (uint32_t)sum;
                sum += x[i];
                incl[i] = (uint32_t)sum;
            }
            DeviceArray<uint32_t> in(x), out(n);
            OK(b40c_scan_u32(in.ptr(), out.ptr(), (int64_t)n, 1, &total));
            REQUIRE(out.get(n) == excl && total == sum, "exclusive scan");
            OK(b40c_scan_u32(in.ptr(), in.ptr(), (int64_t)n, 0, &total));
            REQUIRE(in.get(n) == incl && total == sum, "inclusive scan in place");
        }
    }
}

void case_builds() {
    for (const HostGraph& h : {path_graph(7), star_graph(3000), skewed_graph(11, 6, false, 3)}) {
        std::printf("build %s\n", h.name.c_str());
        std::fflush(stdout);
        std::vector<int32_t> r, c;
        for (int32_t v = 0; v < h.n; ++v)
            for (int32_t i = h.off[(size_t)v]; i < h.off[(size_t)v + 1]; ++i) {
                r.push_back(v);
                c.push_back(h.cols[(size_t)i]);
                if (i % 3 == 0) {
                    r.push_back(v);
                    c.push_back(h.cols[(size_t)i]);
                }
            }
        for (size_t i = r.size(); i > 1; --i) {
            const size_t j = (i * 2654435761u) % i;
            std::swap(r[i - 1], r[j]);
            std::swap(c[i - 1], c[j]);
        }
        b40c_graph* g = nullptr;
        OK(b40c_graph_from_coo_unique(h.n, (int64_t)r.size(), r.data(), c.data(), 0, &g));
        int32_t n = 0;
        int64_t m = 0;
        OK(b40c_graph_info(g, &n, &m));
        REQUIRE(n == h.n && m == h.m(), "%d vertices and %lld edges", n, (long long)m);
        std::vector<int32_t> off((size_t)n + 1), cols((size_t)m);
        OK(b40c_graph_copy_to_host(g, off.data(), cols.data()));
        REQUIRE(off == h.off && cols == h.cols, "the CSR differs");
        b40c_graph_destroy(g);
        r[r.size() / 2] = h.n;
        REQUIRE(b40c_graph_from_coo_unique(h.n, (int64_t)r.size(), r.data(), c.data(), 0, &g) == B40C_ERR_INVALID_ARG,
                "an id outside the graph was accepted");
    }
    b40c_graph* g = nullptr;
    OK(b40c_graph_build_rmat(10, 8, 0.57, 0.19, 0.19, 1, &g));
    b40c_graph_destroy(g);
    OK(b40c_graph_build_lattice3d(9, 1, nullptr, &g));
    b40c_graph_destroy(g);
}

// ---- batched queries -----------------------------------------------------------

void case_batched(int levels, int persistent) {
    const std::vector<HostGraph> hs = {path_graph(9), star_graph(700), skewed_graph(9, 8, true, 1), grid_graph(6)};
    std::vector<b40c_graph*> gs;
    for (const HostGraph& h : hs) {
        b40c_graph* g = nullptr;
        OK(b40c_graph_from_host_csr(h.n, h.m(), h.off.data(), h.cols.data(), &g));
        gs.push_back(g);
    }
    b40c_multigraph* mg = nullptr;
    OK(b40c_multigraph_pack(gs.data(), (int32_t)gs.size(), &mg));
    for (b40c_graph* g : gs) b40c_graph_destroy(g);
    b40c_msbfs* m = nullptr;
    OK(b40c_msbfs_create(mg, 1 << 22, 256, &m));
    OK(b40c_msbfs_set_levels_per_step(m, levels));
    OK(b40c_msbfs_set_persistent(m, persistent));
    std::vector<std::pair<int, int32_t>> asked;
    std::vector<int32_t> ids;
    for (int k = 0; k < 40; ++k) {
        const int gi = k % (int)hs.size();
        const int32_t src = (int32_t)((k * 37) % hs[(size_t)gi].n);
        int32_t id = -1;
        OK(b40c_msbfs_submit(m, gi, src, &id));
        asked.emplace_back(gi, src);
        ids.push_back(id);
    }
    OK(b40c_msbfs_run(m));
    std::printf("batched: %d levels a step, persistent %d: run\n", levels, persistent);
    std::fflush(stdout);
    for (size_t k = 0; k < ids.size(); ++k) {
        const size_t q = k < 20 ? k : ids.size() - 1 - (k - 20);  // in order, then from the end
        const HostGraph& h = hs[(size_t)asked[q].first];
        std::vector<int32_t> depth((size_t)h.n), pred((size_t)h.n);
        int32_t sd = 0;
        OK(b40c_msbfs_result(m, ids[q], depth.data(), q % 3 ? pred.data() : nullptr, &sd));
        const std::vector<int32_t> want = serial_bfs(h, asked[q].second);
        REQUIRE(depth == want, "query %zu on %s", q, h.name.c_str());
        for (int32_t v = 0; q % 3 && v < h.n; ++v)
            if (v != asked[q].second && want[(size_t)v] >= 0)
                REQUIRE(pred[(size_t)v] >= 0 && want[(size_t)pred[(size_t)v]] == want[(size_t)v] - 1, "query %zu pred[%d]", q, v);
    }
    b40c_msbfs_destroy(m);
    b40c_multigraph_destroy(mg);
}

// Which results are copied out: in the order of submission many at a time, in
// other orders none that is not asked for next.  One workgroup per query copied.
void case_result_orders() {
    const HostGraph h = skewed_graph(8, 8, true, 1);
    DeviceGraph g(h);
    b40c_multigraph* mg = nullptr;
    OK(b40c_multigraph_pack(&g.g, 1, &mg));
    const int Q = 60;
    for (const char* form : {"submitted", "reversed", "evens first", "shuffled"}) {
        b40c_msbfs* m = nullptr;
        OK(b40c_msbfs_create(mg, 1 << 22, Q, &m));
        std::vector<int32_t> ids((size_t)Q), take;
        for (int k = 0; k < Q; ++k) OK(b40c_msbfs_submit(m, 0, k, &ids[(size_t)k]));
        OK(b40c_msbfs_run(m));
        for (int k = 0; k < Q; ++k) take.push_back(form[0] == 'r' ? Q - 1 - k : form[0] == 'e' ? (2 * k < Q ? 2 * k : 2 * k - Q + 1) : k);
        if (form[1] == 'h') std::shuffle(take.begin(), take.end(), std::mt19937(1));
        std::atomic<int> copied{0}, launches{0};
        emu::dev().on_start = [&](const std::string& k, unsigned id) {
            if (k != "k_ms_stage") return;
            ++copied;
            if (id == 0) ++launches;
        };
        for (int32_t k : take) {
            std::vector<int32_t> depth((size_t)h.n);
            OK(b40c_msbfs_result(m, ids[(size_t)k], depth.data(), nullptr, nullptr));
            REQUIRE(depth == serial_bfs(h, k), "query %d", k);
        }
        std::printf("%s: %d copied by %d launches\n", form, copied.load(), launches.load());
        std::fflush(stdout);
        if (form[0] == 's' && form[1] == 'u') {
            REQUIRE(copied == Q && launches <= 7, "more copies or launches than a doubling window takes");
            // The next batch goes on with the window learnt.
            launches = 0;
            for (int k = 0; k < Q; ++k) OK(b40c_msbfs_submit(m, 0, k, &ids[(size_t)k]));
            OK(b40c_msbfs_run(m));
            for (int k = 0; k < Q; ++k) OK(b40c_msbfs_result(m, ids[(size_t)k], std::vector<int32_t>((size_t)h.n).data(), nullptr, nullptr));
            REQUIRE(launches <= 2, "%d launches for a second batch", launches.load());
        } else {
            REQUIRE(copied <= Q + Q / 10, "results were copied that were not asked for next");
        }
        emu::dev().on_start = nullptr;
        b40c_msbfs_destroy(m);
    }
    b40c_multigraph_destroy(mg);
}

}  // namespace

int main(int argc, char** argv) {
    if (argc < 2) return 2;
    const std::string name = argv[1];
    auto arg = [&](int i) {
        REQUIRE(argc > 2 + i, "%s wants more arguments", name.c_str());
        return std::atoi(argv[2 + i]);
    };
    if (name == "searches")
        case_searches(arg(0), arg(1), arg(2));
    else if (name == "wide_persistent")
        case_wide_persistent();
    else if (name == "late_first_workgroup")
        case_late_first_workgroup();
    else if (name == "narrow_occupancy")
        case_narrow_occupancy();
    else if (name == "tuning_round_trip")
        case_tuning_round_trip();
    else if (name == "no_frontier_pieces")
        case_no_frontier_pieces();
    else if (name == "tiny_queues")
        case_tiny_queues();
    else if (name == "duty")
        case_duty();
    else if (name == "shared_problem")
        case_shared_problem(arg(0));
    else if (name == "sorts")
        case_sorts();
    else if (name == "sort_few_resident")
        case_sort_few_resident();
    else if (name == "sort_grouped")
        case_sort_grouped();
    else if (name == "sort_after_error")
        case_sort_after_error();
    else if (name == "short_of_memory")
        case_short_of_memory();
    else if (name == "primitives")
        case_primitives();
    else if (name == "late_blocks")
        case_late_blocks();
    else if (name == "late_sorts")
        case_late_sorts();
    else if (name == "scan_segments")
        case_scan_segments();
    else if (name == "builds")
        case_builds();
    else if (name == "result_orders")
        case_result_orders();
    else if (name == "batched")
        case_batched(arg(0), arg(1));
    else
        die("unknown case %s", name.c_str());
    std::printf("ok\n");
    std::fflush(nullptr);
    _Exit(0);  // the workgroup threads never end
}
