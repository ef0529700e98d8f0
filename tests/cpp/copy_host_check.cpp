// The host side of copy plans against a HIP runtime made for it: what a plan asks of the runtime, in which
// order, and what it answers when a launch is late, lost or seen by another thread.  The functions below
// stand before those of libamdhip64 in the process; no GPU is used.  Memory is the host's, kernels are
// known by their names, and those that the host waits for do what it waits for.
//
// usage: copy_host_check <scenario>; prints "OK" and exits 0 on success.
#include <hip/hip_runtime_api.h>
#include <signal.h>
#include <sys/mman.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <memory>
#include <mutex>
#include <numeric>
#include <set>
#include <string>
#include <thread>
#include <tuple>
#include <utility>
#include <vector>

#include "nixl_amd_hip.h"

#define REQUIRE(cond)                                                          \
    do {                                                                       \
        if (!(cond)) {                                                         \
            std::fprintf(stderr, "%s:%d: %s failed (%s)\n", __FILE__, __LINE__, #cond, nixl_amd_last_error()); \
            std::exit(1);                                                      \
        }                                                                      \
    } while (0)

namespace {

// ---- streams and events -----------------------------------------------------------------------

// Work runs when it is queued, or, on a stream that is held, when that is let go.
struct Stream {
    std::deque<std::function<void()>> work;
    bool held = false;
    bool waited_for = false; // by the host
    hipError_t failure = hipSuccess; // what was queued does not run any more
    std::vector<std::string> kernels; // launched on it

    void
    queue(std::function<void()> w) {
        if (held)
            work.push_back(std::move(w));
        else
            w();
    }

    void
    let_go() {
        if (failure != hipSuccess) return;
        held = false;
        for (; !work.empty(); work.pop_front())
            work.front()();
    }
};

struct Event {
    std::shared_ptr<bool> done = std::make_shared<bool>(true);
    Stream *on = nullptr;
};

std::recursive_mutex g_lock;
hipError_t g_launch_status = hipSuccess; // of one launch,
int g_good_launches = 0; // behind so many that are accepted
int g_refused_pinned = 0; // allocations of pinned memory that fail from here on
std::vector<size_t> g_pinned; // those asked for
int g_refused_device = 0; // allocations of device memory that fail from here on
bool g_only_relaxed = false; // such allocations would end another stream's capture
thread_local hipStreamCaptureMode t_mode = hipStreamCaptureModeGlobal;
void (*g_synchronized)(Stream &) = nullptr; // in front of a wait for a stream
Stream *g_created = nullptr; // the last stream that the library made

Stream &
stream_of(hipStream_t s) {
    static Stream of_all;
    static thread_local Stream of_thread;
    if (!s || s == hipStreamLegacy) return of_all;
    if (s == hipStreamPerThread) return of_thread;
    return *reinterpret_cast<Stream *>(s);
}

Event &
event_of(hipEvent_t e) {
    return *reinterpret_cast<Event *>(e);
}

// ---- kernels ----------------------------------------------------------------------------------

std::map<const void *, std::string> &
kernel_names() {
    static std::map<const void *, std::string> names;
    return names;
}

std::map<const void *, void *> &
device_variables() {
    static std::map<const void *, void *> variables;
    return variables;
}

// The arguments of the kernels that the host waits for, as copy_kernels.hip declares them.
struct Done {
    uint32_t *counts, *word;
    uint32_t value;
};

struct ListTotals {
    unsigned long long bytes_arrived;
    alignas(128) unsigned long long extra_continued;
    uint32_t bad;
};
static_assert(sizeof(ListTotals) == 256);

struct ListVerdict {
    unsigned long long bytes;
    uint32_t bad, continued, extra, there;
};

struct ListArgs {
    void *recs;
    const nixl_amd_copy_list_entry_t *src, *dst;
    uint32_t n_src, n_dst;
    const int32_t *src_index, *dst_index;
    const void *runs;
    const uint32_t *run_of;
    uint32_t first_workgroup, n, n_workgroups;
    ListTotals *totals;
    ListVerdict *verdict;
};

std::set<ListTotals *> g_totals; // that requests have counted in

// Of the copies whose indices repeat themselves.
struct GridIndices {
    struct Side {
        uint64_t base, stride;
        uint32_t first, step, listed, place;
    } src, dst;
    uint32_t row_length[4]; // the number itself, and how to divide by it
    uint32_t by_column, ids[1792 / 2];

    uint64_t
    address(const Side &s, uint32_t r) const {
        const uint32_t row = r / row_length[0], column = r % row_length[0];
        if (!s.listed) return s.base + static_cast<uint64_t>(s.first + r) * s.stride;
        const uint32_t i = s.place + (by_column ? column : row);
        REQUIRE(i < 1792);
        const uint32_t id = i % 2 ? ids[i / 2] >> 16 : ids[i / 2] & 0xffffu;
        return s.base + static_cast<uint64_t>(s.first + id + (by_column ? row : column) * s.step) * s.stride;
    }
};

std::unique_ptr<GridIndices> g_grid; // of the last such launch

std::function<void()>
work_of(const std::string &kernel, dim3 grid, void **args) {
    const auto is = [&](const char *name) { return kernel.find(name) != std::string::npos; };
    if (is("GridIndices")) g_grid = std::make_unique<GridIndices>(*static_cast<GridIndices *>(args[0]));
    if (is("copy_inline_done_kernel")) {
        const Done done = *static_cast<Done *>(args[3]);
        return [done] { *done.word = done.value; };
    }
    if (is("done_kernel")) {
        uint32_t *const word = *static_cast<uint32_t **>(args[0]);
        const uint32_t value = *static_cast<uint32_t *>(args[1]);
        return [word, value] { *word = value; };
    }
    if (is("clear_totals_kernel")) {
        auto *const totals = *static_cast<ListTotals **>(args[0]);
        return [totals] { *totals = ListTotals{}; };
    }
    if (is("list_records_kernel")) {
        const ListArgs a = *static_cast<ListArgs *>(args[0]);
        g_totals.insert(a.totals);
        return [a, grid] {
            ListTotals &t = *a.totals;
            if (a.first_workgroup == 0) REQUIRE(t.bytes_arrived == 0 && t.extra_continued == 0 && t.bad == 0); // nothing of an earlier request's
            t.bytes_arrived += grid.x;
            t.extra_continued += 3 * grid.x;
            t.bad += 7 * grid.x;
            if (t.bytes_arrived != a.n_workgroups) return;
            REQUIRE(t.extra_continued == 3 * a.n_workgroups && t.bad == 7 * a.n_workgroups);
            *a.totals = ListTotals{};
            a.verdict->bytes = a.n;
            a.verdict->there = 1;
        };
    }
    return [] {};
}

// ---- what a scenario looks at -----------------------------------------------------------------

int
launched(const Stream &s, const char *kernel) {
    int n = 0;
    for (const std::string &name : s.kernels)
        n += name.find(kernel) != std::string::npos;
    return n;
}

hipStream_t
handle(Stream &s) {
    return reinterpret_cast<hipStream_t>(&s);
}

nixl_amd_copy_tuning_t
tuning_for(Stream &s) {
    nixl_amd_copy_tuning_t t{};
    t.stream = &s;
    return t;
}

// A plan of one block, launched and watched on `s` (it tells its end itself).
nixl_amd_copy_plan_t *
block_plan() {
    alignas(128) static uint8_t from[8192], to[8192];
    const nixl_amd_copy_desc_t desc{reinterpret_cast<uintptr_t>(from), reinterpret_cast<uintptr_t>(to), sizeof(from)};
    nixl_amd_copy_plan_t *plan = nullptr;
    REQUIRE(nixl_amd_copy_plan_create(&desc, 1, 0, nullptr, &plan) == 0);
    return plan;
}

// Two lists on the device with entries of equal lengths, and pairs that name them.
struct Lists {
    static constexpr size_t kEntries = 2000;
    std::vector<uint8_t> memory = std::vector<uint8_t>(kEntries * 256);
    nixl_amd_copy_list_t *src = nullptr, *dst = nullptr;
    std::vector<int32_t> index = std::vector<int32_t>(kEntries);

    Lists() {
        std::iota(index.begin(), index.end(), 0);
        std::vector<nixl_amd_copy_list_entry_t> table(kEntries);
        for (size_t i = 0; i < kEntries; ++i) {
            table[i] = {};
            table[i].addr = reinterpret_cast<uintptr_t>(memory.data()) + i * 256;
            table[i].len = 256;
        }
        REQUIRE(nixl_amd_copy_list_create(table.data(), kEntries, 0, &src) == 0);
        REQUIRE(nixl_amd_copy_list_create(table.data(), kEntries, 0, &dst) == 0);
    }

    ~Lists() {
        (void)nixl_amd_copy_list_destroy(src);
        (void)nixl_amd_copy_list_destroy(dst);
    }

    int
    request(const nixl_amd_copy_tuning_t *tuning, nixl_amd_copy_plan_t **plan) {
        size_t continued = 0;
        return nixl_amd_copy_plan_create_listed_on(src, index.data(), dst, index.data(), index.size(), tuning, &continued, plan);
    }
};

// ---- scenarios --------------------------------------------------------------------------------

// A caller's stream whose last watched transfer has been seen done and that has other work of the
// caller's since then: a plan made for it is written elsewhere, and a request against
// device-resident lists does not wait for that work.  On a stream that the caller keeps for
// transfers the word answers.
void
work_behind_a_watched_launch() {
    REQUIRE(nixl_amd_copy_watch_prepare() == 0);
    Lists lists;
    for (const bool own : {false, true}) {
        Stream s;
        if (own) REQUIRE(nixl_amd_copy_watch_stream(0, &s, 1) == 0);
        const nixl_amd_copy_tuning_t tuning = tuning_for(s);
        nixl_amd_copy_plan_t *first = block_plan();
        REQUIRE(nixl_amd_copy_plan_launch_watched(first, &s) == 0);
        REQUIRE(nixl_amd_copy_plan_status(first, 0) == 0);
        nixl_amd_copy_plan_t *request = nullptr;
        if (!own) {
            s.held = true;
            s.queue([] {}); // the caller's
        }
        REQUIRE(lists.request(&tuning, &request) == 0);
        REQUIRE(!s.waited_for);
        REQUIRE(launched(s, "list_records_kernel") == (own ? 1 : 0));
        s.let_go();
        REQUIRE(nixl_amd_copy_plan_launch_watched(request, &s) == 0);
        REQUIRE(nixl_amd_copy_plan_status(request, 1) == 0);
        REQUIRE(nixl_amd_copy_plan_destroy(request) == 0);
        REQUIRE(nixl_amd_copy_plan_destroy(first) == 0);
        if (own) { // and not while that transfer runs, nor when the stream is no longer kept for them
            s.held = true;
            first = block_plan();
            REQUIRE(nixl_amd_copy_plan_launch_watched(first, &s) == 0);
            REQUIRE(lists.request(&tuning, &request) == 0);
            REQUIRE(launched(s, "list_records_kernel") == 1);
            s.let_go();
            REQUIRE(nixl_amd_copy_plan_status(first, 0) == 0);
            REQUIRE(nixl_amd_copy_plan_destroy(first) == 0);
            REQUIRE(nixl_amd_copy_plan_destroy(request) == 0);
            REQUIRE(nixl_amd_copy_watch_stream(0, &s, 0) == 0);
            s.held = true;
            s.queue([] {});
            REQUIRE(lists.request(&tuning, &request) == 0);
            REQUIRE(launched(s, "list_records_kernel") == 1 && !s.waited_for);
            REQUIRE(nixl_amd_copy_plan_destroy(request) == 0);
            s.let_go();
        }
    }
    for (void *shared : {static_cast<void *>(nullptr), static_cast<void *>(hipStreamLegacy), static_cast<void *>(hipStreamPerThread)})
        REQUIRE(nixl_amd_copy_watch_stream(0, shared, 1) == NIXL_AMD_ERR_INVALID);
}

// Requests by index whose vectors repeat themselves, listed by column or by row, on one side or both, and such with
// one index changed: the addresses that a copy is told are those of the indices, and what it is told so or by records.
void
indices_that_repeat_themselves() {
    constexpr uintptr_t kSrc = 1ull << 40, kDst = 1ull << 41;
    uint32_t seed = 1;
    const auto random = [&](uint32_t below) { return ((seed = seed * 1664525u + 1013904223u) >> 8) % below; };
    Stream s;
    const auto made = [&](const std::vector<int32_t> &src, const std::vector<int32_t> &dst, uint64_t entries, int sort = 0, uint64_t len = 1024) {
        const nixl_amd_copy_run_t src_run{kSrc, len, 0, entries}, dst_run{kDst, 2 * len, 0, entries};
        nixl_amd_copy_tuning_t tuning = tuning_for(s);
        tuning.sort_scatter = sort;
        nixl_amd_copy_plan_t *plan = nullptr;
        const int rc = nixl_amd_copy_plan_create_indexed_lists(&src_run, 1, src.data(), entries, &dst_run, 1, dst.data(), entries, src.size(), len,
                                                               0, &tuning, &plan);
        if (rc) return rc;
        g_grid.reset();
        REQUIRE(nixl_amd_copy_plan_launch(plan, &s) == 0);
        REQUIRE(nixl_amd_copy_plan_status(plan, 1) == 0);
        if (g_grid)
            for (uint32_t r = 0; r < src.size(); ++r) {
                REQUIRE(g_grid->address(g_grid->src, r) == kSrc + static_cast<uint64_t>(src[r]) * len);
                REQUIRE(g_grid->address(g_grid->dst, r) == kDst + static_cast<uint64_t>(dst[r]) * 2 * len);
            }
        REQUIRE(nixl_amd_copy_plan_destroy(plan) == 0);
        return 0;
    };
    const uint32_t shapes[][2] = {{225, 4}, {64, 15}, {130, 7}, {130, 8}, {900, 17}, {3, 65535}, {3, 65536}, {3, 299}, {3, 300}, {250, 61}, {896, 2}, {897, 2}, {1791, 3}, {1792, 3}, {1793, 3}, {7, 1000}, {150, 3}};
    for (const auto &[n_ids, others] : shapes)
        for (const bool by_column : {true, false})
            for (const int sides : {1, 2, 3}) // listed: the source, the destination, both
                for (const uint32_t range : {3000u, 65536u, 65537u}) {
                    const size_t n = static_cast<size_t>(n_ids) * others;
                    if (static_cast<uint64_t>(range + 150) * others > INT32_MAX) continue;
                    std::vector<int32_t> v[2];
                    uint64_t entries = 0;
                    for (int side = 0; side < 2; ++side) {
                        std::vector<uint32_t> ids(n_ids);
                        for (uint32_t &id : ids)
                            id = random(range);
                        ids[0] = 5; // neither even steps, nor all from one id on
                        ids[1] = 0;
                        ids[2] = range - 1;
                        const uint32_t step = range + random(100), first = random(50);
                        v[side].resize(n);
                        for (size_t r = 0; r < n; ++r) {
                            const size_t length = by_column ? n_ids : others, row = r / length, column = r % length;
                            v[side][r] = static_cast<int32_t>(!(sides >> side & 1) ? first + r :
                                                              by_column            ? first + ids[column] + row * step :
                                                                                     first + ids[row] + column * step);
                            entries = std::max(entries, static_cast<uint64_t>(v[side][r]) + 1);
                        }
                    }
                    const bool fits = range <= 65536 && n_ids * (sides == 3 ? 2 : 1) <= 1792 && (by_column ? others <= 65535 : others >= 8), few = n <= 896 && sides != 3;
                    REQUIRE(made(v[0], v[1], entries) == 0);
                    REQUIRE((g_grid != nullptr) == (fits && !few && n > 448));
                    REQUIRE(made(v[0], v[1], entries - 1) == NIXL_AMD_ERR_INDEX);
                    for (const size_t at : {size_t(0), size_t(n_ids), n / 2, n - 1}) // one that breaks it
                        for (int side = 0; side < 2; ++side) {
                            auto changed = v[side];
                            std::swap(changed, v[side]);
                            v[side][at] ^= 1;
                            REQUIRE(made(v[0], v[1], entries + 1) == 0);
                            REQUIRE(g_grid == nullptr);
                            v[side][at] = -1;
                            REQUIRE(made(v[0], v[1], entries) == NIXL_AMD_ERR_INDEX);
                            v[side] = changed;
                        }
                    s.kernels.clear();
                    REQUIRE(made(v[0], v[1], entries, 1) == 0); // what is to be sorted has records
                    const bool sorted = launched(s, "index_records_kernelILb1E") != 0;
                    REQUIRE(!sorted || !g_grid);
                    if (n >= 1024 && sides == 2 && by_column) REQUIRE(sorted);
                }
    // listed by row, large blocks of more than half a GiB and many that are neighbours have records
    for (const auto &[rows, length, step, len, grid] : std::vector<std::tuple<int, int, int, uint64_t, bool>>{
             {256, 128, 700, 16384, true}, {256, 128, 700, 17408, false}, {64, 512, 700, 16384, true}, {64, 512, 700, 32768, false},
             {32, 512, 700, 32768, true}, {768, 16, 1, 8192, true}, {769, 16, 1, 8192, false}}) {
        std::vector<int32_t> listed(static_cast<size_t>(rows) * length), flat(listed.size());
        std::iota(flat.begin(), flat.end(), 0);
        for (size_t r = 0; r < listed.size(); ++r) // every other place, in an order of its own
            listed[r] = static_cast<int32_t>((r / length * 5 % rows) * (step == 1 ? 2 * length : 2) + r % length * step);
        REQUIRE(made(listed, flat, 1u << 30, 0, len) == 0);
        REQUIRE((g_grid != nullptr) == grid);
    }
    // a scatter of more than half a GiB is sorted if its blocks are large
    std::vector<int32_t> by_column(700 * 64), flat(by_column.size());
    std::iota(flat.begin(), flat.end(), 0);
    for (size_t r = 0; r < by_column.size(); ++r)
        by_column[r] = static_cast<int32_t>((r % 700) * (r % 700) % 701 + r / 700 * 800);
    for (const uint64_t len : {11264u, 12288u, 15360u, 16384u}) {
        s.kernels.clear();
        REQUIRE(made(flat, by_column, 1u << 30, 0, len) == 0);
        REQUIRE((g_grid != nullptr) == (len < 16384));
        REQUIRE((launched(s, "index_records_kernelILb1E") != 0) == (len >= 16384));
    }
}

// A watched launch that fails is reported, whatever stream it went to: by a status that is polled
// (the runtime is asked now and then), and by one that waits.
nixl_amd_copy_plan_t *
launch_fails(hipStream_t stream) {
    REQUIRE(nixl_amd_copy_watch_prepare() == 0);
    Stream &s = stream_of(stream);
    nixl_amd_copy_plan_t *plan = block_plan();
    s.held = true;
    REQUIRE(nixl_amd_copy_plan_launch_watched(plan, stream) == 0);
    for (int i = 0; i < 10000; ++i)
        REQUIRE(nixl_amd_copy_plan_status(plan, 0) == NIXL_AMD_ERR_BUSY); // it is late, no more
    s.failure = hipErrorLaunchFailure;
    int rc = NIXL_AMD_ERR_BUSY;
    for (int i = 0; i < 10000 && rc == NIXL_AMD_ERR_BUSY; ++i)
        rc = nixl_amd_copy_plan_status(plan, 0);
    REQUIRE(rc == NIXL_AMD_ERR_HIP);
    REQUIRE(nixl_amd_copy_plan_status(plan, 1) == NIXL_AMD_ERR_HIP);
    for (int i = 0; i < 10; ++i)
        REQUIRE(nixl_amd_copy_plan_status(plan, 0) == NIXL_AMD_ERR_HIP); // and stays so
    return plan;
}

void
launch_on_a_named_stream_fails() {
    Stream s, good;
    nixl_amd_copy_plan_t *plan = launch_fails(handle(s));
    g_launch_status = hipErrorOutOfMemory; // a launch that is refused changes nothing
    REQUIRE(nixl_amd_copy_plan_launch_watched(plan, &good) == NIXL_AMD_ERR_HIP);
    REQUIRE(nixl_amd_copy_plan_status(plan, 0) == NIXL_AMD_ERR_HIP);
    for (const bool watched : {true, false}) { // another launch does
        REQUIRE((watched ? nixl_amd_copy_plan_launch_watched : nixl_amd_copy_plan_launch)(plan, &good) == 0);
        REQUIRE(nixl_amd_copy_plan_status(plan, 0) == 0);
        REQUIRE(nixl_amd_copy_plan_destroy(plan) == 0);
        Stream bad;
        plan = launch_fails(handle(bad));
    }
    REQUIRE(nixl_amd_copy_plan_destroy(plan) == 0); // nothing runs that would read its arrays
}

void
launch_on_the_legacy_stream_fails() {
    REQUIRE(nixl_amd_copy_plan_destroy(launch_fails(nullptr)) == 0);
    stream_of(nullptr) = {};
    REQUIRE(nixl_amd_copy_plan_destroy(launch_fails(hipStreamLegacy)) == 0);
}

// A watched launch on one thread's per-thread stream, asked for from another thread: late is not failed.
void
launch_on_the_stream_of_a_thread() {
    REQUIRE(nixl_amd_copy_watch_prepare() == 0);
    Stream &s = stream_of(hipStreamPerThread);
    nixl_amd_copy_plan_t *plan = block_plan();
    s.held = true;
    REQUIRE(nixl_amd_copy_plan_launch_watched(plan, hipStreamPerThread) == 0);
    std::thread([&] {
        for (int i = 0; i < 10000; ++i)
            REQUIRE(nixl_amd_copy_plan_status(plan, 0) == NIXL_AMD_ERR_BUSY);
    }).join();
    s.let_go();
    REQUIRE(nixl_amd_copy_plan_status(plan, 0) == 0);
    REQUIRE(nixl_amd_copy_plan_destroy(plan) == 0);
}

// Two threads ask for one launch, as a progress thread and a caller do.  While the first is about to
// look at the word after it has asked the stream, the second sees the end and gives the word back, and another
// launch takes it and ends.  The moment is that of the read itself: the page is taken away when the
// stream is asked, and the fault is where the second thread runs.
void (*g_asked)(hipStream_t) = nullptr; // when the runtime is asked for a stream
uint8_t *g_words = nullptr; // what the words lie in
size_t g_words_size = 0;
std::function<void()> g_at_read;

void
launch_seen_by_two_threads() {
    REQUIRE(nixl_amd_copy_watch_prepare() == 0 && g_words);
    static Stream s;
    static nixl_amd_copy_plan_t *plan = block_plan();
    static bool reached = false;
    struct sigaction act{};
    act.sa_handler = [](int) {
        REQUIRE(g_at_read && !reached);
        REQUIRE(mprotect(g_words, g_words_size, PROT_READ | PROT_WRITE) == 0);
        reached = true;
        g_at_read();
    };
    act.sa_flags = SA_NODEFER;
    REQUIRE(sigaction(SIGSEGV, &act, nullptr) == 0);
    g_at_read = [] {
        std::thread([] {
            s.let_go();
            REQUIRE(nixl_amd_copy_plan_status(plan, 0) == 0);
            nixl_amd_copy_plan_t *other = block_plan();
            REQUIRE(nixl_amd_copy_plan_launch_watched(other, &s) == 0); // and has run
        }).join();
    };
    g_asked = [](hipStream_t) {
        g_asked = nullptr;
        REQUIRE(mprotect(g_words, g_words_size, PROT_NONE) == 0);
    };
    s.held = true;
    REQUIRE(nixl_amd_copy_plan_launch_watched(plan, &s) == 0);
    int rc = NIXL_AMD_ERR_BUSY;
    for (int i = 0; i < 10000 && rc == NIXL_AMD_ERR_BUSY; ++i)
        rc = nixl_amd_copy_plan_status(plan, 0);
    REQUIRE(reached && rc == 0);
}

// 70 requests against device-resident lists that wait for their verdicts at once: each counts in totals of its own
// that are zero when it starts; 64 find such totals ready, the others clear some.
void
many_requests_wait_for_verdicts() {
    constexpr int kRequests = 70, kReady = 64;
    Lists lists;
    nixl_amd_copy_plan_t *plan = nullptr;
    REQUIRE(lists.request(nullptr, &plan) == 0); // makes the library's stream
    REQUIRE(nixl_amd_copy_plan_destroy(plan) == 0);
    static Stream *uploads = nullptr;
    for (int round = 0; round < 2; ++round) {
        uploads = g_created;
        uploads->kernels.clear();
        uploads->held = true;
        g_totals.clear();
        g_synchronized = [](Stream &) {
            for (int n = 0; n < kRequests; std::this_thread::yield()) {
                const std::lock_guard<std::recursive_mutex> lock(g_lock);
                n = launched(*uploads, "list_records_kernel");
            }
        };
        nixl_amd_copy_plan_t *plans[kRequests] = {};
        std::vector<std::thread> threads;
        for (nixl_amd_copy_plan_t *&p : plans)
            threads.emplace_back([&lists, &p] { REQUIRE(lists.request(nullptr, &p) == 0); });
        for (std::thread &t : threads)
            t.join();
        REQUIRE(g_totals.size() == kRequests);
        REQUIRE(launched(*uploads, "clear_totals_kernel") == kRequests - kReady);
        for (nixl_amd_copy_plan_t *p : plans)
            REQUIRE(nixl_amd_copy_plan_destroy(p) == 0);
        g_synchronized = nullptr;
    }
}

// Requests whose launches are refused, the first or a later one, leave their totals to others, at zero.
void
refused_launches_keep_no_totals() {
    Lists lists;
    nixl_amd_copy_plan_t *plan = nullptr;
    REQUIRE(lists.request(nullptr, &plan) == 0);
    REQUIRE(nixl_amd_copy_plan_destroy(plan) == 0);
    Stream &uploads = *g_created;
    lists.index.resize(150000); // three launches, as vectors
    for (size_t i = 0; i < lists.index.size(); ++i)
        lists.index[i] = static_cast<int32_t>(i * 7919 % Lists::kEntries);
    for (const int good : {0, 1, 2})
        for (int i = 0; i < 100; ++i) {
            g_good_launches = good;
            g_launch_status = hipErrorOutOfMemory;
            REQUIRE(lists.request(nullptr, &plan) == NIXL_AMD_ERR_HIP);
        }
    uploads.kernels.clear();
    g_totals.clear();
    REQUIRE(lists.request(nullptr, &plan) == 0);
    REQUIRE(launched(uploads, "clear_totals_kernel") == 0);
    REQUIRE(nixl_amd_copy_plan_destroy(plan) == 0);
}

// A request of byte descriptors while pinned memory is short: what cannot be had ahead is asked for again
// when its size is known, and if it cannot be had then either the request is refused.
void
pinned_memory_is_short() {
    Stream s;
    const nixl_amd_copy_tuning_t tuning = tuning_for(s);
    size_t n = 100;
    for (const int refused : {1, 2, 0, 1, 2, 0}) {
        std::vector<nixl_amd_copy_desc_t> descs(n *= 4); // longer than what earlier requests gave back
        for (size_t i = 0; i < n; ++i)
            descs[i] = {(1ull << 40) + i * 64 + 1, (1ull << 41) + i * 64, 33};
        g_refused_pinned = refused;
        nixl_amd_copy_plan_t *plan = nullptr;
        const int rc = nixl_amd_copy_plan_create(descs.data(), n, 0, &tuning, &plan);
        REQUIRE(rc == (refused == 2 ? NIXL_AMD_ERR_HIP : NIXL_AMD_OK) && g_refused_pinned == 0);
        const hipError_t left = hipGetLastError();
        if (rc) continue;
        REQUIRE(left == hipSuccess); // for the caller's next call
        REQUIRE(nixl_amd_copy_plan_launch(plan, &s) == 0);
        REQUIRE(nixl_amd_copy_plan_destroy(plan) == 0);
    }
}

// What cannot be had ahead is not asked for ahead again in the same request.
void
pinned_memory_is_asked_for_once() {
    Stream s;
    const nixl_amd_copy_tuning_t tuning = tuning_for(s);
    std::vector<nixl_amd_copy_desc_t> descs;
    for (size_t i = 0; i < 64; ++i) {
        descs.push_back({(1ull << 40) + i * (2ull << 20) + 1, (1ull << 41) + i * (2ull << 20), (1 << 20) + 2});
        descs.push_back({(3ull << 40) + i * 4096, (4ull << 40) + i * 4096, 640});
    }
    nixl_amd_copy_plan_t *plan = nullptr;
    g_refused_pinned = 1000;
    g_pinned.clear();
    REQUIRE(nixl_amd_copy_plan_create(descs.data(), descs.size(), 0, &tuning, &plan) == NIXL_AMD_ERR_HIP);
    REQUIRE(g_pinned.size() <= 2);
    g_refused_pinned = 0;
    (void)hipGetLastError();
}

// What byte descriptors are written to ahead is as long as they need, whatever else is in the list.
void
pinned_memory_is_for_byte_descriptors() {
    Stream s;
    const nixl_amd_copy_tuning_t tuning = tuning_for(s);
    constexpr size_t kDescs = 100000;
    std::vector<nixl_amd_copy_desc_t> descs;
    for (size_t i = 0; i < kDescs; ++i) // a record of 16 bytes for each
        descs.push_back({(1ull << 40) + i * 4096, (2ull << 40) + i * 4096, 640});
    for (size_t i = 0; i < kDescs; i += 100) // and an item of 24 for some
        descs[i] = {(3ull << 40) + i * 64 + 1, (4ull << 40) + i * 64, 33};
    for (const size_t n : {size_t(50), kDescs}) {
        nixl_amd_copy_plan_t *plan = nullptr;
        g_pinned.clear();
        REQUIRE(nixl_amd_copy_plan_create(descs.data(), n, 0, &tuning, &plan) == 0);
        nixl_amd_copy_plan_info_t info{};
        REQUIRE(nixl_amd_copy_plan_query(plan, &info) == 0);
        for (const size_t size : g_pinned)
            REQUIRE(size <= std::max<size_t>(512 << 10, 2 * info.plan_device_bytes));
        REQUIRE(nixl_amd_copy_plan_destroy(plan) == 0);
    }
}

// Loads through the last-level cache (policy 3) or past it (4): where sources follow one another and destinations are
// regular from 88 MiB of payload on past it, otherwise from 112.
void
loads_through_the_last_level_cache() {
    Stream s;
    const nixl_amd_copy_tuning_t tuning = tuning_for(s);
    constexpr uint64_t kSrc = 1ull << 40, kDst = 1ull << 41, kMiB = 1 << 20;
    const auto policy = [&](nixl_amd_copy_plan_t *plan) {
        s.kernels.clear();
        REQUIRE(nixl_amd_copy_plan_launch(plan, &s) == 0);
        REQUIRE(nixl_amd_copy_plan_destroy(plan) == 0);
        REQUIRE(s.kernels.size() == 1);
        const std::string &name = s.kernels[0];
        for (const char *kernel : {"copy_inline_kernelILi", "copy_grid_kernelILi", "copy_piece_kernelILi", "copy_uniform_kernelILi1ELi"})
            if (const size_t at = name.find(kernel); at != std::string::npos) return name[at + std::strlen(kernel)] - '0';
        return 0;
    };
    const auto of = [&](const std::vector<nixl_amd_copy_desc_t> &descs) {
        nixl_amd_copy_plan_t *plan = nullptr;
        REQUIRE(nixl_amd_copy_plan_create(descs.data(), descs.size(), 0, &tuning, &plan) == 0);
        return policy(plan);
    };
    enum { kOne, kFollowing, kApart, kGathered, kScattered, kStrided };
    for (const uint64_t mib : {64, 88, 92, 112, 116, 200})
        for (const uint64_t len : {uint64_t(2048), uint64_t(16384), kMiB, kMiB + 1024})
            for (const int shape : {kOne, kFollowing, kApart, kGathered, kScattered, kStrided}) {
                const uint64_t n = shape == kOne ? 1 : mib * kMiB / len, each = shape == kOne ? mib * kMiB : len;
                const auto place = [&](uint64_t i, bool any, uint64_t step) { return (any ? i * 7919 % n * 3 + i % 2 : i) * step; };
                std::vector<nixl_amd_copy_desc_t> descs(n);
                for (uint64_t i = 0; i < n; ++i)
                    descs[i] = {kSrc + place(i, shape == kApart || shape == kGathered, each),
                                kDst + place(i, shape == kApart || shape == kScattered, shape == kStrided ? 3 * each : each), each};
                const bool past = shape <= kFollowing || shape == kStrided ? mib > 88 && (len != 2048 || shape == kOne || mib > 112) : shape == kGathered ? mib > 112 : len == 2048 && mib > 112;
                REQUIRE(of(descs) == (past ? 4 : 3));
                if (each % 1024 != 0 || len == 2048 || len > 16384 || shape == kOne) continue;
                std::vector<int32_t> src(n), dst(n); // the same by index
                for (uint64_t i = 0; i < n; ++i) {
                    src[i] = static_cast<int32_t>((descs[i].src - kSrc) / each);
                    dst[i] = static_cast<int32_t>((descs[i].dst - kDst) / each);
                }
                const nixl_amd_copy_run_t from{kSrc, each, 0, 4 * n}, to{kDst, each, 0, 4 * n};
                nixl_amd_copy_plan_t *plan = nullptr;
                REQUIRE(nixl_amd_copy_plan_create_indexed_lists(&from, 1, src.data(), 4 * n, &to, 1, dst.data(), 4 * n, n, each, 0, &tuning, &plan) == 0);
                REQUIRE(policy(plan) == (past ? 4 : 3));
            }
}

// A request without records that is launched again and again on the stream it was made for: the sixteenth launch makes some, in
// front of its copy, and launches on that stream use them; others, and all where there can be none, go without.
void
records_for_many_launches() {
    constexpr uintptr_t kSrc = 1ull << 40, kDst = 1ull << 41;
    REQUIRE(nixl_amd_copy_watch_prepare() == 0);
    const auto made = [&](size_t n, bool grid, bool scatter, uint64_t len, void *stream) {
        std::vector<int32_t> listed(n), flat(n);
        std::iota(flat.begin(), flat.end(), 0);
        const size_t ids = grid ? 1000 : n;
        for (size_t i = 0; i < n; ++i)
            listed[i] = static_cast<int32_t>((i % ids) * (i % ids) * 31 % 65521 + i / ids * 65521); // no even steps
        const nixl_amd_copy_run_t src{kSrc, len, 0, 1u << 30}, dst{kDst, len, 0, 1u << 30};
        nixl_amd_copy_tuning_t tuning{};
        tuning.stream = stream;
        nixl_amd_copy_plan_t *plan = nullptr;
        REQUIRE(nixl_amd_copy_plan_create_indexed_lists(&src, 1, (scatter ? flat : listed).data(), 1u << 30, &dst, 1, (scatter ? listed : flat).data(),
                                                        1u << 30, n, len, 0, &tuning, &plan) == 0);
        return plan;
    };
    const auto launch = [&](nixl_amd_copy_plan_t *plan, Stream &s, bool ok = true) { // the kernels of one launch
        s.kernels.clear();
        REQUIRE((nixl_amd_copy_plan_launch_watched(plan, &s) == 0) == ok);
        REQUIRE(nixl_amd_copy_plan_status(plan, 1) == 0);
        return s.kernels;
    };
    const auto has = [](const std::vector<std::string> &kernels, size_t i, const char *name) { return i < kernels.size() && kernels[i].find(name) != std::string::npos; };
    const auto device_bytes = [](nixl_amd_copy_plan_t *plan) {
        nixl_amd_copy_plan_info_t info{};
        REQUIRE(nixl_amd_copy_plan_query(plan, &info) == 0);
        return info.plan_device_bytes;
    };
    struct Case {
        size_t n;
        bool grid, scatter;
        uint64_t len;
        const char *records; // kernel
        char policy; // of the copy from then on
    };
    for (const Case &c : {Case{600, false, false, 8192, "ILb0ENS_13InlineIndicesE", '3'}, {2000, true, false, 1024, "ILb0ENS_11GridIndicesE", '3'},
                          {16000, true, true, 16384, "ILb0ENS_11GridIndicesE", '3'}, {17000, true, true, 16384, "ILb1ENS_11GridIndicesE", '4'},
                          {32000, true, true, 15360, "ILb0ENS_11GridIndicesE", '3'}, {17000, true, false, 16384, "ILb0ENS_11GridIndicesE", '4'}}) {
        Stream home, other;
        nixl_amd_copy_plan_t *plan = made(c.n, c.grid, c.scatter, c.len, &home);
        REQUIRE(device_bytes(plan) == 0);
        const auto without = [&](const std::vector<std::string> &kernels) { return has(kernels, 0, c.grid ? "GridIndices" : "InlineIndices") && !has(kernels, 0, "later_records"); };
        for (int i = 1; i <= 15; ++i) {
            REQUIRE(without(launch(plan, home)));
            REQUIRE(without(launch(plan, other)));
        }
        REQUIRE(without(launch(plan, other)) && device_bytes(plan) == 0);
        g_only_relaxed = true;
        auto kernels = launch(plan, home);
        g_only_relaxed = false;
        const auto with = [&](size_t at) { return has(kernels, at, "copy_uniform_kernelILi1E") && has(kernels, at, (std::string("ILi1ELi") + c.policy + "E").c_str()); };
        REQUIRE(has(kernels, 0, "later_records_kernel") && has(kernels, 0, c.records) && with(1));
        REQUIRE(device_bytes(plan) == c.n * 16);
        for (int i = 0; i < 20; ++i) {
            kernels = launch(plan, home);
            REQUIRE(with(0));
            REQUIRE(without(launch(plan, other)));
        }
        REQUIRE(nixl_amd_copy_plan_destroy(plan) == 0);
        // no memory, or no launch of the kernel that makes them: not tried again
        for (const bool memory : {true, false}) {
            plan = made(c.n, c.grid, c.scatter, c.len, &home);
            for (int i = 0; i < 15; ++i)
                (void)launch(plan, home);
            std::vector<nixl_amd_copy_plan_t *> takers; // of the memory that plans gave back
            if (memory)
                for (int i = 0; i < 4; ++i) {
                    takers.push_back(made(c.n, c.grid, c.scatter, c.len, &other));
                    for (int j = 0; j < 16; ++j)
                        (void)launch(takers.back(), other);
                }
            if (memory)
                g_refused_device = 1;
            else
                g_launch_status = hipErrorOutOfMemory, g_good_launches = 0;
            REQUIRE(without(launch(plan, home)) && device_bytes(plan) == 0);
            REQUIRE(g_refused_device == 0 && g_launch_status == hipSuccess && hipGetLastError() == hipSuccess);
            for (int i = 0; i < 40; ++i)
                REQUIRE(without(launch(plan, home)));
            for (nixl_amd_copy_plan_t *taker : takers)
                REQUIRE(nixl_amd_copy_plan_destroy(taker) == 0);
            REQUIRE(nixl_amd_copy_plan_destroy(plan) == 0);
        }
        // an error that somebody else left behind is taken for theirs: they are waited for before their memory goes back
        plan = made(c.n, c.grid, c.scatter, c.len, &home);
        for (int i = 0; i < 15; ++i)
            (void)launch(plan, home);
        g_refused_device = 1;
        void *none = nullptr;
        REQUIRE(hipMalloc(&none, 1) != hipSuccess);
        home.waited_for = false;
        home.held = true;
        home.kernels.clear();
        REQUIRE(nixl_amd_copy_plan_launch_watched(plan, &home) == 0);
        REQUIRE(has(home.kernels, 0, "later_records_kernel") && home.waited_for);
        REQUIRE(nixl_amd_copy_plan_status(plan, 1) == 0);
        REQUIRE(without(launch(plan, home)) && device_bytes(plan) == 0);
        REQUIRE(nixl_amd_copy_plan_destroy(plan) == 0);
        // the copy behind them fails: nothing of theirs runs when the plan may be destroyed
        plan = made(c.n, c.grid, c.scatter, c.len, &home);
        for (int i = 0; i < 15; ++i)
            (void)launch(plan, home);
        home.waited_for = false;
        g_launch_status = hipErrorOutOfMemory;
        g_good_launches = 1;
        home.held = true;
        REQUIRE(nixl_amd_copy_plan_launch_watched(plan, &home) == NIXL_AMD_ERR_HIP);
        REQUIRE(home.waited_for && home.work.empty());
        kernels = launch(plan, home);
        REQUIRE(with(0));
        REQUIRE(nixl_amd_copy_plan_destroy(plan) == 0);
        // made for no stream, or for one that is not the same in every thread
        for (void *stream : {static_cast<void *>(nullptr), static_cast<void *>(hipStreamPerThread), static_cast<void *>(hipStreamLegacy)}) {
            plan = made(c.n, c.grid, c.scatter, c.len, stream);
            for (int i = 0; i < 40; ++i) {
                REQUIRE(nixl_amd_copy_plan_launch(plan, stream) == 0);
                REQUIRE(without(launch(plan, home)));
            }
            REQUIRE(device_bytes(plan) == 0);
            REQUIRE(nixl_amd_copy_plan_destroy(plan) == 0);
        }
    }
}

} // namespace

// ---- the runtime ------------------------------------------------------------------------------

#define LOCKED const std::lock_guard<std::recursive_mutex> lock(g_lock)

extern "C" {

void **
__hipRegisterFatBinary(const void *) {
    static void *module = nullptr;
    return &module;
}

void
__hipUnregisterFatBinary(void **) {}

void
__hipRegisterFunction(void **, const void *stub, char *, const char *name, unsigned, void *, void *, void *, void *, int *) {
    kernel_names()[stub] = name;
}

void
__hipRegisterVar(void **, void *symbol, char *, char *, int, size_t size, int, int) {
    void *p = std::aligned_alloc(128, (size + 127) / 128 * 128);
    std::memset(p, 0, size);
    device_variables()[symbol] = p;
}

struct CallConfiguration {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
};
static thread_local std::vector<CallConfiguration> g_calls;

hipError_t
__hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
    g_calls.push_back({grid, block, shared, stream});
    return hipSuccess;
}

hipError_t
__hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *stream) {
    const CallConfiguration c = g_calls.back();
    g_calls.pop_back();
    *grid = c.grid;
    *block = c.block;
    *shared = c.shared;
    *stream = c.stream;
    return hipSuccess;
}

static thread_local hipError_t g_last_status = hipSuccess;

hipError_t
hipLaunchKernel(const void *stub, dim3 grid, dim3, void **args, size_t, hipStream_t stream) {
    LOCKED;
    if (g_launch_status != hipSuccess && g_good_launches-- <= 0) {
        g_last_status = std::exchange(g_launch_status, hipSuccess); // once
        return g_last_status;
    }
    const std::string &name = kernel_names().at(stub);
    Stream &s = stream_of(stream);
    s.kernels.push_back(name);
    s.queue(work_of(name, grid, args));
    return hipSuccess;
}

hipError_t
hipGetSymbolAddress(void **p, const void *symbol) {
    *p = device_variables().at(symbol);
    return hipSuccess;
}

hipError_t
hipGetDeviceCount(int *n) {
    *n = 1;
    return hipSuccess;
}

hipError_t
hipGetDevice(int *device) {
    *device = 0;
    return hipSuccess;
}

hipError_t
hipSetDevice(int) {
    return hipSuccess;
}

hipError_t
hipDeviceGetAttribute(int *value, hipDeviceAttribute_t, int) {
    *value = 1;
    return hipSuccess;
}

hipError_t
hipGetLastError() {
    return std::exchange(g_last_status, hipSuccess);
}

const char *
hipGetErrorString(hipError_t) {
    return "an error";
}

hipError_t
hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *mode) {
    std::swap(*mode, t_mode);
    return hipSuccess;
}

hipError_t
hipMalloc(void **p, size_t n) {
    LOCKED;
    REQUIRE(!g_only_relaxed || t_mode == hipStreamCaptureModeRelaxed);
    if (g_refused_device > 0) {
        --g_refused_device;
        return g_last_status = hipErrorOutOfMemory;
    }
    *p = std::aligned_alloc(4096, (n + 4095) / 4096 * 4096);
    std::memset(*p, 0xa5, n); // nobody may count on zeroes
    return hipSuccess;
}

hipError_t
hipHostMalloc(void **p, size_t n, unsigned flags) {
    LOCKED;
    g_pinned.push_back(n);
    if (g_refused_pinned > 0) {
        --g_refused_pinned;
        return g_last_status = hipErrorOutOfMemory;
    }
    const hipError_t e = hipMalloc(p, n);
    if (flags & hipHostMallocPortable) { // the words that launches are watched by
        g_words = static_cast<uint8_t *>(*p);
        g_words_size = (n + 4095) / 4096 * 4096;
    }
    return e;
}

hipError_t
hipFree(void *p) {
    std::free(p);
    return hipSuccess;
}

hipError_t
hipHostFree(void *p) {
    return hipFree(p);
}

hipError_t
hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind, hipStream_t stream) {
    LOCKED;
    stream_of(stream).queue([=] { std::memcpy(dst, src, n); });
    return hipSuccess;
}

hipError_t
hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    g_created = new Stream;
    *s = handle(*g_created);
    return hipSuccess;
}

hipError_t
hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *status) {
    *status = hipStreamCaptureStatusNone;
    return hipSuccess;
}

hipError_t
hipStreamQuery(hipStream_t stream) {
    LOCKED;
    const Stream &s = stream_of(stream);
    if (g_asked) {
        g_asked(stream);
        return hipSuccess; // the launch has just ended
    }
    if (s.failure != hipSuccess) return s.failure;
    return s.work.empty() ? hipSuccess : hipErrorNotReady;
}

hipError_t
hipStreamSynchronize(hipStream_t stream) {
    Stream &s = stream_of(stream);
    if (g_synchronized) g_synchronized(s);
    LOCKED;
    s.waited_for = true;
    s.let_go();
    return s.failure;
}

hipError_t
hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) {
    return hipSuccess;
}

hipError_t
hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>(new Event);
    return hipSuccess;
}

hipError_t
hipEventCreate(hipEvent_t *e) {
    return hipEventCreateWithFlags(e, 0);
}

hipError_t
hipEventDestroy(hipEvent_t e) {
    delete &event_of(e);
    return hipSuccess;
}

hipError_t
hipEventRecord(hipEvent_t event, hipStream_t stream) {
    LOCKED;
    Event &e = event_of(event);
    e.done = std::make_shared<bool>(false);
    e.on = &stream_of(stream);
    e.on->queue([done = e.done] { *done = true; });
    return hipSuccess;
}

hipError_t
hipEventQuery(hipEvent_t event) {
    LOCKED;
    const Event &e = event_of(event);
    if (*e.done) return hipSuccess;
    return e.on->failure != hipSuccess ? e.on->failure : hipErrorNotReady;
}

hipError_t
hipEventSynchronize(hipEvent_t event) {
    LOCKED;
    const Event &e = event_of(event);
    if (*e.done) return hipSuccess;
    e.on->waited_for = true;
    e.on->let_go();
    return e.on->failure;
}

hipError_t
hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 0.f;
    return hipSuccess;
}

} // extern "C"

int
main(int argc, char **argv) {
    const std::map<std::string, void (*)()> scenarios{
        {"work_behind_a_watched_launch", work_behind_a_watched_launch},
        {"indices_that_repeat_themselves", indices_that_repeat_themselves},
        {"launch_on_a_named_stream_fails", launch_on_a_named_stream_fails},
        {"launch_on_the_legacy_stream_fails", launch_on_the_legacy_stream_fails},
        {"launch_on_the_stream_of_a_thread", launch_on_the_stream_of_a_thread},
        {"launch_seen_by_two_threads", launch_seen_by_two_threads},
        {"many_requests_wait_for_verdicts", many_requests_wait_for_verdicts},
        {"refused_launches_keep_no_totals", refused_launches_keep_no_totals},
        {"pinned_memory_is_short", pinned_memory_is_short},
        {"pinned_memory_is_asked_for_once", pinned_memory_is_asked_for_once},
        {"pinned_memory_is_for_byte_descriptors", pinned_memory_is_for_byte_descriptors},
        {"loads_through_the_last_level_cache", loads_through_the_last_level_cache},
        {"records_for_many_launches", records_for_many_launches},
    };
    REQUIRE(argc == 2 && scenarios.count(argv[1]));
    scenarios.at(argv[1])();
    std::printf("OK\n");
    return 0;
}
