// Seventy requests against device-resident lists at once, on the GPU: all of them are held at their first launch
// until the last one is there, so that more wait for their verdicts than find totals ready.  Those that find
// none clear some of their own in front of their records.
//
// usage: list_totals_check; prints "OK" and exits 0 on success.
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <thread>
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

constexpr int kRequests = 70, kReady = 64;
std::atomic<int> g_arrived{0}, g_launches{0};
thread_local bool t_requesting = false, t_arrived = false;

} // namespace

// In front of libamdhip64's.
extern "C" hipError_t
hipLaunchKernel(const void *stub, dim3 grid, dim3 block, void **args, size_t shared, hipStream_t stream) {
    static const auto launch = reinterpret_cast<decltype(&hipLaunchKernel)>(dlsym(RTLD_NEXT, "hipLaunchKernel"));
    if (t_requesting) {
        g_launches.fetch_add(1);
        if (!t_arrived) {
            t_arrived = true;
            g_arrived.fetch_add(1);
            while (g_arrived.load() < kRequests)
                std::this_thread::yield();
        }
    }
    return launch(stub, grid, block, args, shared, stream);
}

int
main() {
    constexpr size_t kEntries = 3000, kRoom = 512;
    uint8_t *mem = nullptr;
    REQUIRE(hipMalloc(reinterpret_cast<void **>(&mem), (kRequests + 1) * kEntries * kRoom) == hipSuccess);
    std::vector<uint8_t> want(kEntries * kRoom), got(kEntries * kRoom);
    for (size_t i = 0; i < want.size(); ++i)
        want[i] = static_cast<uint8_t>(i * 2654435761u >> 13);
    REQUIRE(hipMemcpy(mem, want.data(), want.size(), hipMemcpyHostToDevice) == hipSuccess);
    const auto len = [](size_t entry) { return 128 + 16 * (entry % 17); };
    std::vector<nixl_amd_copy_list_t *> lists(kRequests + 1);
    for (size_t l = 0; l < lists.size(); ++l) {
        std::vector<nixl_amd_copy_list_entry_t> table(kEntries);
        for (size_t i = 0; i < kEntries; ++i) {
            table[i].addr = reinterpret_cast<uintptr_t>(mem) + (l * kEntries + i) * kRoom;
            table[i].len = static_cast<uint32_t>(len(i));
        }
        REQUIRE(nixl_amd_copy_list_create(table.data(), kEntries, 0, &lists[l]) == 0);
    }
    for (int round = 0; round < 3; ++round) {
        REQUIRE(hipMemset(mem + want.size(), 0, kRequests * want.size()) == hipSuccess);
        REQUIRE(hipDeviceSynchronize() == hipSuccess);
        g_arrived = g_launches = 0;
        std::vector<nixl_amd_copy_plan_t *> plans(kRequests, nullptr);
        std::vector<std::thread> threads;
        for (int r = 0; r < kRequests; ++r)
            threads.emplace_back([&, r] {
                std::vector<int32_t> index; // request r: every entry but some, in an order of its own
                uint64_t bytes = 0;
                for (size_t i = 0; i < kEntries; ++i) {
                    const size_t e = (i * 7 + static_cast<size_t>(r)) % kEntries; // 7 and 3000 have no common factor
                    if (e % 70 == static_cast<size_t>(r)) continue;
                    index.push_back(static_cast<int32_t>(e));
                    bytes += len(e);
                }
                t_requesting = true;
                REQUIRE(nixl_amd_copy_plan_create_listed(lists[0], index.data(), lists[r + 1], index.data(), index.size(), nullptr,
                                                         nullptr, &plans[r]) == 0);
                t_requesting = false;
                nixl_amd_copy_plan_info_t info{};
                REQUIRE(nixl_amd_copy_plan_query(plans[r], &info) == 0);
                REQUIRE(info.payload_bytes == bytes && info.vec_descs == index.size());
            });
        for (std::thread &t : threads)
            t.join();
        REQUIRE(g_launches == kRequests + (kRequests - kReady)); // one of records each
        for (int r = 0; r < kRequests; ++r) {
            REQUIRE(nixl_amd_copy_plan_launch(plans[r], nullptr) == 0);
            REQUIRE(nixl_amd_copy_plan_status(plans[r], 1) == 0);
            REQUIRE(nixl_amd_copy_plan_destroy(plans[r]) == 0);
            REQUIRE(hipMemcpy(got.data(), mem + (r + 1) * want.size(), got.size(), hipMemcpyDeviceToHost) == hipSuccess);
            for (size_t i = 0; i < got.size(); ++i) {
                const size_t e = i / kRoom;
                const bool copied = e % 70 != static_cast<size_t>(r) && i % kRoom < len(e);
                REQUIRE(got[i] == (copied ? want[i] : 0));
            }
        }
        std::printf("round %d\n", round);
        std::fflush(stdout);
    }
    for (nixl_amd_copy_list_t *l : lists)
        REQUIRE(nixl_amd_copy_list_destroy(l) == 0);
    REQUIRE(hipFree(mem) == hipSuccess);
    std::printf("OK\n");
    return 0;
}
