// The HIP backend deals requests to its streams in turn: one turn a request, also for a request
// that the indexed entry or the block plan declines and that goes on to the general lowering, and
// none for one that the indexed entry or the one for device-resident lists refuses.
//
// usage: stream_turns_check <path to libplugin_HIP.so>; prints "OK" and exits 0 on success.
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <numeric>
#include <vector>

#include "backend/backend_plugin.h"
#include "hip_backend.h"

#define REQUIRE(cond)                                                          \
    do {                                                                       \
        if (!(cond)) {                                                         \
            std::fprintf(stderr, "%s:%d: %s failed\n", __FILE__, __LINE__, #cond); \
            std::exit(1);                                                      \
        }                                                                      \
    } while (0)

int
main(int argc, char **argv) {
    REQUIRE(argc == 2);
    void *lib = dlopen(argv[1], RTLD_NOW | RTLD_LOCAL | RTLD_NODELETE);
    REQUIRE(lib);
    auto init = reinterpret_cast<nixlBackendPlugin *(*)()>(dlsym(lib, "nixl_plugin_init"));
    using indexed_fn = int (*)(nixlBackendEngine *, int, const nixlStrideDesc *, size_t, const int *, const nixlStrideDesc *, size_t,
                               const int *, size_t, const char *, nixlBackendReqH **);
    auto indexed = reinterpret_cast<indexed_fn>(dlsym(lib, "nixl_hip_prep_xfer_indexed"));
    auto prep_list = reinterpret_cast<int (*)(nixlBackendEngine *, const nixlStrideDesc *, size_t, void **)>(dlsym(lib, "nixl_hip_prep_list"));
    auto release_list = reinterpret_cast<void (*)(void *)>(dlsym(lib, "nixl_hip_release_list"));
    using listed_fn = int (*)(nixlBackendEngine *, int, const void *, const int *, const void *, const int *, size_t, const char *, size_t *,
                              size_t *, nixlBackendReqH **);
    auto listed = reinterpret_cast<listed_fn>(dlsym(lib, "nixl_hip_prep_xfer_listed"));
    REQUIRE(init && indexed && prep_list && release_list && listed);
    nixlBackendPlugin *plugin = init();

    constexpr unsigned n_streams = 3;
    nixl_b_params_t custom{{"num_streams", std::to_string(n_streams)}};
    nixlBackendInitParams params;
    params.localAgent = "turns";
    params.type = "HIP";
    params.customParams = &custom;
    params.enableProgTh = false;
    params.pthrDelay = 0;
    params.syncMode = nixl_thread_sync_t::NIXL_THREAD_SYNC_NONE;
    nixlBackendEngine *engine = plugin->create_engine(&params);
    REQUIRE(engine && !engine->getInitErr());

    constexpr size_t blocks = 200, len = 8192, room = (blocks + 1) * len;
    uint8_t *mem = nullptr;
    REQUIRE(hipMalloc(reinterpret_cast<void **>(&mem), 2 * room) == hipSuccess);
    const auto at = reinterpret_cast<uintptr_t>(mem);
    nixlBackendMD *md = nullptr;
    REQUIRE(engine->registerMem(nixlBlobDesc(at, 2 * room, 0, ""), VRAM_SEG, md) == NIXL_SUCCESS);
    std::vector<int> index(blocks);
    std::iota(index.begin(), index.end(), 0);

    // What the agent does with a request by index: the indexed entry, and the descriptors if it
    // declines.  `offset` 0 is taken by the indexed entry, 16 (no line) and 8 (no 16 bytes) are not.
    const auto request = [&](uintptr_t offset, size_t n, bool by_index) {
        nixlBackendReqH *handle = nullptr;
        const nixlStrideDesc l(at + offset, len, 0, md, len, blocks), r(at + room + offset, len, 0, md, len, blocks);
        const int st = by_index ? indexed(engine, NIXL_WRITE, &l, 1, index.data(), &r, 1, index.data(), n, "turns", &handle) :
                                  NIXL_ERR_NOT_SUPPORTED;
        REQUIRE(st == (by_index && offset == 0 ? NIXL_SUCCESS : NIXL_ERR_NOT_SUPPORTED));
        if (st != NIXL_SUCCESS) {
            nixl_meta_dlist_t local(VRAM_SEG), remote(VRAM_SEG);
            for (size_t i = 0; i < n; ++i) {
                local.addDesc(nixlMetaDesc(at + offset + i * len, len, 0, md));
                remote.addDesc(nixlMetaDesc(at + room + offset + i * len, len, 0, md));
            }
            REQUIRE(engine->prepXfer(NIXL_WRITE, local, remote, "turns", handle) == NIXL_SUCCESS);
        }
        REQUIRE(handle);
        return handle;
    };

    for (const bool by_index : {true, false})
        for (const uintptr_t offset : {0, 16, 8})
            for (const size_t n : {size_t{3}, blocks}) {
                std::vector<hipStream_t> streams;
                for (unsigned i = 0; i < 2 * n_streams; ++i) {
                    nixlBackendReqH *handle = request(offset, n, by_index);
                    streams.push_back(static_cast<nixlHipReqH *>(handle)->stream);
                    REQUIRE(engine->releaseReqH(handle) == NIXL_SUCCESS);
                }
                for (unsigned i = 0; i < n_streams; ++i) {
                    REQUIRE(streams[i] && streams[i] == streams[i + n_streams]);
                    for (unsigned j = 0; j < i; ++j)
                        REQUIRE(streams[i] != streams[j]);
                }
            }

    // Two lists on the device, the second with one entry that is longer: requests that name it are refused.
    constexpr size_t entries = 1500, piece = 256;
    const nixlStrideDesc plain(at, piece, 0, md, 2 * piece, entries);
    nixlStrideDesc odd[2] = {nixlStrideDesc(at + room, piece, 0, md, 2 * piece, entries - 1),
                             nixlStrideDesc(at + room + (entries - 1) * 2 * piece, 2 * piece, 0, md, 2 * piece, 1)};
    odd[1].start_idx = entries - 1;
    void *lists[2] = {nullptr, nullptr};
    REQUIRE(prep_list(engine, &plain, 1, &lists[0]) == NIXL_SUCCESS && prep_list(engine, odd, 2, &lists[1]) == NIXL_SUCCESS);
    std::vector<int> good(entries - 1), longer(entries), outside(blocks);
    std::iota(good.begin(), good.end(), 0);
    std::iota(longer.begin(), longer.end(), 0);
    std::iota(outside.begin(), outside.end(), 1);
    std::vector<hipStream_t> taken;
    for (unsigned i = 0; i < 2 * n_streams; ++i) {
        nixlBackendReqH *handle = nullptr;
        size_t bytes = 0, merged = 0;
        REQUIRE(listed(engine, NIXL_WRITE, lists[0], longer.data(), lists[1], longer.data(), entries, "turns", &bytes, &merged, &handle) ==
                NIXL_ERR_NOT_SUPPORTED);
        const nixlStrideDesc l(at, len, 0, md, len, blocks), r(at + room, len, 0, md, len, blocks);
        REQUIRE(indexed(engine, NIXL_WRITE, &l, 1, outside.data(), &r, 1, index.data(), blocks, "turns", &handle) == NIXL_ERR_INVALID_PARAM);
        if (i % 2) {
            REQUIRE(listed(engine, NIXL_WRITE, lists[0], good.data(), lists[1], good.data(), entries - 1, "turns", &bytes, &merged, &handle) ==
                    NIXL_SUCCESS);
            REQUIRE(bytes == (entries - 1) * piece);
        } else {
            handle = request(0, blocks, true);
        }
        taken.push_back(static_cast<nixlHipReqH *>(handle)->stream);
        REQUIRE(engine->releaseReqH(handle) == NIXL_SUCCESS);
    }
    for (unsigned i = 0; i < n_streams; ++i) {
        REQUIRE(taken[i] && taken[i] == taken[i + n_streams]);
        for (unsigned j = 0; j < i; ++j)
            REQUIRE(taken[i] != taken[j]);
    }
    release_list(lists[0]);
    release_list(lists[1]);

    REQUIRE(engine->deregisterMem(md) == NIXL_SUCCESS);
    plugin->destroy_engine(engine);
    REQUIRE(hipFree(mem) == hipSuccess);
    std::printf("OK\n");
    return 0;
}
