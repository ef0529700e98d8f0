// Requests by index with a backend that takes descriptors, on the CPU: std::vector arguments are
// read where they are, indices that the caller keeps itself are copied first, and both make the
// same request; an index outside its list is refused either way.
//
// usage: index_vectors_check <directory holding libplugin_MEMCPY.so>; prints "OK".
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <numeric>
#include <vector>
#include "nixl.h"
#define REQUIRE(c) do { if (!(c)) { std::fprintf(stderr, "%s:%d: %s failed\n", __FILE__, __LINE__, #c); std::exit(1);} } while (0)

constexpr size_t kBlocks = 50001, kLen = 16;
static int g_copies = 0; // allocations of one index vector's size

void *
operator new(std::size_t n) {
    if (n == kBlocks * sizeof(int)) ++g_copies;
    if (void *p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

int main(int argc, char **argv) {
    REQUIRE(argc == 2);
    setenv("NIXL_PLUGIN_DIR", argv[1], 1);
    nixlAgent agent("A", nixlAgentConfig(false));
    nixlBackendH *backend = nullptr;
    REQUIRE(agent.createBackend("MEMCPY", {}, backend) == NIXL_SUCCESS);
    std::vector<uint8_t> src(kBlocks * kLen), dst(kBlocks * kLen);
    nixl_reg_dlist_t reg(DRAM_SEG);
    reg.addDesc(nixlBlobDesc((uintptr_t)src.data(), src.size(), 0, ""));
    reg.addDesc(nixlBlobDesc((uintptr_t)dst.data(), dst.size(), 0, ""));
    REQUIRE(agent.registerMem(reg) == NIXL_SUCCESS);
    nixlDlistH *sides[2] = {nullptr, nullptr};
    for (int side = 0; side < 2; ++side) {
        nixl_xfer_dlist_t list(DRAM_SEG);
        for (size_t i = 0; i < kBlocks; ++i)
            list.addDesc(nixlBasicDesc((uintptr_t)(side ? dst : src).data() + i * kLen, kLen, 0));
        REQUIRE(agent.prepXferDlist(side ? "A" : "", list, sides[side]) == NIXL_SUCCESS);
    }
    std::vector<int> li(kBlocks), ri(kBlocks);
    std::iota(li.begin(), li.end(), 0);
    for (size_t i = 0; i < kBlocks; ++i)
        ri[i] = static_cast<int>((i * 7919) % kBlocks);
    for (const bool vectors : {true, false}) {
        for (size_t i = 0; i < src.size(); ++i)
            src[i] = static_cast<uint8_t>(i * 31 + i / 251 + vectors);
        std::memset(dst.data(), 0, dst.size());
        const auto make = [&](nixlXferReqH *&req) {
            return vectors ? agent.makeXferReq(NIXL_WRITE, sides[0], li, sides[1], ri, req) :
                             agent.makeXferReq(NIXL_WRITE, sides[0], li.data(), li.size(), sides[1], ri.data(), ri.size(), req);
        };
        nixlXferReqH *req = nullptr;
        g_copies = 0;
        REQUIRE(make(req) == NIXL_SUCCESS);
        REQUIRE(g_copies == (vectors ? 0 : 2));
        nixl_status_t st = agent.postXferReq(req);
        while (st == NIXL_IN_PROG)
            st = agent.getXferStatus(req);
        REQUIRE(st == NIXL_SUCCESS);
        for (size_t i = 0; i < kBlocks; ++i)
            REQUIRE(std::memcmp(&dst[ri[i] * kLen], &src[li[i] * kLen], kLen) == 0);
        REQUIRE(agent.releaseXferReq(req) == NIXL_SUCCESS);
        for (std::vector<int> *side : {&li, &ri})
            for (const int bad : {-1, static_cast<int>(kBlocks)}) {
                const int good = (*side)[kBlocks / 2];
                (*side)[kBlocks / 2] = bad;
                REQUIRE(make(req) == NIXL_ERR_INVALID_PARAM);
                (*side)[kBlocks / 2] = good;
            }
    }
    REQUIRE(agent.releasedDlistH(sides[0]) == NIXL_SUCCESS && agent.releasedDlistH(sides[1]) == NIXL_SUCCESS);
    std::puts("OK");
}
