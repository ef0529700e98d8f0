// The registered region that every descriptor of a list is resolved to (nixlMemSection::populate), against the two
// searches of src/infra/nixl_memory_section.cpp:56-104 written out here: from the start where a descriptor is ordered
// before the one in front of it, else on from that one's region.  Random regions that adjoin, overlap, start
// alike, are registered twice or lie on other devices, and descriptors in random and in ascending order, at the
// regions' edges and across them.  Host only.
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "agent_impl.h"

#define REQUIRE(cond)                                                              \
    do {                                                                           \
        if (!(cond)) {                                                             \
            std::fprintf(stderr, "%s:%d: %s failed\n", __FILE__, __LINE__, #cond); \
            std::exit(1);                                                          \
        }                                                                          \
    } while (0)

namespace {

// The regions' metadata, in list order; empty if some descriptor lies in none.
std::vector<nixlBackendMD *>
expected(const nixlSecDescList &base, const nixl_xfer_dlist_t &query) {
    std::vector<nixlBackendMD *> found;
    const int n = static_cast<int>(base.size());
    int at = -1;
    for (int i = 0; i < query.descCount(); ++i) {
        if (i == 0 || query[i] < query[i - 1]) {
            at = base.coveringIndex(query[i]);
        } else {
            while (at < n && !base[at].covers(query[i]))
                ++at;
            if (at == n) at = -1;
        }
        if (at < 0) return {};
        found.push_back(base[at].metadataP);
    }
    return found;
}

} // namespace

int
main() {
    std::mt19937 rng(7);
    const auto below = [&](uint32_t n) { return std::uniform_int_distribution<uint32_t>(0, n - 1)(rng); };
    size_t resolved = 0, refused = 0;
    for (int round = 0; round < 4000; ++round) {
        nixlMemSection section;
        std::vector<nixlSectionDesc> batch;
        const uint32_t n_regions = 1 + below(12), devices = 1 + below(2);
        for (uint32_t r = 0; r < n_regions; ++r) {
            nixlSectionDesc d(64 * (1 + below(20)), 64 * (1 + below(6)), below(devices));
            if (r && below(4) == 0) static_cast<nixlBasicDesc &>(d) = batch.back(); // again, or longer from the same start
            if (r && below(4) == 0) d.len += 64;
            d.metadataP = reinterpret_cast<nixlBackendMD *>(uintptr_t{16} * (r + 1));
            batch.push_back(d);
        }
        const auto regions = batch;
        nixlSecDescList &base = section.sections[{VRAM_SEG, nullptr}];
        base.add(std::move(batch));
        nixl_xfer_dlist_t query(VRAM_SEG);
        const uint32_t n_query = 1 + below(24);
        for (uint32_t q = 0; q < n_query; ++q) {
            const nixlSectionDesc &in = regions[below(n_regions)];
            const size_t from = below(3) == 0 ? 0 : below(static_cast<uint32_t>(in.len));
            size_t len = below(3) == 0 ? in.len - from : 1 + below(static_cast<uint32_t>(in.len - from));
            if (below(60) == 0) len += 64; // perhaps beyond its region
            query.addDesc(nixlBasicDesc(in.addr + from, len, in.devId));
        }
        if (round % 3 == 0) std::sort(query.begin(), query.end());
        const auto want = expected(base, query);
        nixl_meta_dlist_t got(VRAM_SEG);
        const nixl_status_t st = section.populate(query, nullptr, got);
        REQUIRE((st == NIXL_SUCCESS) == !want.empty());
        if (want.empty()) {
            ++refused;
            REQUIRE(got.isEmpty());
            continue;
        }
        ++resolved;
        REQUIRE(static_cast<size_t>(got.descCount()) == want.size());
        for (size_t i = 0; i < want.size(); ++i)
            REQUIRE(got[i].metadataP == want[i] && static_cast<const nixlBasicDesc &>(got[i]) == query[i]);
    }
    REQUIRE(resolved > 1000 && refused > 100);
    std::printf("%zu lists resolved, %zu refused\nOK\n", resolved, refused);
    return 0;
}
