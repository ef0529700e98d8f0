// Division by a multiplication (nixl_amd/csrc/kernels/common.h), which every copy and row kernel addresses memory
// by, against the division itself.  No GPU is used: both sides run the same code.
//
// usage: fast_div_check; prints "OK" and exits 0 on success.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <random>

#include "common.h"

static void
check(uint32_t divisor, uint32_t n) {
    const FastDiv by(divisor);
    uint32_t rest = ~0u;
    const uint32_t q = by.quotient(n, rest);
    if (by.divisor == divisor && by.quotient(n) == n / divisor && q == n / divisor && rest == n % divisor) return;
    std::fprintf(stderr, "%u / %u\n", n, divisor);
    std::exit(1);
}

// The dividends at which a quotient that is one off shows: around the first, a middle and the last multiple, and some.
static void
check(uint32_t divisor, std::mt19937 &rng) {
    const uint32_t last = 0xffffffffu / divisor * divisor, middle = 0xffffffffu / divisor / 2 * divisor;
    for (const uint32_t multiple : {0u, divisor, middle, last, static_cast<uint32_t>(rng() / divisor * divisor)})
        for (const uint32_t off : {0xffffffffu, 0u, 1u})
            check(divisor, multiple + off);
    for (const uint32_t n : {0x7fffffffu, 0x80000000u, 0xfffffffeu, 0xffffffffu, static_cast<uint32_t>(rng())})
        check(divisor, n);
}

int
main() {
    std::mt19937 rng(1);
    for (uint32_t d = 1; d <= 200000; ++d)
        check(d, rng);
    for (int bit = 0; bit < 32; ++bit)
        for (const uint32_t off : {0xffffffffu, 0u, 1u})
            if (const uint32_t d = (1u << bit) + off) check(d, rng);
    for (uint32_t d = 0xffffffffu; d > 0xffff0000u; --d)
        check(d, rng);
    for (int i = 0; i < 200000; ++i)
        if (const uint32_t d = static_cast<uint32_t>(rng()) >> (i % 32)) check(d, rng);
    for (const uint32_t d : {1u, 2u, 3u, 7u, 9u, 641u}) // every dividend of 24 bits, and the topmost ones
        for (uint32_t n = 0; n < 1u << 24; ++n) {
            check(d, n);
            check(d, ~n);
        }
    for (uint32_t n = 0; n < 1000; ++n)
        if (FastDiv().quotient(n) != n) return 1; // by one
    std::printf("OK\n");
    return 0;
}
