// Gather/scatter copy kernels for descriptor lists and the C ABI that plans and launches
// them (declared in include/nixl_amd_hip.h).
//
// Data layout of a plan in HBM
//   16-byte-aligned descriptors of 256 B to 8 KiB, and longer ones whose source or
//   destination does not start on a 128-byte line, become pieces of at most 4 KiB: a
//   16-byte record {src, dst | (units - 1) << 56} and one wavefront each
//   (wavefront-per-descriptor for anything up to 4 KiB); pieces after the first start on a
//   destination line.
//   Longer line-aligned ones are chunks of 64*UPL 16-byte units; one wavefront moves one
//   chunk: lane l moves units k*64 + l of the chunk, k < UPL, so every load/store instruction
//   of a wave touches 1 KiB of consecutive bytes.  A chunk is a 16-byte record {src address,
//   dst address} in `uniform[]`; the uniform kernel reads its record with one scalar load and
//   issues UPL 128-bit loads and UPL 128-bit stores per lane with wave-uniform base addresses —
//   no search, no LDS, few registers.  The end of a descriptor that is no whole number of
//   chunks is one more, of as many units as it needs (their number rides in the record's top bytes).
//   Tiny ones (below 256 B) are concatenated, in request order, into one virtual stream measured
//   in 16-byte units and cut into such chunks; the mixed kernel stages the descriptors a chunk
//   touches (span[c] = {first, last}; src[j], dst[j], prefix[j] = first unit of descriptor j,
//   prefix[n] = total) in a per-wave LDS slice and walks them.
//   Descriptors that are not 16-byte aligned in src, dst and len are cut into byte-range
//   work items of at most 4 KiB (16 of many long ones) handled by a third, byte-exact kernel; a
//   long one whose source and destination lie alike inside their 128-byte lines is chunks as well,
//   unless the request is small and brings no other chunks.
//   Lists of equal-length, line-aligned descriptors of whole chunks (KV blocks) take none of
//   these steps: one pass writes their records, or, when the request is two index vectors
//   into two strided runs, a kernel writes them from the indices on the device.  Arenas and
//   the pinned buffers they are uploaded from are pooled.
//
// What is equal to the reference: the bytes.  For every descriptor, in list order,
// dst[0..len) = src[0..len), the result of the per-descriptor put/get loop at
// src/plugins/ucx/ucx_backend.cpp:1216-1244.  Descriptors of one request must not
// overlap each other's destination ranges (the reference's puts are unordered too).
#include <algorithm>
#include <atomic>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <thread>
#include <type_traits>
#include <vector>

#if defined(__x86_64__)
#include <immintrin.h>
#endif

#include "common.h"

namespace {

constexpr int kMixedWaves = 4; // waves per workgroup of the mixed and byte-path kernels
constexpr int kMixedThreads = kWaveSize * kMixedWaves;
constexpr int kGenericLoads = 4; // 16-byte loads a lane keeps in flight for a byte-path work item
// Reach of an item, from the destination line it starts in: one round of those loads, or (a few
// long tensors, where the items are what the plan's making costs) four.
constexpr uint32_t kGenericRound = kWaveSize * kGenericLoads * 16, kGenericItemBytes = 4 * kGenericRound;
constexpr int kMaxLdsDescs = 64; // descriptors a wave stages in LDS for one chunk
constexpr int kNumXcd = 8; // accelerator dies; workgroup i is dispatched to die i % 8

struct UniformRec {
    uint64_t src;
    uint64_t dst;
};

// The record of a chunk that is not whole, the end of a descriptor: its 16-byte units, less one, in
// the top bytes of the two addresses, and the sign of dst, by which it is known.
constexpr uint64_t kEndAddress = (1ull << 56) - 1;

__device__ __forceinline__ UniformRec
end_rec(uint64_t src, uint64_t dst, uint32_t units) {
    const uint64_t more = units - 1; // < 1024
    return UniformRec{src | more >> 7 << 56, dst | more << 57 >> 1 | 1ull << 63};
}

__device__ __forceinline__ uint32_t
end_units(uint64_t src, uint64_t dst) {
    return (static_cast<uint32_t>(src >> 56) << 7 | (static_cast<uint32_t>(dst >> 56) & 127u)) + 1u;
}

struct MixedArgs {
    const uint64_t *src; // [n]
    const uint64_t *dst; // [n]
    const uint64_t *prefix; // [n + 1], units
    const uint2 *span; // [n_mixed], {first desc, last desc} of a chunk
    uint64_t total_units;
    uint32_t n_mixed;
};

// A piece of a small descriptor: at most kPieceUnits (256) 16-byte units, one wavefront's work.
// 16 bytes a record: the unit count, less one, rides in the top byte of the destination
// address (device and pinned host addresses stay far below 2^56; the host checks it).
struct PieceRec {
    uint64_t src;
    uint64_t dst_units; // dst | (units - 1) << 56
};
constexpr int kPieceUnitsShift = 56;

// Lengths of the entries of a list that stays on the device: what the piece kernel is made for.
constexpr uint32_t kListMinBytes = 128, kListMaxBytes = 8176;

// A byte range of at most kGenericItemBytes, 16 bytes a record like a piece: the length, less
// one, rides in the top bytes of the two addresses (low eight bits in dst's).
struct GenericItem {
    uint64_t src_len; // src | (len - 1) >> 8 << 56
    uint64_t dst_len; // dst | ((len - 1) & 255) << 56
};

// 16-byte vector in the global address space, so that accesses compile to
// global_load/store_dwordx4 rather than flat instructions.  Nothing is said of its alignment: the
// first and last chunks of odd tensors and the items of the byte path start anywhere.  The
// hardware takes such addresses, and aligned ones compile to the same instructions.
using v4u = __attribute__((__vector_size__(4 * sizeof(unsigned)))) unsigned;
using v4u_any = __attribute__((__vector_size__(4 * sizeof(unsigned)), __aligned__(1))) unsigned;
using gv4_ptr = __attribute__((address_space(1))) v4u_any *;
using gv4_cptr = const __attribute__((address_space(1))) v4u_any *;

// Cache policy of a plan's loads and stores (tuning field `nontemporal`), measured on MI355X
// with 16 KiB blocks (TB/s of traffic; sequential = consecutive descriptors adjoin):
//                                     seq->seq  random->seq  seq->random  random->random
//   1  nt loads,    nt stores           6.66       6.28         5.76          5.12
//   2  plain loads, plain stores        6.44       5.30         5.80          5.12
//   3  plain loads, sc1 nt stores       6.65       6.07         5.90          5.31
//   4  nt loads,    sc1 nt stores       6.71       6.35         5.80          5.15
// "sc1 nt" is a streaming store with device scope.  A plan whose destinations adjoin or
// advance by a constant step takes 4, any other plan 3; and 3 any plan whose payload is read and
// written inside the last-level cache of 256 MiB (copy_policy): up to 112 MiB, and up to 88 where sources follow
// one another.  Policies 4 and 3 there, us from launch to end, three requests with buffers of their own in turn (and one
// again and again):
//                                     64 MiB       88 MiB       96 MiB       104 MiB      112 MiB
//   one descriptor                    28.0 25.9    35.1 33.5    37.6 38.6    39.9 41.1    42.5 43.6 (42.3 38.9)
//   16 KiB, both sides following      28.5 25.9    36.3 35.7    39.0 39.4    41.2 41.9    43.9 44.3 (43.9 39.7)
//   16 KiB, destinations a step on    28.2 26.0    36.9 37.1    38.4 39.2    41.5 42.1    44.0 44.8 (43.9 39.7)
//   16 KiB gathered                   30.2 28.1    38.3 36.9    41.2 39.2    43.7 42.2    46.2 45.8 (46.1 40.6)
//   1 MiB gathered                                 37.8 36.4    40.2 39.1    43.0 42.0    45.2 44.1 (44.6 41.2)
//   2 KiB gathered (pieces)                        40.5 35.9    42.9 42.4    45.9 45.4    49.7 49.3 (49.5 42.0)
//   16 KiB scattered                  32.1 26.5    40.7 37.0    43.7 43.0    46.6 46.1    49.1 49.1 (49.3 40.0)
// 16 KiB gathered 128 MiB 51.5 and 51.9 (51.1 45.3), 144 MiB 56.9 and 58.5.  At 16 and 32 MiB 3 is 0.3 to 2.6 faster.
constexpr int kPolNtNt = 1, kPolPlain = 2, kPolPlainSc1Nt = 3, kPolNtSc1Nt = 4;
constexpr uint64_t kInLastLevelCache = 112ull << 20, kFollowingInLastLevelCache = 88ull << 20; // of payload

// `regular`: destinations adjoin, advance by a constant step or are sorted, or the copy does not depend on it.
// `following`: so do sources adjoin.
constexpr int
copy_policy(uint64_t payload, bool regular, bool following) {
    return regular && payload > (following ? kFollowingInLastLevelCache : kInLastLevelCache) ? kPolNtSc1Nt : kPolPlainSc1Nt;
}

template<int POL>
__device__ __forceinline__ v4u
load16(uint64_t addr) {
    gv4_cptr g = (gv4_cptr)(addr);
    if constexpr (POL == kPolNtNt || POL == kPolNtSc1Nt)
        return __builtin_nontemporal_load(g);
    else
        return *g;
}

template<int POL>
__device__ __forceinline__ void
store16(uint64_t addr, const v4u &v) {
    gv4_ptr g = (gv4_ptr)(addr);
    if constexpr (POL == kPolNtNt)
        __builtin_nontemporal_store(v, g);
    else if constexpr (POL == kPolPlain)
        *g = v;
    else
        // The compiler does not see that this is a store of more than two registers, after which they
        // may not be written for two wait states: chunks of two units a lane lost half of a lane's
        // 16 bytes to the address of the next store.
        asm volatile("global_store_dwordx4 %0, %1, off sc1 nt\n\ts_nop 1" : : "v"(g), "v"(v) : "memory");
}

// The same for a line that is not written whole, without the streaming hint: with it such a store goes to memory
// as a partial write at once.
template<int POL>
__device__ __forceinline__ void
store16_part(uint64_t addr, const v4u &v) {
    if constexpr (POL == kPolPlain)
        store16<POL>(addr, v);
    else
        asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" : : "v"((gv4_ptr)(addr)), "v"(v) : "memory");
}

// Stores 16 bytes that the kernel behind this one reads, through the die's cache as it goes: what a
// kernel leaves in there is written back when it ends, in front of the next one's start.  Requests of
// 1280, 4096 and 3904 blocks by index, launch to end: 18.6 -> 18.3 us, 26.0 -> 25.6 and 26.9 -> 26.4.  Non-temporal
// stores send the records to memory and the next kernel there for them: 19.0, 26.4 and 27.1.  (The kernel that uploads the
// 108 KB of items of 3000 byte descriptors takes 4.8 either way.)
template<class T>
__device__ __forceinline__ void
store_ahead(T *at, const T &x) {
    static_assert(sizeof(T) == 16);
    v4u v;
    __builtin_memcpy(&v, &x, 16);
    store16_part<kPolPlainSc1Nt>(reinterpret_cast<uint64_t>(at), v);
}

// Workgroups are handed to the 8 dies round-robin.  With the swizzle on, die x works
// through one contiguous eighth of the record array instead of every eighth record.
__device__ __forceinline__ uint32_t
logical_workgroup(uint32_t n_wgs, bool swizzle) {
    const uint32_t b = blockIdx.x;
    if (!swizzle) return b;
    const uint32_t per = (n_wgs + kNumXcd - 1) / kNumXcd;
    return (b % kNumXcd) * per + b / kNumXcd; // may be >= n_wgs; caller checks
}

// One wavefront per full, single-descriptor chunk.  A record covers `chunks_per_rec`
// consecutive chunks of one descriptor (1 when the runs of such chunks differ in length;
// with equal-length descriptors, e.g. KV blocks, one record per descriptor), so that the
// record array stays small next to the payload.
template<int UPL, int POL, int WAVES>
__global__ void __launch_bounds__(kWaveSize *WAVES)
copy_uniform_kernel(const UniformRec *recs, uint32_t first_chunk, uint32_t n_chunks, uint32_t n_wgs, int swizzle, FastDiv chunks_per_rec) {
    const uint32_t lane = threadIdx.x & (kWaveSize - 1);
    const uint32_t wave = threadIdx.x / kWaveSize;
    const uint32_t wg = logical_workgroup(n_wgs, swizzle != 0);
    if (wg >= n_wgs || wg * WAVES + wave >= n_chunks) return;
    const uint32_t c = uniform(first_chunk + wg * WAVES + wave); // n_chunks, n_wgs: of this launch
    uint32_t chunk;
    const uint32_t r = chunks_per_rec.quotient(c, chunk);
    const uint64_t off = static_cast<uint64_t>(chunk) * (kWaveSize * UPL * 16u) + lane * 16u;
    // The record is the same for every lane and does not change while the kernel runs: read
    // through the constant address space it comes with ONE scalar load (left as an ordinary
    // global access the compiler makes it a 16-byte vector load by all 64 lanes, followed by
    // four lane-0 read-outs).
    const auto *words = reinterpret_cast<const __attribute__((address_space(4))) uint64_t *>(reinterpret_cast<uintptr_t>(recs + r));
    const uint64_t s = words[0] + off; // UniformRec::src
    const uint64_t d = words[1] + off; // UniformRec::dst
    v4u v[UPL];
    if (static_cast<int64_t>(words[1]) < 0) {
        const uint32_t units = end_units(words[0], words[1]);
#pragma unroll
        for (int k = 0; k < UPL; ++k)
            if (k * kWaveSize + lane < units) v[k] = load16<POL>((s & kEndAddress) + k * (kWaveSize * 16u));
#pragma unroll
        for (int k = 0; k < UPL; ++k)
            if (k * kWaveSize + lane < units) store16<POL>((d & kEndAddress) + k * (kWaveSize * 16u), v[k]);
        return;
    }
#pragma unroll
    for (int k = 0; k < UPL; ++k)
        v[k] = load16<POL>(s + k * (kWaveSize * 16u));
#pragma unroll
    for (int k = 0; k < UPL; ++k)
        store16<POL>(d + k * (kWaveSize * 16u), v[k]);
}

// The same for a request of a few blocks, whose records travel as the kernel's arguments: nothing
// is uploaded, so nothing has to be waited for between the making of the request and its copy.
// 64 blocks of 32 KiB, from the making of the request to its end: 51 us with uploaded records, 19
// with these.  128 records are 2 KiB of the 4 KiB a launch can carry.
constexpr uint32_t kInlineRecs = 128;

struct InlineRecs {
    UniformRec rec[kInlineRecs];

    __device__ __forceinline__ UniformRec
    at(uint32_t r) const {
        return rec[r];
    }
};

// A request of some more, by index into two lists of one stride each: what travels is the indices, and every wave
// makes its record of them.  A vector that is consecutive is its first index.  Requests made, moved and waited for, us, with
// records that a kernel makes in front of the copy and so, blocks of 8 KiB gathered: 192 17.4 and 14.8, 512 17.6 and 14.9, 896
// 18.8 and 15.5; scattered 896 17.9 and 15.5.  896 words are 3.5 of the 4 KiB that a launch can carry; 16-bit indices
// would make twice as many blocks fit, of pools with few entries.
constexpr uint32_t kInlineIndices = 896;

struct InlineIndices {
    struct Side {
        uint64_t base, stride;
        uint32_t first; // index, of a consecutive vector
        uint32_t listed; // ~0 where the vector is in `index`, from `place` on, 0 where it is consecutive (and `place` 0)
        uint32_t place;
    };

    Side src, dst;
    int32_t index[kInlineIndices];

    __device__ __forceinline__ UniformRec
    at(uint32_t r) const { // r < n <= kInlineIndices
        const auto address = [&](const Side &s) {
            // no branch, so that the words of both sides are loaded together and behind nothing but the sides
            const uint32_t word = static_cast<uint32_t>(index[s.place + r]);
            return s.base + ((word & s.listed) | ((s.first + r) & ~s.listed)) * s.stride;
        };
        return UniformRec{address(src), address(dst)};
    }
};

// A request by index of any length whose vectors repeat themselves: the blocks of some sequences in every layer of
// a cache, listed layer by layer or block by block.  Seen as a grid, rows of equal length, index (row, column)
// of a listed side is an id of the column and `step` times the row, or an id of the row and `step` times the
// column; a side that is not listed is consecutive.  The ids, counted from the smallest one of a side, take 16 bits.
// No records are made and nothing is uploaded.  Requests made, moved and waited for, us, with records and so: 900 blocks of 1 KiB 15.0 and
// 12.4, 65 520 44.0 and 31.9; of 4 KiB 2048 15.9 and 14.5, 8192 22.8 and 19.3, 32 768 60.2 and 53.5, 131 072 204 and 181; 15 250 of 9 KiB 62.4
// and 58.5; 8192 of 16 KiB 54.5 and 51.9, 65 520 341 and 333; 2048 of 128 KiB 92.4 and 90.0.  What it costs the host to see
// that indices are no grid is 0.1 to 0.3 us.
constexpr uint32_t kGridIds = 1792;
constexpr uint32_t kMaxGridRows = 65535; // the second dimension of a launch

struct GridIndices {
    struct Side {
        uint64_t base, stride;
        uint32_t first; // index, of a consecutive vector; what ids are counted from
        uint32_t step;
        uint32_t listed; // ~0 where the ids are in `ids`, from `place` on, 0 where the vector is consecutive (and `place` 0)
        uint32_t place;
    };

    Side src, dst;
    FastDiv row_length;
    uint32_t by_column; // whose ids are listed: ~0 those of the columns, 0 those of the rows
    alignas(4) uint16_t ids[kGridIds];

    __device__ __forceinline__ UniformRec
    at(uint32_t r) const {
        uint32_t column;
        const uint32_t row = row_length.quotient(r, column);
        return at(row, column, r);
    }

    __device__ __forceinline__ UniformRec
    at(uint32_t row, uint32_t column, uint32_t r) const {
        const uint32_t named = (column & by_column) | (row & ~by_column), other = row ^ column ^ named; // named < kGridIds
        const auto address = [&](const Side &s) {
            // no branch, as above
            const uint32_t i = s.place + named;
            uint32_t two; // by a scalar load, which a word alone can have
            __builtin_memcpy(&two, ids + (i & ~1u), sizeof(two));
            const uint32_t id = (two >> (i % 2 * 16)) & 0xffffu;
            return s.base + (s.first + ((id + other * s.step) & s.listed) + (r & ~s.listed)) * s.stride;
        };
        return UniformRec{address(src), address(dst)};
    }
};

template<int POL, typename Recs>
__global__ void __launch_bounds__(kWaveSize)
copy_inline_kernel(Recs recs, FastDiv chunks_per_rec) {
    uint32_t chunk;
    const uint32_t r = chunks_per_rec.quotient(blockIdx.x, chunk);
    const uint64_t off = static_cast<uint64_t>(chunk) * (kWaveSize * 16u) + threadIdx.x * 16u;
    const UniformRec rec = recs.at(r);
    store16<POL>(rec.dst + off, load16<POL>(rec.src + off));
}

// Of such a request of many blocks: a row of the launch a row of the grid, so that a wave divides once (36 600 blocks of 9 KiB 121.5 -> 118.4
// us; with a third dimension instead of the other division, so few workgroups a row, 142.9).
template<int POL>
__global__ void __launch_bounds__(kWaveSize)
copy_grid_kernel(GridIndices grid, FastDiv chunks_per_rec) {
    uint32_t chunk;
    const uint32_t column = chunks_per_rec.quotient(blockIdx.x, chunk);
    const uint64_t off = static_cast<uint64_t>(chunk) * (kWaveSize * 16u) + threadIdx.x * 16u;
    const UniformRec rec = grid.at(blockIdx.y, column, blockIdx.y * grid.row_length.divisor + column);
    store16<POL>(rec.dst + off, load16<POL>(rec.src + off));
}

// ---- the end of a launch as a word in host memory ----------------------------------------------
//
// A host that polls a word sees a transfer's end sooner than one that asks for an event behind it: the
// event is a packet of its own that the command processor takes up, releases caches for and signals, and
// asking for it is a call into the runtime.  Blocks launched and waited for, us, mean (and the 90th percentile):
// event, word of a one-wave kernel behind the copy, word of the copy's last workgroup:
//   1 x 8 KiB     14.0 (17.2)  11.2 (11.4)   8.4 ( 8.6)
//   64 x 32 KiB   14.5 (19.0)  11.2 (12.6)  10.4 (10.5)
//   128 x 64 KiB  15.9 (20.6)  11.8 (12.7)  11.8 (11.9)
//   128 x 1 MiB   53.4 (54.7)  49.4 (50.5)  53.0 (54.3)
// So a copy of a few blocks counts its own workgroups, and others are followed by done_kernel.
constexpr int kDoneSlots = 128; // launches of a device that can be watched at once; others take an event
// Up to kDoneOneGroup workgroups are counted on one address, more in kDoneGroups groups and then the groups
// (an arrival at an address takes 11 ns behind another one, 512 of them 5.8 us; a second count 0.7).
constexpr int kDoneGroups = 16;
constexpr uint32_t kDoneOneGroup = 64;
constexpr int kDoneLine = 32; // words of a 128-byte line
__device__ uint32_t g_done_counts[kDoneSlots][kDoneGroups + 1][kDoneLine]; // zero whenever no launch uses the slot

struct Done {
    uint32_t *counts; // [kDoneGroups + 1][kDoneLine]; the last one counts groups
    uint32_t *word; // pinned host memory
    uint32_t value;
};

// One thread of every workgroup, when all that the workgroup stored has reached memory.  The last one
// leaves the counts at zero, and writes the word behind that.
__device__ __forceinline__ void
arrive(const Done &done) {
    const uint32_t n = gridDim.x, groups = n <= kDoneOneGroup ? 1 : kDoneGroups, g = blockIdx.x % groups;
    const auto last = [](uint32_t *count, uint32_t of) {
        if (__hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u != of) return false;
        __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        return true;
    };
    if (!last(done.counts + g * kDoneLine, (n - g + groups - 1) / groups)) return;
    if (groups > 1 && !last(done.counts + kDoneGroups * kDoneLine, groups)) return;
    __hip_atomic_store(done.word, done.value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ void __launch_bounds__(kWaveSize)
done_kernel(uint32_t *word, uint32_t value) {
    if (threadIdx.x == 0) __hip_atomic_store(word, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// copy_inline_kernel for a launch that tells its own end: few workgroups of 16 chunks each, so that
// there are few to count.  Only with the policies whose stores are written through to memory
// (device scope): their completion is what s_waitcnt waits for, no cache has to be written back.
constexpr int kDoneWaves = 8, kDoneChunks = 2; // chunks a wave

template<int POL, typename Recs>
__global__ void __launch_bounds__(kWaveSize *kDoneWaves)
copy_inline_done_kernel(Recs recs, FastDiv chunks_per_rec, uint32_t n_chunks, Done done) {
    static_assert(POL == kPolPlainSc1Nt || POL == kPolNtSc1Nt);
    const uint32_t lane = threadIdx.x & (kWaveSize - 1);
    const uint32_t first = uniform(blockIdx.x * (kDoneWaves * kDoneChunks) + threadIdx.x / kWaveSize);
    v4u v[kDoneChunks];
    uint64_t to[kDoneChunks];
#pragma unroll
    for (int j = 0; j < kDoneChunks; ++j) {
        const uint32_t c = first + j * kDoneWaves;
        if (c >= n_chunks) continue;
        uint32_t chunk;
        const uint32_t r = chunks_per_rec.quotient(c, chunk);
        const uint64_t off = static_cast<uint64_t>(chunk) * (kWaveSize * 16u) + lane * 16u;
        const UniformRec rec = recs.at(r);
        to[j] = rec.dst + off;
        v[j] = load16<POL>(rec.src + off);
    }
#pragma unroll
    for (int j = 0; j < kDoneChunks; ++j)
        if (first + j * kDoneWaves < n_chunks) store16<POL>(to[j], v[j]);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // the stores are inline asm, which the compiler does not wait for
    __syncthreads();
    if (threadIdx.x == 0) arrive(done);
}

// Moves the arrays of a plan from the pinned buffer they were built in to the device, 16 bytes a
// lane.  A copy engine is slower for all but large plans: it has to be started and its end
// signalled to the kernels behind it (90 KB: 6.5 us here, 8.5 there and the signal on top), while
// beyond a MiB it moves 63 GB/s and lanes reading over the bus 26.
__global__ void __launch_bounds__(256)
upload_kernel(uint4 *__restrict__ dst, const uint4 *__restrict__ src, size_t n) {
    for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += static_cast<size_t>(gridDim.x) * blockDim.x)
        store_ahead(dst + i, src[i]);
}

// One wavefront per piece: the descriptor's own {src, dst, units} record, up to
// kPieceLoads 128-bit loads in flight per lane, then the stores.  No search and no LDS:
// the shape for descriptors of a few hundred bytes to a few KiB.

// Loads of pieces are ordinary or non-temporal by the bytes of their request alone.  One request again and
// again | three with buffers of their own in turn, us from launch to end, ordinary and non-temporal loads (and
// non-temporal loads and stores throughout), 512 B to 4 KiB, 1024 pieces 8.8 8.8 (9.2) | 8.8 8.8 (9.2); 8192 10.7 11.8 (13.6) |
// 12.2 14.0 (13.9); 16 384 14.6 18.3 (20.0) | 17.2 20.3 (20.3); 65 536, 113 MB, 42.4 54.5 (57.9) | 54.4 54.6 (58.6); 131 072, 225 MB,
// 90.8 99.6 (108) | 106.9 99.4 (108); 512 B to 2 KiB, 131 072, 144 MB, 62.8 67.7 (76.6) | 74.9 67.7 (76.5).
constexpr int kPieceLoads = 4;
constexpr uint32_t kPieceUnits = kWaveSize * kPieceLoads; // 4 KiB

// Workgroups are handed to the 8 dies round-robin; die x takes the x-th eighth of the records
// (grid = a multiple of 8 workgroups, `per_die` of them a die), so that a line of records is
// fetched into one die's cache instead of into several: with records dealt out round-robin the
// record lines were read 3.3 times over.
template<int POL, int LOADS, int WAVES>
__global__ void __launch_bounds__(kWaveSize *WAVES)
copy_piece_kernel(const PieceRec *__restrict__ recs, uint32_t n_recs, uint32_t per_die) { // recs, n_recs: of this launch
    const uint32_t lane = threadIdx.x & (kWaveSize - 1);
    const uint32_t wg = (blockIdx.x % kNumXcd) * per_die + blockIdx.x / kNumXcd;
    const uint32_t p = uniform(wg * WAVES + threadIdx.x / kWaveSize);
    if (p >= n_recs) return;
    const PieceRec packed = recs[p]; // same address in every lane of the wave: a scalar load
    struct {
        uint64_t src, dst;
    } rec{packed.src, packed.dst_units & ((1ull << kPieceUnitsShift) - 1ull)};
    const uint32_t units = static_cast<uint32_t>(packed.dst_units >> kPieceUnitsShift) + 1u; // >= 1
    // Lane 0 of every instruction sits on a 128-byte line of the destination: the piece's
    // units are shifted up by the destination's offset inside its line (the plan cuts pieces
    // so that shift + units <= kPieceUnits), and each store instruction then writes whole
    // lines except at the two ends of the piece.  A line written half by one instruction
    // and half by the next would go out as two partial writes.
    //
    // What bounds it is the memory's writes at random places, and of those the partial ones: the lines
    // at the two ends are stored without the streaming hint.  262 144 descriptors, log-uniform
    // lengths, us with the hint everywhere and so: 512 B to 4 KiB at 16-byte addresses 206 and 191, 512 B to
    // 2 KiB 141 and 126, 256 B to 2 KiB 115 and 104; at 64-byte and 128-byte addresses no difference (187 and 186, 178
    // and 178).  Whole lines without it 258; only what is no whole half of a line without it 208.
    const uint32_t shift = static_cast<uint32_t>(rec.dst >> 4) & 7u;
    const uint32_t end = shift + units;
    // Loads are unconditional (a lane outside the piece re-reads its first or last unit) so
    // that all of them are in flight together; only the stores are predicated.
    v4u v[LOADS];
#pragma unroll
    for (int k = 0; k < LOADS; ++k) {
        const uint32_t at = k * kWaveSize + lane;
        const uint32_t u = min(at < shift ? 0u : at - shift, units - 1);
        v[k] = load16<POL>(rec.src + u * 16ull);
    }
#pragma unroll
    for (int k = 0; k < LOADS; ++k) {
        const uint32_t at = k * kWaveSize + lane, line = at & ~7u; // first unit of the lane's line
        if (at < shift || at >= end) continue;
        if (line >= shift && line + 8 <= end)
            store16<POL>(rec.dst + (at - shift) * 16ull, v[k]);
        else
            store16_part<POL>(rec.dst + (at - shift) * 16ull, v[k]);
    }
}

// One wavefront per chunk of the stream of tiny descriptors.
template<int UPL, int POL>
__global__ void __launch_bounds__(kMixedThreads)
copy_mixed_kernel(MixedArgs a) {
    constexpr uint32_t kChunkUnits = kWaveSize * UPL;
    __shared__ uint64_t lds_prefix[kMixedWaves][kMaxLdsDescs + 1];
    __shared__ uint64_t lds_src[kMixedWaves][kMaxLdsDescs];
    __shared__ uint64_t lds_dst[kMixedWaves][kMaxLdsDescs];

    const uint32_t lane = threadIdx.x & (kWaveSize - 1);
    const uint32_t wave = threadIdx.x / kWaveSize;
    const uint32_t n_waves = gridDim.x * kMixedWaves;

    for (uint32_t m = uniform(blockIdx.x * kMixedWaves + wave); m < a.n_mixed; m += n_waves) {
        const uint2 sp = a.span[m];
        const uint32_t j0 = uniform(sp.x);
        const uint32_t j1 = uniform(sp.y);
        const uint64_t u0 = static_cast<uint64_t>(m) * kChunkUnits;
        const uint64_t remaining = a.total_units - u0; // > 0
        const uint32_t n_units = remaining < kChunkUnits ? static_cast<uint32_t>(remaining) : kChunkUnits;
        const uint32_t nd = j1 - j0 + 1;

        if (nd <= kMaxLdsDescs) {
            // Stage this chunk's descriptors in the wave's LDS slice, then each lane walks
            // forward through them as its unit index grows by 64 per step.  Only this
            // wave touches the slice, and a wave's LDS operations complete in order.
            __builtin_amdgcn_wave_barrier();
            if (lane < nd) {
                lds_prefix[wave][lane] = a.prefix[j0 + lane];
                lds_src[wave][lane] = a.src[j0 + lane];
                lds_dst[wave][lane] = a.dst[j0 + lane];
            }
            if (lane == 0) lds_prefix[wave][nd] = a.prefix[j0 + nd];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

            uint32_t jj = 0;
            uint64_t sa[UPL], da[UPL];
            v4u v[UPL];
#pragma unroll
            for (int k = 0; k < UPL; ++k) {
                const uint32_t i = k * kWaveSize + lane;
                sa[k] = 0;
                da[k] = 0;
                if (i < n_units) {
                    const uint64_t u = u0 + i;
                    while (jj + 1 < nd && lds_prefix[wave][jj + 1] <= u)
                        ++jj;
                    const uint64_t off = (u - lds_prefix[wave][jj]) * 16u;
                    sa[k] = lds_src[wave][jj] + off;
                    da[k] = lds_dst[wave][jj] + off;
                }
            }
#pragma unroll
            for (int k = 0; k < UPL; ++k)
                if (sa[k]) v[k] = load16<POL>(sa[k]);
#pragma unroll
            for (int k = 0; k < UPL; ++k)
                if (da[k]) store16<POL>(da[k], v[k]);
            __builtin_amdgcn_wave_barrier();
        } else {
            // More than 64 tiny descriptors in one chunk: bisect the global prefix array.
            for (uint32_t i = lane; i < n_units; i += kWaveSize) {
                const uint64_t u = u0 + i;
                uint32_t lo = j0, hi = j1;
                while (lo < hi) {
                    const uint32_t mid = lo + (hi - lo + 1) / 2;
                    if (a.prefix[mid] <= u)
                        lo = mid;
                    else
                        hi = mid - 1;
                }
                const uint64_t off = (u - a.prefix[lo]) * 16u;
                store16<POL>(a.dst[lo] + off, load16<POL>(a.src[lo] + off));
            }
        }
    }
}

// One wavefront per byte-range work item; correct for any alignment and length.  An item ends
// at most kGenericRound (or kGenericItemBytes) behind the destination line it starts in (the plan
// cuts them so), so its body of whole 16-byte units is one round (or four) of kGenericLoads
// instructions with lane 0 of each on a destination line, as in the piece kernel; loads take
// their 16 bytes from any address.
// All loads of a round (body, up to 15 head and 15 tail bytes) are in flight before its first
// store: what bounds a list of a few thousand such descriptors is that round trip and the
// number of waves sharing it, not bytes (3000 descriptors of up to 64 KiB, 18 MB: 7 us; with items
// of 16 KiB whose lanes had one load in flight a 64 KiB descriptor alone was 64 of those trips
// in a row on four waves).
__global__ void __launch_bounds__(kMixedThreads)
copy_generic_kernel(const GenericItem *items, uint32_t n_items) {
    using byte_ptr = __attribute__((address_space(1))) uint8_t *;
    using byte_cptr = const __attribute__((address_space(1))) uint8_t *;
    const uint32_t lane = threadIdx.x & (kWaveSize - 1);
    const uint32_t wave = threadIdx.x / kWaveSize;
    const uint32_t n_waves = gridDim.x * kMixedWaves;
    for (uint32_t it = uniform(blockIdx.x * kMixedWaves + wave); it < n_items; it += n_waves) {
        const uint64_t src_len = uniform64(items[it].src_len), dst_len = uniform64(items[it].dst_len);
        constexpr uint64_t kAddress = (1ull << kPieceUnitsShift) - 1ull;
        const uint64_t src = src_len & kAddress, dst = dst_len & kAddress;
        const uint32_t len = (static_cast<uint32_t>(src_len >> kPieceUnitsShift) << 8 | static_cast<uint32_t>(dst_len >> kPieceUnitsShift)) + 1u;
        // bytes until dst is 16-byte aligned (at most 15), whole units, the rest
        const uint32_t head = min(static_cast<uint32_t>(-dst) & 15u, len);
        const uint32_t body = (len - head) / 16u;
        const uint32_t done = head + body * 16u;
        const uint32_t tail = len - done; // < 16
        const uint32_t shift = (static_cast<uint32_t>(dst + head) >> 4) & 7u; // body's offset inside its line

        uint8_t first = 0, last = 0;
        if (lane < head) first = *(byte_cptr)(src + lane);
        if (lane < tail) last = *(byte_cptr)(src + done + lane);
        // unconditional, as in the piece kernel: a lane outside the body re-reads its first or last
        // unit (an item without a body has no round)
        const uint32_t end = body ? body + shift : 0;
        for (uint32_t round = 0; round < end; round += kGenericLoads * kWaveSize) {
            v4u v[kGenericLoads];
#pragma unroll
            for (int k = 0; k < kGenericLoads; ++k) {
                const uint32_t at = round + k * kWaveSize + lane;
                const uint32_t u = min(at < shift ? 0u : at - shift, body - 1);
                v[k] = *(gv4_cptr)(src + head + u * 16ull);
            }
#pragma unroll
            for (int k = 0; k < kGenericLoads; ++k) {
                const uint32_t at = round + k * kWaveSize + lane;
                if (at >= shift && at - shift < body) store16<kPolNtNt>(dst + head + (at - shift) * 16ull, v[k]);
            }
        }
        if (lane < head) *(byte_ptr)(dst + lane) = first;
        if (lane < tail) *(byte_ptr)(dst + done + lane) = last;
    }
}

// Reorders the records of a scattering plan (sources that follow each other, destinations
// that do not) so that inside every window of 1024 records the destinations ascend.  Which
// record a wavefront takes does not change the bytes that arrive; it changes the order in
// which DRAM sees the writes: 16 KiB blocks scattered over a pool went from 5.8 to 6.1 TB/s.
//
// One workgroup per window and one record per thread, a bitonic network over one 64-bit key a
// record: its destination in lines (blocks start on 128-byte lines) and its place in
// the window, by which it finds its source afterwards.  Partners less than a wave apart exchange
// keys between lanes; 10 of the 55 steps go through LDS.  What bounds it is that chain.  Records of an
// indexed request are sorted before they are written at all: 65 536 of them 14.0 us, where writing them
// took 8.5 and sorting records of two words in LDS with a barrier a step 14.6, and a pass of that
// many blocks there and back 778 -> 770.
constexpr uint32_t kSortWindow = 1024;
constexpr int kSortPlaceBits = 10, kSortLineBits = 7;
static_assert(kSortWindow == 1u << kSortPlaceBits); // addresses below 2^61: user space ends at 2^57

// Thread i brings record i of the window (or none) and leaves with the i-th by destination.
__device__ __forceinline__ UniformRec
sort_window(const UniformRec &rec, bool in) {
    __shared__ uint64_t lds[kSortWindow];
    const uint32_t tid = threadIdx.x;
    uint64_t key = in ? rec.dst >> kSortLineBits << kSortPlaceBits | tid : ~0ull; // what is none sorts to the end
#pragma unroll
    for (uint32_t size = 2; size <= kSortWindow; size <<= 1) {
        const bool up = (tid & size) == 0;
#pragma unroll
        for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
            uint64_t other;
            if (stride >= kWaveSize) {
                __syncthreads();
                lds[tid] = key;
                __syncthreads();
                other = lds[tid ^ stride];
            } else {
                other = __shfl_xor(static_cast<unsigned long long>(key), static_cast<int>(stride));
            }
            const bool lower = (tid & stride) == 0; // the one of the two that keeps the smaller key in an ascending stretch
            key = (lower == up) == (key < other) ? key : other;
        }
    }
    __syncthreads();
    lds[tid] = rec.src;
    __syncthreads();
    return UniformRec{lds[key & (kSortWindow - 1)], key >> kSortPlaceBits << kSortLineBits};
}

__global__ void __launch_bounds__(kSortWindow)
sort_records_kernel(UniformRec *recs, uint32_t n) {
    const uint32_t i = blockIdx.x * kSortWindow + threadIdx.x;
    const UniformRec sorted = sort_window(i < n ? recs[i] : UniformRec{}, i < n);
    if (i < n) store_ahead(recs + i, sorted);
}

// Records of an indexed plan: block i goes from src_base + src_index[i] * src_stride to
// dst_base + dst_index[i] * dst_stride.  The index vectors are the only per-request data
// that crosses the bus, at most 8 bytes per block: one whose indices are consecutive (the staging
// side of a gather or a scatter) stays where it is.  65 536 pairs, both
// vectors read 15 us, one 8.5.
struct IndexVector {
    const int32_t *at; // null: first, first + 1, ...
    int32_t first;
};

__device__ __forceinline__ uint64_t
index_at(const IndexVector &v, uint32_t i) {
    return static_cast<uint64_t>(v.at ? v.at[i] : static_cast<int32_t>(v.first + i));
}

// Threads of a workgroup of the two kernels; SORTED: the records leave in the order of sort_window.
template<bool SORTED>
constexpr uint32_t kIndexThreads = SORTED ? kSortWindow : 256;

template<bool SORTED>
__global__ void __launch_bounds__(kIndexThreads<SORTED>)
index_records_kernel(UniformRec *recs, IndexVector src_index, IndexVector dst_index, uint32_t n, uint64_t src_base,
                     uint64_t src_stride, uint64_t dst_base, uint64_t dst_stride) {
    const uint32_t i = blockIdx.x * kIndexThreads<SORTED> + threadIdx.x;
    UniformRec rec{};
    if (i < n) rec = UniformRec{src_base + index_at(src_index, i) * src_stride, dst_base + index_at(dst_index, i) * dst_stride};
    if constexpr (SORTED) rec = sort_window(rec, i < n);
    if (i < n) store_ahead(recs + i, rec);
}

// Records of a plan whose waves made their own so far (InlineIndices, GridIndices; later_records).  A launch and its chain of
// loads: 300 listed blocks 2.2 us, a grid of 4096 2.8, of 131 072 3.1; sorted 32 640 8.6.
template<bool SORTED, typename Recs>
__global__ void __launch_bounds__(kIndexThreads<SORTED>)
later_records_kernel(UniformRec *recs, Recs from, uint32_t n) {
    const uint32_t i = blockIdx.x * kIndexThreads<SORTED> + threadIdx.x;
    UniformRec rec{};
    if (i < n) rec = from.at(i);
    if constexpr (SORTED) rec = sort_window(rec, i < n);
    if (i < n) store_ahead(recs + i, rec);
}

// The same for lists of several runs (a pool registered as several regions): index i of a
// list lies in the run r with first[r] <= i < first[r + 1], at base[r] + (i - first[r]) *
// stride[r].  The run tables (at most kMaxIndexRuns entries a side) are staged in LDS and
// searched by bisection.
constexpr uint32_t kMaxIndexRuns = 256;

__device__ __forceinline__ uint64_t
run_address(const uint64_t *first, const uint64_t *base, const uint64_t *stride, uint32_t n_runs, uint64_t index) {
    uint32_t lo = 0, hi = n_runs; // first[lo] <= index < first[hi] (first[n_runs] = infinity)
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (first[mid] <= index) lo = mid;
        else hi = mid;
    }
    return base[lo] + (index - first[lo]) * stride[lo];
}

template<bool SORTED>
__global__ void __launch_bounds__(kIndexThreads<SORTED>)
index_records_runs_kernel(UniformRec *recs, IndexVector src_index, IndexVector dst_index, uint32_t n,
                          const nixl_amd_copy_run_t *src_runs, uint32_t n_src, const nixl_amd_copy_run_t *dst_runs,
                          uint32_t n_dst) {
    __shared__ uint64_t first[2][kMaxIndexRuns], base[2][kMaxIndexRuns], stride[2][kMaxIndexRuns];
    for (uint32_t r = threadIdx.x; r < n_src; r += blockDim.x) {
        first[0][r] = src_runs[r].first_index;
        base[0][r] = src_runs[r].base;
        stride[0][r] = src_runs[r].stride;
    }
    for (uint32_t r = threadIdx.x; r < n_dst; r += blockDim.x) {
        first[1][r] = dst_runs[r].first_index;
        base[1][r] = dst_runs[r].base;
        stride[1][r] = dst_runs[r].stride;
    }
    __syncthreads();
    const uint32_t i = blockIdx.x * kIndexThreads<SORTED> + threadIdx.x;
    UniformRec rec{};
    if (i < n)
        rec = UniformRec{run_address(first[0], base[0], stride[0], n_src, index_at(src_index, i)),
                         run_address(first[1], base[1], stride[1], n_dst, index_at(dst_index, i))};
    if constexpr (SORTED) rec = sort_window(rec, i < n);
    if (i < n) store_ahead(recs + i, rec);
}

// Records of a listed plan: pair i joins entry src_index[i] of one prepared list with entry
// dst_index[i] of another, both resident on the device (nixl_amd_copy_list).  A thread per pair
// checks it (indices inside their lists, equal lengths) and writes the piece records of its
// descriptor: the first at recs[i], those of a descriptor that spans several pieces behind the
// n first ones, in whatever order the workgroups get there (the order of records decides
// nothing about the bytes that arrive).
//
// What bounds it is the way of the pairs over the bus, so they come in one of two forms, both read
// where they are in pinned host memory (every word is read once, a copy to the device first would
// only add its latency).  RUNS: stretches of pairs whose indices advance by one on both sides, as
// those of a request that names blocks of consecutive entries, are 16 bytes each, and a workgroup
// bisects the few that its pairs lie in; else the two vectors as they came, 8 bytes a pair.
//
// The verdict reaches the host through pinned memory, written by the workgroup that finishes last;
// the host waits for it, because a bad pair must fail the request.  A workgroup adds to the totals
// with two atomics, on two lines, and nothing in front of the verdict writes a cache back: a device-scope fence around the
// additions did, for records that only the next kernel reads.  Kernel time, medians under the profiler, with such fences,
// sums over a wave through LDS and one line; without them and with sums between lanes; and with two lines: runs of 64 pairs, 1024 pairs 9.3, 8.0 and
// 8.0 us, 16 384 9.6, 8.4 and 8.4, 65 536 10.3, 8.8 and 8.7, 262 144 13.8, 10.4 and 9.9; vectors, 1024 pairs 9.4, 8.6 and 8.4, 16 384 11.4,
// 10.2 and 10.3, 65 536 18.5, 17.1 and 17.4.
struct IndexRun {
    uint32_t first; // pair the run starts with; it ends where the next one starts
    uint32_t src, dst; // indices of that pair
    uint32_t unused;
};

// n < 2^31 pairs over the records a pair can have (plan_create_listed), so that a request's bytes stay
// below 2^43 and its workgroups below or at 2^21.
constexpr int kListBytesBits = 43;

struct ListTotals {
    unsigned long long bytes_arrived; // bytes of the good pairs | workgroups that have added theirs << kListBytesBits
    // records beyond the first of their pair | pairs that continue the pair before them inside one
    // dense run on both sides << 32
    alignas(128) unsigned long long extra_continued; // on a line of its own: additions to one line wait for each other
    uint32_t bad; // pairs that name no entry or join entries of different lengths
};

// Totals that are zero whenever no launch uses them (the workgroup that writes the verdict leaves them so), so
// that a request needs no launch in front of its records' to clear some: 2.2 us of its host and 1.5 and a gap of
// the GPU (passes of 4096 pairs of 512 B - 4 KiB 31.4 -> 28.8 us, 32 768 56.5 -> 54.4, 262 144 by 2.3).
// A request has a slot of its own while it waits for its verdict; with more than kListSlots at once the
// others clear totals in their plans.
constexpr int kListSlots = 64; // of a device
struct alignas(128) ListSlot {
    ListTotals totals;
};
__device__ ListSlot g_list_slots[kListSlots];

struct ListVerdict {
    unsigned long long bytes;
    uint32_t bad, continued, extra;
    uint32_t there; // set last
};

constexpr int kListThreads = 1024;
// Pairs a launch, where the vectors are sent as they came: while it reads them over the bus the host
// copies the next ones into the pinned buffer.
constexpr size_t kListSlice = 65536;
static_assert(kListSlice % kListThreads == 0);

struct ListArgs {
    PieceRec *recs; // [n * pieces a descriptor can have]
    const nixl_amd_copy_list_entry_t *src, *dst;
    uint32_t n_src, n_dst;
    const int32_t *src_index, *dst_index; // [n]
    const IndexRun *runs; // instead
    const uint32_t *run_of; // [n_workgroups + 1]: run that workgroup b's first pair lies in, then the last run
    uint32_t first_workgroup; // of this launch; a plan's pairs may come in several
    uint32_t n;
    uint32_t n_workgroups; // of all launches together
    ListTotals *totals; // zero, and zero again when the verdict is there
    ListVerdict *verdict;
};

template<bool RUNS>
__global__ void __launch_bounds__(kListThreads)
list_records_kernel(ListArgs a) {
    constexpr int kWaves = kListThreads / kWaveSize;
    static_assert(kListThreads * kListMaxBytes <= 0xffffffffu);
    __shared__ uint32_t wave_bytes[kWaves], wave_bad[kWaves], wave_continued[kWaves], wave_extra[kWaves], extra_at;
    __shared__ IndexRun runs[RUNS ? kListThreads + 1 : 1];
    __shared__ uint2 last[RUNS ? 1 : kWaves];
    const uint32_t workgroup = a.first_workgroup + blockIdx.x, i = workgroup * kListThreads + threadIdx.x;
    const int lane = threadIdx.x & (kWaveSize - 1), wave = threadIdx.x / kWaveSize;
    uint32_t si = 0, di = 0;
    bool follows; // the pair before this one names the entries before this one's
    if constexpr (RUNS) {
        const uint32_t r0 = a.run_of[workgroup], n_runs = a.run_of[workgroup + 1] - r0 + 1; // at most a run a pair and the next
        if (threadIdx.x < n_runs) runs[threadIdx.x] = a.runs[r0 + threadIdx.x];
        if (threadIdx.x == 0 && n_runs > kListThreads) runs[kListThreads] = a.runs[r0 + kListThreads];
        __syncthreads();
        uint32_t lo = 0, hi = n_runs; // runs[lo].first <= i < runs[hi].first
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) / 2;
            if (runs[mid].first <= i) lo = mid;
            else hi = mid;
        }
        si = runs[lo].src + (i - runs[lo].first);
        di = runs[lo].dst + (i - runs[lo].first);
        follows = i != runs[lo].first;
    } else {
        if (i < a.n) {
            si = static_cast<uint32_t>(a.src_index[i]);
            di = static_cast<uint32_t>(a.dst_index[i]);
        }
        // the pair before this one: the neighbour's, for the first lane of a wave by LDS and for that of
        // the workgroup a load (one a wave is a quarter more requests over the bus)
        uint32_t sp = __shfl_up(si, 1), dp = __shfl_up(di, 1);
        uint32_t first_sp = 0, first_dp = 0;
        if (threadIdx.x == 0 && i > 0) {
            first_sp = static_cast<uint32_t>(a.src_index[i - 1]);
            first_dp = static_cast<uint32_t>(a.dst_index[i - 1]);
        }
        if (lane == kWaveSize - 1) last[wave] = make_uint2(si, di);
        __syncthreads();
        if (lane == 0) {
            sp = wave ? last[wave - 1].x : first_sp;
            dp = wave ? last[wave - 1].y : first_dp;
        }
        follows = i > 0 && si == sp + 1 && di == dp + 1;
    }
    const bool here = i < a.n;
    const bool named = here && si < a.n_src && di < a.n_dst; // a negative index is a large unsigned one
    nixl_amd_copy_list_entry_t s{}, d{};
    if (named) {
        s = a.src[si];
        d = a.dst[di];
    }
    const bool good = named && s.len == d.len;
    const uint32_t units = s.len / 16u, head = kPieceUnits - (static_cast<uint32_t>(d.addr >> 4) & 7u);
    uint32_t count = min(units, head), more = good ? units - count : 0;
    const uint32_t mine = (more + kPieceUnits - 1) / kPieceUnits; // records beyond the first
    if (good) store_ahead(a.recs + i, PieceRec{s.addr, d.addr | (static_cast<uint64_t>(count - 1) << kPieceUnitsShift)});

    // sums over a workgroup fit 32 bits: at most kListMaxBytes a pair
    const uint32_t n_bad = __popcll(__ballot(here && !good));
    const uint32_t n_continued = __popcll(__ballot(good && follows && s.continues && d.continues));
    const uint32_t bytes = wave_sum_dpp(good ? s.len : 0), incl = wave_scan_dpp(mine);
    if (lane == kWaveSize - 1) {
        wave_bytes[wave] = bytes;
        wave_bad[wave] = n_bad;
        wave_continued[wave] = n_continued;
        wave_extra[wave] = incl;
    }
    __syncthreads();
    uint32_t sum = 0, b = 0; // of the workgroup, in the first wave
    if (wave == 0) {
        sum = wave_sum_dpp(lane < kWaves ? wave_bytes[lane] : 0);
        b = wave_sum_dpp(lane < kWaves ? wave_bad[lane] : 0);
        const uint32_t c = wave_sum_dpp(lane < kWaves ? wave_continued[lane] : 0);
        const uint32_t x = lane < kWaves ? wave_extra[lane] : 0, run = wave_scan_dpp(x);
        if (lane < kWaves) wave_extra[lane] = run - x; // records of the waves before
        if (lane == kWaves - 1) {
            const unsigned long long packed = run | static_cast<unsigned long long>(c) << 32;
            if (b) atomicAdd(&a.totals->bad, b);
            if (packed) extra_at = static_cast<uint32_t>(atomicAdd(&a.totals->extra_continued, packed));
        }
    }
    __syncthreads();
    if (threadIdx.x == kWaves - 1) {
        // The verdict waits for nothing but additions, which are done where all dies see them: no cache is written
        // back for it (the records are for the kernel behind this one).
        const auto settle = [] { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
        settle(); // this workgroup's additions
        const unsigned long long before = __hip_atomic_fetch_add(&a.totals->bytes_arrived, sum | 1ull << kListBytesBits,
                                                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (before >> kListBytesBits == a.n_workgroups - 1) {
            const unsigned long long both = __hip_atomic_exchange(&a.totals->extra_continued, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const uint32_t bad = __hip_atomic_exchange(&a.totals->bad, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&a.totals->bytes_arrived, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const auto tell = [](auto *where, auto what) { __hip_atomic_store(where, what, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); };
            tell(&a.verdict->bytes, (before & ((1ull << kListBytesBits) - 1)) + sum);
            tell(&a.verdict->bad, bad);
            tell(&a.verdict->continued, static_cast<uint32_t>(both >> 32));
            tell(&a.verdict->extra, static_cast<uint32_t>(both));
            settle(); // the totals are zero, the words in front of the last one there
            tell(&a.verdict->there, 1u);
        }
    }
    if (!more) return;
    uint32_t at = a.n + extra_at + wave_extra[wave] + (incl - mine);
    for (uint32_t first = count; more; first += count, more -= count) {
        count = min(more, kPieceUnits);
        store_ahead(a.recs + at++,
                    PieceRec{s.addr + first * 16ull, (d.addr + first * 16ull) | (static_cast<uint64_t>(count - 1) << kPieceUnitsShift)});
    }
}

__global__ void __launch_bounds__(kWaveSize)
clear_totals_kernel(ListTotals *totals) {
    if (threadIdx.x == 0) *totals = ListTotals{};
}

// A long descriptor as chunks of its own: chunk k starts k chunks behind the place `back` bytes in
// front of the descriptor.  With a whole number of chunks and back = 0 that is all there is to it;
// else the last chunk (and, with a `back` that puts the others on the destination's lines, the
// first) is an end, of as many 16-byte units as its bytes need: less than a unit of it lies over its
// neighbour, where both write the same bytes.  (Where an address leaves no room for the number of
// units, an end is a whole chunk and the rest of it lies there.)  So every chunk belongs to one
// descriptor, whatever the length, and no descriptor moves another one's chunks off the lines.
// Cut from one stream of all descriptors, with a whole chunk over its neighbour at each end, and so,
// us: 512 tensors of 2 MiB + 16 B 372, 330 and 328; 60 000 descriptors of 8 to 64 KiB in multiples
// of 16 bytes, shuffled, 1000, 844 and 838; 65 536 of 8 KiB + 128 B 195, 206 and 185; at 16 units a
// lane 32 768 of 16 KiB + 16 B 253, 412 and 217.
struct ChunkRun {
    uint64_t src, dst, len; // len >= a chunk
    uint32_t first; // chunk of the plan that the run starts with
    uint32_t back; // less than a chunk
};

// Records of a plan of such runs: a thread per chunk finds its run by bisection (the
// table stays in the L2), so that one long run among short ones costs no more than any other;
// 32 bytes per run cross the bus instead of 16 per chunk.
__global__ void __launch_bounds__(256)
expand_runs_kernel(UniformRec *recs, const ChunkRun *runs, uint32_t n_runs, uint32_t n_chunks, uint32_t chunk_bytes, int ends) {
    for (uint64_t c64 = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; c64 < n_chunks;
         c64 += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
        const uint32_t c = static_cast<uint32_t>(c64);
        uint32_t lo = 0, hi = n_runs; // runs[lo].first <= c < runs[hi].first
        while (hi - lo > 1) {
            const uint32_t mid = lo + (hi - lo) / 2;
            if (runs[mid].first <= c) lo = mid;
            else hi = mid;
        }
        const ChunkRun run = runs[lo];
        const uint64_t at = static_cast<uint64_t>(c - run.first) * chunk_bytes;
        const uint64_t left = run.len + run.back - at; // of the run, from this chunk on
        if (ends && left < chunk_bytes) {
            const uint32_t units = static_cast<uint32_t>(left + 15u) / 16u;
            const uint64_t off = run.len - units * 16u;
            store_ahead(recs + c, end_rec(run.src + off, run.dst + off, units));
        } else if (ends && at < run.back) {
            store_ahead(recs + c, end_rec(run.src, run.dst, (chunk_bytes - run.back + 15u) / 16u));
        } else {
            const uint64_t off = min(at > run.back ? at - run.back : 0, run.len - chunk_bytes);
            store_ahead(recs + c, UniformRec{run.src + off, run.dst + off});
        }
    }
}

// Largest grid of one launch: HIP refuses grids of 2^32 or more threads, i.e. 2^22 workgroups of
// 16 waves; a plan with more work than that goes out as several launches.
constexpr uint32_t kMaxGrid = 1u << 21;

struct UniformLaunch {
    const UniformRec *recs;
    uint32_t first_chunk, n_chunks, n_wgs, chunks_per_rec;
    int swizzle;
    dim3 grid;
    hipStream_t stream;
};

template<int UPL, int POL>
void
launch_uniform(int waves, const UniformLaunch &u) {
#define NIXL_AMD_UNIFORM(WV)                                                                              \
    hipLaunchKernelGGL((copy_uniform_kernel<UPL, POL, WV>), u.grid, dim3(kWaveSize * WV), 0, u.stream, u.recs, \
                       u.first_chunk, u.n_chunks, u.n_wgs, u.swizzle, FastDiv(u.chunks_per_rec))
    switch (waves) {
    case 1: NIXL_AMD_UNIFORM(1); break;
    case 2: NIXL_AMD_UNIFORM(2); break;
    case 4: NIXL_AMD_UNIFORM(4); break;
    case 8: NIXL_AMD_UNIFORM(8); break;
    default: NIXL_AMD_UNIFORM(16); break;
    }
#undef NIXL_AMD_UNIFORM
}

template<int POL>
void
launch_uniform_upl(int upl, int waves, const UniformLaunch &u) {
    switch (upl) {
    case 1: launch_uniform<1, POL>(waves, u); break;
    case 2: launch_uniform<2, POL>(waves, u); break;
    case 4: launch_uniform<4, POL>(waves, u); break;
    case 8: launch_uniform<8, POL>(waves, u); break;
    default: launch_uniform<16, POL>(waves, u); break;
    }
}

template<int POL>
void
launch_mixed_upl(int upl, dim3 grid, hipStream_t s, const MixedArgs &a) {
    const dim3 block(kMixedThreads);
    switch (upl) {
    case 1: hipLaunchKernelGGL((copy_mixed_kernel<1, POL>), grid, block, 0, s, a); break;
    case 2: hipLaunchKernelGGL((copy_mixed_kernel<2, POL>), grid, block, 0, s, a); break;
    case 4: hipLaunchKernelGGL((copy_mixed_kernel<4, POL>), grid, block, 0, s, a); break;
    case 8: hipLaunchKernelGGL((copy_mixed_kernel<8, POL>), grid, block, 0, s, a); break;
    default: hipLaunchKernelGGL((copy_mixed_kernel<16, POL>), grid, block, 0, s, a); break;
    }
}

template<int POL>
void
launch_pieces(uint32_t w, uint32_t n_wgs, hipStream_t s, const PieceRec *recs, uint32_t n) {
    const dim3 block(kWaveSize * w);
    const uint32_t per_die = (n_wgs + kNumXcd - 1) / kNumXcd;
    const dim3 grid(per_die * kNumXcd); // surplus workgroups exit at once
    if (w == 1)
        hipLaunchKernelGGL((copy_piece_kernel<POL, kPieceLoads, 1>), grid, block, 0, s, recs, n, per_die);
    else if (w == 2)
        hipLaunchKernelGGL((copy_piece_kernel<POL, kPieceLoads, 2>), grid, block, 0, s, recs, n, per_die);
    else
        hipLaunchKernelGGL((copy_piece_kernel<POL, kPieceLoads, 4>), grid, block, 0, s, recs, n, per_die);
}

// Calls f.template operator()<POL>() for the plan's policy.
template<typename F>
void
with_policy(int policy, F &&f) {
    switch (policy) {
    case kPolNtNt: f.template operator()<kPolNtNt>(); break;
    case kPolPlain: f.template operator()<kPolPlain>(); break;
    case kPolPlainSc1Nt: f.template operator()<kPolPlainSc1Nt>(); break;
    default: f.template operator()<kPolNtSc1Nt>(); break;
    }
}

} // namespace

namespace {

// Plan arenas and the pinned buffers they are uploaded from are recycled: a request whose
// descriptor list changes every time (paged KV) would otherwise pay a hipMalloc and a
// pageable-memory copy per request.  Blocks come in power-of-two sizes; the cache keeps the
// most recently returned ones up to a count and a byte limit and frees the oldest beyond that.
class BlockCache {
public:
    explicit BlockCache(bool pinned) : pinned_(pinned) {}

    // A block of at least `bytes` on `device` (ignored for pinned memory); `cap` receives its size.  Both are left as
    // they are if there is none.
    hipError_t
    get(int device, size_t bytes, void **out, size_t *cap) {
        size_t size = 4096;
        while (size < bytes)
            size <<= 1;
        {
            std::lock_guard<std::mutex> lock(mutex_);
            for (size_t i = 0; i < free_.size(); ++i)
                if (free_[i].size == size && (pinned_ || free_[i].device == device)) {
                    *out = free_[i].ptr;
                    *cap = size;
                    held_ -= size;
                    free_.erase(free_.begin() + static_cast<long>(i));
                    return hipSuccess;
                }
        }
        void *ptr = nullptr;
        const hipError_t e = pinned_ ? hipHostMalloc(&ptr, size, hipHostMallocDefault) : hipMalloc(&ptr, size);
        if (e != hipSuccess) return e;
        *out = ptr;
        *cap = size;
        return hipSuccess;
    }

    // The block just given back is the likeliest to be asked for again (the next request of the
    // same shape), so when the cache is full the oldest blocks make room for it.
    void
    put(int device, void *ptr, size_t size) {
        std::vector<Block> evicted;
        {
            std::lock_guard<std::mutex> lock(mutex_);
            if (size <= kMaxHeld) {
                while (!free_.empty() && (held_ + size > kMaxHeld || free_.size() >= kMaxBlocks)) {
                    evicted.push_back(free_.front());
                    held_ -= free_.front().size;
                    free_.erase(free_.begin());
                }
                free_.push_back(Block{ptr, size, device});
                held_ += size;
            } else {
                evicted.push_back(Block{ptr, size, device});
            }
        }
        for (const Block &b : evicted) {
            if (pinned_)
                (void)hipHostFree(b.ptr);
            else
                (void)hipFree(b.ptr);
        }
    }

private:
    struct Block {
        void *ptr;
        size_t size;
        int device;
    };
    static constexpr size_t kMaxHeld = 256u << 20;
    static constexpr size_t kMaxBlocks = 32;
    const bool pinned_;
    std::mutex mutex_;
    std::vector<Block> free_;
    size_t held_ = 0;
};

BlockCache &
arena_cache() {
    static BlockCache *c = new BlockCache(false); // never destroyed: device memory outlives static teardown order
    return *c;
}

// Plans are uploaded on a stream of their own that does not synchronise with the default
// stream, so that preparing one request does not wait for another that is still copying.
constexpr int kMaxDevices = 64;

hipError_t
library_stream(hipStream_t (&streams)[kMaxDevices], int device, hipStream_t *out) {
    static std::mutex mutex;
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(mutex);
    if (!streams[device]) {
        const hipError_t e = hipStreamCreateWithFlags(&streams[device], hipStreamNonBlocking);
        if (e != hipSuccess) return e;
    }
    *out = streams[device];
    return hipSuccess;
}

hipError_t
upload_stream(int device, hipStream_t *out) {
    static hipStream_t streams[kMaxDevices] = {};
    return library_stream(streams, device, out);
}

// A stream on which nothing but events lie, each behind the caller's stream of a plan that was
// destroyed before its launch (recycle_after).
hipError_t
recycle_stream(int device, hipStream_t *out) {
    static hipStream_t streams[kMaxDevices] = {};
    return library_stream(streams, device, out);
}

BlockCache &
upload_cache() {
    static BlockCache *c = new BlockCache(true);
    return *c;
}

// Memory of the lists that stay on the device.  A cache of its own: a list is far larger than a
// request's records, and one that is released would push those out of theirs.
BlockCache &
list_cache() {
    static BlockCache *c = new BlockCache(false);
    return *c;
}

// The slots of g_list_slots that no request uses.
class ListSlots {
public:
    // A free one, or null.  The device is current.
    ListTotals *
    take() {
        std::lock_guard<std::mutex> lock(mutex_);
        if (!known_) {
            void *first = nullptr;
            if (hipGetSymbolAddress(&first, HIP_SYMBOL(g_list_slots)) != hipSuccess) {
                (void)hipGetLastError();
                return nullptr;
            }
            for (int i = kListSlots - 1; i >= 0; --i)
                free_.push_back(&(static_cast<ListSlot *>(first) + i)->totals);
            known_ = true;
        }
        if (free_.empty()) return nullptr;
        ListTotals *totals = free_.back();
        free_.pop_back();
        return totals;
    }

    // Only when its request's verdict is there, or it has been cleared again.
    void
    put(ListTotals *totals) {
        std::lock_guard<std::mutex> lock(mutex_);
        free_.push_back(totals);
    }

private:
    std::mutex mutex_;
    bool known_ = false;
    std::vector<ListTotals *> free_;
};

ListSlots &
list_slots(int device) {
    static auto *all = new ListSlots[kMaxDevices]; // never destroyed: requests may be released while the process ends
    return all[device];
}

// Words by which launches are watched: kDoneSlots a device, each with its counts on the device (zero
// between uses) and a value of its own for every launch, so that no word an earlier launch wrote is
// taken for this one's.  The words of all devices are one pinned block, allocated once by
// nixl_amd_copy_watch_prepare (a launch allocates nothing) and kept until the process ends.
class DoneSlots {
public:
    static constexpr int kStride = 16; // words: a cache line each

    explicit DoneSlots(uint32_t *words) : words_(words) {
        for (int i = kDoneSlots - 1; i >= 0; --i)
            free_.push_back(i);
    }

    // A free slot with the next value of its word, or -1.  The device is current.
    int
    take(Done *done) {
        std::lock_guard<std::mutex> lock(mutex_);
        if (free_.empty()) return -1;
        if (!counts_) {
            void *counts = nullptr;
            if (hipGetSymbolAddress(&counts, HIP_SYMBOL(g_done_counts)) != hipSuccess) {
                (void)hipGetLastError();
                return -1;
            }
            counts_ = static_cast<uint32_t *>(counts);
        }
        const int slot = free_.back();
        free_.pop_back();
        *done = Done{counts_ + static_cast<size_t>(slot) * ((kDoneGroups + 1) * kDoneLine), words_ + slot * kStride, ++value_[slot]};
        return slot;
    }

    // Only when no launch uses it any more.
    void
    put(int slot) {
        std::lock_guard<std::mutex> lock(mutex_);
        free_.push_back(slot);
    }

    bool
    arrived(int slot, uint32_t value) const {
        return __atomic_load_n(words_ + slot * kStride, __ATOMIC_ACQUIRE) == value;
    }

    // Nothing but launches of plans is queued on `stream`, or (not `own`) that holds no longer.
    void
    own_stream(hipStream_t stream, bool own) {
        std::lock_guard<std::mutex> lock(mutex_);
        Last *const at = find(stream);
        if (own && !at)
            last_.push_back(Last{stream, -1, 0});
        else if (own)
            at->slot = -1; // another stream at the address of an earlier one
        else if (at)
            last_.erase(last_.begin() + (at - last_.data()));
    }

    // The last launch on `stream` that this library made, if it is watched; slot -1: it is not.
    void
    last_on(hipStream_t stream, int slot, uint32_t value) {
        std::lock_guard<std::mutex> lock(mutex_);
        if (Last *const at = find(stream)) *at = Last{stream, slot, value};
    }

    // Whether a stream that has no other work than plans has run the last of them: 1, 0, or -1 if that is not
    // known here.
    int
    last_ended(hipStream_t stream) {
        std::lock_guard<std::mutex> lock(mutex_);
        const Last *const l = find(stream);
        if (!l || l->slot < 0) return -1;
        return l->value != value_[l->slot] || arrived(l->slot, l->value); // a used slot was free again
    }

private:
    struct Last {
        hipStream_t stream;
        int slot;
        uint32_t value;
    };

    Last *
    find(hipStream_t stream) {
        for (Last &l : last_)
            if (l.stream == stream) return &l;
        return nullptr;
    }

    std::vector<Last> last_; // of the streams that were named to own_stream
    uint32_t *const words_;
    uint32_t *counts_ = nullptr;
    std::mutex mutex_;
    std::vector<int> free_;
    uint32_t value_[kDoneSlots] = {};
};

std::atomic<DoneSlots **> g_done_slots{nullptr}; // [kMaxDevices] once prepared, never destroyed

DoneSlots *
done_slots(int device) {
    DoneSlots **all = g_done_slots.load(std::memory_order_acquire);
    return all && device >= 0 && device < kMaxDevices ? all[device] : nullptr;
}

// Queues the copy of `bytes` of a pinned block to a device block on `up`; both blocks are powers
// of two from 4 KiB, so whole 16-byte units of the last one lie inside them.
hipError_t
upload(hipStream_t up, void *dst, const void *staging, size_t bytes) {
    constexpr size_t kByKernel = 1u << 20;
    if (bytes > kByKernel) return hipMemcpyAsync(dst, staging, bytes, hipMemcpyHostToDevice, up);
    const size_t units = (bytes + 15) / 16;
    const dim3 grid(static_cast<unsigned>(std::min<size_t>((units + 255) / 256, 1024)));
    hipLaunchKernelGGL(upload_kernel, grid, dim3(256), 0, up, static_cast<uint4 *>(dst), static_cast<const uint4 *>(staging), units);
    return hipGetLastError();
}

} // namespace

struct nixl_amd_copy_plan {
    int device = 0;
    int upl = 1;
    int policy = kPolNtSc1Nt;
    int piece_policy = kPolNtSc1Nt;
    int waves = 1;
    int swizzle = 0;
    uint32_t max_wgs = 0;
    // device arrays
    void *arena = nullptr;
    size_t arena_bytes = 0; // bytes in use
    size_t arena_cap = 0; // size of the block
    const UniformRec *uniform_recs = nullptr;
    uint32_t n_uniform = 0; // uniform chunks
    uint32_t chunks_per_rec = 1;
    uint32_t uniform_wgs = 0;
    std::unique_ptr<InlineRecs> inline_recs; // instead of uniform_recs: a plan of a few blocks, nothing on the device
    std::unique_ptr<InlineIndices> inline_indices; // or of some more
    std::unique_ptr<GridIndices> inline_grid; // or whose indices repeat themselves
    // Records all the same, for its launches on the stream it was made for, from one of these on (later_records).
    hipStream_t home = nullptr;
    uint32_t launches_at_home = 0;
    bool sort_later = false;
    int later_policy = kPolNtSc1Nt;
    void *later = nullptr;
    size_t later_cap = 0;
    std::atomic<size_t> later_bytes{0}; // in use: the plan may be queried from any thread
    MixedArgs mixed_args{};
    uint32_t mixed_wgs = 0;
    const PieceRec *piece_recs = nullptr;
    uint32_t n_pieces = 0;
    const GenericItem *generic_items = nullptr;
    uint32_t n_generic = 0;
    uint32_t generic_wgs = 0;
    nixl_amd_copy_plan_info_t info{};
    hipEvent_t ev0 = nullptr, ev1 = nullptr; // timing events, created on first use
    // A plan is returned before its arrays are on the device: they are written by kernels queued
    // on a stream.  On the library's upload stream `uploaded` is recorded behind them, and the
    // first launches wait for it on their own stream.  On the stream the caller named (where the
    // launch is going to follow) nothing has to be waited for; the pinned buffer that the kernels
    // read then stays with the plan until a launch behind them is known to have run (see end_build).
    hipEvent_t uploaded = nullptr;
    hipStream_t built_on = nullptr; // the caller's stream, until a launch is known to be behind the build
    std::atomic<bool> seen_done{false}; // nixl_amd_copy_plan_status has seen a launch complete
    bool reserved = false; // one of kMaxHeldStaging is this plan's, its buffer not handed over yet
    std::atomic<void *> staging{nullptr}; // taken out by whoever gives it back: the status may be asked from any thread
    size_t staging_cap = 0;
    // Recorded behind the kernels of a launch (not on a capturing stream, not if it is watched by a
    // word): destroying the plan while it has not completed is refused, because the arena would go back to the pool
    // and the next plan's upload would overwrite records a running kernel still reads.
    hipEvent_t launched = nullptr;
    std::atomic<bool> launched_valid{false}; // and not seen complete
    // Instead of the event, for launches whose caller allows it: the slot of the launch's word.
    std::atomic<int> slot{-1};
    uint32_t slot_value = 0;
    hipStream_t watched_on = nullptr;
    std::atomic<uint32_t> polls{0};
    std::atomic<hipError_t> watch_failure{hipSuccess}; // of the watched launch: its word does not come any more
    bool ever_launched = false; // not counting launches into a capture

    ~nixl_amd_copy_plan();
};

// Pinned buffers whose contents are still travelling to the device: each goes back to the
// upload cache once the event recorded behind its copy has completed, which the next plan
// creation on the device looks for.
struct PendingUpload {
    hipEvent_t done;
    void *staging;
    size_t cap;
    void *arena; // of a plan destroyed before it was launched, or null
    size_t arena_cap;
};
static std::mutex g_pending_mutex;
static std::map<int, std::vector<PendingUpload>> g_pending; // by device

static void
reap_uploads(int device) {
    std::lock_guard<std::mutex> lock(g_pending_mutex);
    auto &list = g_pending[device];
    for (size_t i = 0; i < list.size();) {
        const hipError_t e = hipEventQuery(list[i].done);
        if (e == hipErrorNotReady) {
            (void)hipGetLastError();
            ++i;
            continue;
        }
        (void)hipEventDestroy(list[i].done);
        if (list[i].staging) upload_cache().put(device, list[i].staging, list[i].cap);
        if (list[i].arena) arena_cache().put(device, list[i].arena, list[i].arena_cap);
        list[i] = list.back();
        list.pop_back();
    }
}

// Records `done` behind everything queued on `up` so far: on `up` itself if that is a stream of the
// library's, on one of its own if it is a caller's.  An event that lies on a caller's stream may
// not even be asked for while that stream is captured, which would break a capture that has
// nothing to do with it.
static hipError_t
record_behind(int device, hipStream_t up, bool of_caller, hipEvent_t done) {
    if (!of_caller) return hipEventRecord(done, up);
    hipStream_t aside = nullptr;
    hipEvent_t joint = nullptr;
    hipError_t e = recycle_stream(device, &aside);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&joint, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventRecord(joint, up);
    if (e == hipSuccess) e = hipStreamWaitEvent(aside, joint, 0);
    if (e == hipSuccess) e = hipEventRecord(done, aside);
    if (joint) (void)hipEventDestroy(joint);
    return e;
}

// Hands `staging` and `arena` (either may be null) over: recycled when everything queued on `up` so far has run.
// Without an event to watch, the stream is waited for instead.
static void
recycle_after(int device, hipStream_t up, bool of_caller, void *staging, size_t cap, void *arena = nullptr, size_t arena_cap = 0) {
    hipEvent_t done = nullptr;
    if (hipEventCreateWithFlags(&done, hipEventDisableTiming) == hipSuccess && record_behind(device, up, of_caller, done) == hipSuccess) {
        std::lock_guard<std::mutex> lock(g_pending_mutex);
        g_pending[device].push_back(PendingUpload{done, staging, cap, arena, arena_cap});
        return;
    }
    (void)hipGetLastError();
    if (done) (void)hipEventDestroy(done);
    (void)hipStreamSynchronize(up);
    if (staging) upload_cache().put(device, staging, cap);
    if (arena) arena_cache().put(device, arena, arena_cap);
}

// Pinned buffers that wait with their plans for a first launch: a program may make any number of
// requests and keep them, so only a few may.
constexpr int kMaxHeldStaging = 16;
static std::atomic<int> g_held_staging{0};

nixl_amd_copy_plan::~nixl_amd_copy_plan() {
    if (reserved) g_held_staging.fetch_sub(1, std::memory_order_relaxed);
}

// The kernels that read the plan's pinned buffer have run: back into the cache with it.
static void
give_back_staging(nixl_amd_copy_plan *plan) {
    if (void *staging = plan->staging.exchange(nullptr)) {
        upload_cache().put(plan->device, staging, plan->staging_cap);
        g_held_staging.fetch_sub(1, std::memory_order_relaxed);
    }
}

// The word of a launch is long in coming: whether the stream still has it to run.  hipErrorNotReady
// while it may; an error of the stream's, or of a launch that ended without its word.
static hipError_t
ask_stream(const nixl_amd_copy_plan *plan, int slot) {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    hipError_t e = hipStreamIsCapturing(plan->watched_on, &capture);
    if (e == hipSuccess && capture != hipStreamCaptureStatusNone) return hipErrorNotReady;
    if (e == hipSuccess) e = hipStreamQuery(plan->watched_on);
    if (e != hipSuccess) (void)hipGetLastError();
    if (e == hipErrorNotReady) return e;
    // Another thread may have seen the end meanwhile and given the slot back, and another launch written its own
    // value there: only while the slot is the plan's has a word without the plan's value not been written.
    if (done_slots(plan->device)->arrived(slot, plan->slot_value)) return hipErrorNotReady; // seen by the next look
    if (plan->slot.load(std::memory_order_acquire) != slot) return hipErrorNotReady;
    return e == hipSuccess ? hipErrorUnknown : e;
}

// Whether every launch of the plan has run: hipSuccess, hipErrorNotReady (never with `wait`) or an error.
static hipError_t
ended(nixl_amd_copy_plan *plan, bool wait) {
    for (int slot; (slot = plan->slot.load(std::memory_order_acquire)) >= 0;) {
        DoneSlots &slots = *done_slots(plan->device);
        if (slots.arrived(slot, plan->slot_value)) {
            if (plan->slot.compare_exchange_strong(slot, -1)) slots.put(slot);
            break;
        }
        if (const hipError_t e = plan->watch_failure.load(std::memory_order_relaxed); e != hipSuccess) return e;
        constexpr uint32_t kAskEvery = 4096;
        if (plan->polls.fetch_add(1, std::memory_order_relaxed) % kAskEvery == kAskEvery - 1) {
            const hipError_t e = ask_stream(plan, slot);
            if (e != hipErrorNotReady) {
                plan->watch_failure.store(e, std::memory_order_relaxed);
                return e;
            }
            if (wait) std::this_thread::yield();
        }
        if (!wait) return hipErrorNotReady;
        __builtin_ia32_pause();
    }
    if (!plan->launched_valid) return hipSuccess;
    const hipError_t e = wait ? hipEventSynchronize(plan->launched) : hipEventQuery(plan->launched);
    if (e == hipSuccess)
        plan->launched_valid = false;
    else if (e == hipErrorNotReady)
        (void)hipGetLastError();
    return e;
}

// The plan's records are in place (or `wait` and they are not yet: block until they are).
// Returns hipErrorNotReady when they are still being written and `wait` is false.
static hipError_t
settle_upload(nixl_amd_copy_plan *plan, bool wait) {
    if (!plan->uploaded) return hipSuccess;
    hipError_t e = wait ? hipEventSynchronize(plan->uploaded) : hipEventQuery(plan->uploaded);
    if (e == hipErrorNotReady) {
        (void)hipGetLastError();
        return e;
    }
    (void)hipEventDestroy(plan->uploaded);
    plan->uploaded = nullptr;
    return e;
}

// The records kernels of a listed plan, queued on `up`, have written their verdict.  The word is
// watched for some hundred microseconds (it is there about 5 us before an event behind the kernels
// is seen complete); an end of the kernels without it is an error of theirs.
static hipError_t
await_verdict(const ListVerdict &verdict, hipStream_t up) {
    const auto there = [&] { return __atomic_load_n(&verdict.there, __ATOMIC_ACQUIRE) != 0; };
    for (int spins = 0; spins < 10000; ++spins) {
        if (there()) return hipSuccess;
        __builtin_ia32_pause();
    }
    const hipError_t e = hipStreamSynchronize(up);
    return e != hipSuccess || there() ? e : hipErrorUnknown;
}

// What one pass over an index vector tells.
struct IndexFacts {
    uint32_t highest = 0; // a negative index is a large one
    uint32_t ones = 0; // steps to the index behind the one before
    uint32_t regular = 0; // steps like the one before, or of one where that is dense
};

// v[i] for begin <= i < end, v[i - 1] and v[i - 2] being those before it: differences modulo 2^32 and no
// value carried from one iteration to the next, so that the loop vectorises.
static __attribute__((always_inline)) inline void
study_indices(const uint32_t *v, size_t begin, size_t end, uint32_t dense, IndexFacts &f) {
    uint32_t highest = f.highest, ones = 0, regular = 0;
    for (size_t i = begin; i < end; ++i) {
        const uint32_t step = v[i] - v[i - 1], before = v[i - 1] - v[i - 2];
        highest = std::max(highest, v[i]);
        ones += step == 1u;
        regular += (static_cast<uint32_t>(step == 1u) & dense) | static_cast<uint32_t>(step == before);
    }
    f.highest = highest;
    f.ones += ones;
    f.regular += regular;
}

#if defined(__x86_64__)
__attribute__((target("avx2"))) static void
study_indices_avx2(const uint32_t *v, size_t begin, size_t end, uint32_t dense, IndexFacts &f) {
    study_indices(v, begin, end, dense, f);
}
#endif

// How many of `n` indices follow the first one by one each, looked at in stretches of 1024.
static __attribute__((always_inline)) inline size_t
count_consecutive(const uint32_t *v, uint32_t first, size_t n) {
    size_t i = 0;
    while (i < n) {
        const size_t end = std::min<size_t>(n, i + 1024);
        uint32_t off = 0;
        for (size_t j = i; j < end; ++j)
            off |= v[j] ^ (first + static_cast<uint32_t>(j));
        if (off) break;
        i = end;
    }
    return i;
}

#if defined(__x86_64__)
__attribute__((target("avx2"))) static size_t
count_consecutive_avx2(const uint32_t *v, uint32_t first, size_t n) {
    return count_consecutive(v, first, n);
}
#endif

// Copies `n` indices and studies the copy, a stretch that the first-level cache holds at a time: what
// is found out holds for what the kernel will read, whatever becomes of the caller's array.  Consecutive
// indices, of which the kernel needs the first, are not copied but for that one unless `whole` says so.
static IndexFacts
take_indices(const int32_t *from, size_t n, int32_t *to, bool dense, bool whole) {
#if defined(__x86_64__)
    const bool wide = __builtin_cpu_supports("avx2");
#endif
    IndexFacts f;
    const auto *v = reinterpret_cast<const uint32_t *>(to), *given = reinterpret_cast<const uint32_t *>(from);
    const uint32_t first = given[0];
#if defined(__x86_64__)
    const size_t consecutive = wide ? count_consecutive_avx2(given, first, n) : count_consecutive(given, first, n);
#else
    const size_t consecutive = count_consecutive(given, first, n);
#endif
    if (!whole && consecutive == n && n - 1 <= UINT32_MAX - first) {
        to[0] = static_cast<int32_t>(first);
        f.highest = first + static_cast<uint32_t>(n - 1);
        f.ones = static_cast<uint32_t>(n - 1);
        f.regular = n < 2 ? 0 : static_cast<uint32_t>(n - 2) + (dense ? 1 : 0);
        return f;
    }
    constexpr size_t kStretch = 4096;
    for (size_t begin = 0; begin < n; begin += kStretch) {
        const size_t end = std::min(n, begin + kStretch);
        std::memcpy(to + begin, from + begin, (end - begin) * sizeof(int32_t));
        size_t i = begin;
        for (; i < std::min<size_t>(end, 2); ++i) { // no step, and one without a step before it
            const bool one = i == 1 && v[1] - v[0] == 1u;
            f.highest = std::max(f.highest, v[i]);
            f.ones += one;
            f.regular += one && dense;
        }
#if defined(__x86_64__)
        if (wide) {
            study_indices_avx2(v, i, end, dense, f);
            continue;
        }
#endif
        study_indices(v, i, end, dense, f);
    }
    return f;
}

// Whether `n` indices, in rows of `length`, are a grid (GridIndices): listed by column every row is the one before it `step`
// further on, listed by row every row ascends by `step`.
static __attribute__((always_inline)) inline bool
is_grid(const uint32_t *v, size_t n, uint32_t length, bool by_column, uint32_t step) {
    if (by_column) {
        for (size_t at = length; at < n;) {
            const size_t end = std::min<size_t>(n, at + 1024);
            uint32_t off = 0;
            for (; at < end; ++at)
                off |= (v[at] - v[at - length]) ^ step;
            if (off) return false;
        }
        return true;
    }
    // no other steps than those from a row to the next: counted there first, then in all, which vectorises
    size_t between = 0;
    for (size_t at = length; at < n; at += length)
        between += v[at] - v[at - 1] != step;
    for (size_t at = 1; at < n;) {
        const size_t end = std::min<size_t>(n, at + 1024);
        uint32_t others = 0;
        for (; at < end; ++at)
            others += v[at] - v[at - 1] != step;
        if (others > between) return false;
        between -= others;
    }
    return between == 0;
}

// A grid listed by row has rows of at least kMinGridRow, which are looked at one by one.  Rows that are neighbours in their list have
// records of their own beyond kMaxConsecutive blocks, and blocks larger than kMaxRowBlock beyond kMaxRowBytes.  These lines were drawn
// where records had been measured faster, and that did not hold: passes of gathers through an agent, with records and as a grid on
// either side of the lines, us: 14 336 neighbours of 8 KiB in rows of 16 53.3 and 49.2, 16 384 59.5 and 55.1, 32 768 of 2 KiB in rows of 32 41.2 and
// 34.4, 16 384 of 16 KiB 98.5 and 94.8, rows in ascending order 59.2 and 59.2; scatters 54.9 and 50.8, 60.0 and 55.1, 41.8 and 35.2, 98.3 and 94.4;
// blocks of 24 KiB, 600 MiB, 216.6 and 212.5, of 32 KiB, 640 MiB, 229.9 and 225.8, 1024 MiB 355.7 and 354.4, of 64 KiB, 800 MiB, 278.2 and 276.0, of 256 KiB, 960 MiB,
// 312.6 and 311.7.  Neither blocks nor bytes nor rows decide: nowhere are records faster by more than runs differ.
constexpr size_t kMinGridRow = 8, kMaxConsecutive = 12288;
constexpr uint64_t kMaxRowBlock = 16384, kMaxRowBytes = 512ull << 20;

struct GridShape {
    uint32_t length = 0; // of a row; 0: no grid
    bool by_column;
};

// The shape of `n` >= 4 indices: rows as long as they ascend evenly from the start, or the first length at which
// they start again as they started, as far on as the last row is from the one before it.  Few lengths are looked at
// in full.
static __attribute__((always_inline)) inline GridShape
find_grid(const uint32_t *v, size_t n, bool by_row) {
    const uint32_t step = v[1] - v[0];
    size_t length = 2;
    while (length < n && v[length] - v[length - 1] == step)
        ++length;
    if (step == 1 && n > kMaxConsecutive) by_row = false;
    if (by_row && length >= kMinGridRow && n % length == 0 && n / length <= kGridIds && is_grid(v, n, static_cast<uint32_t>(length), false, step))
        return {static_cast<uint32_t>(length), false};
    constexpr size_t kStretch = 64;
    int looks = 8;
    for (size_t from = 2; from <= std::min<size_t>(n / 2, kGridIds); from += kStretch) {
        const size_t end = std::min(from + kStretch, std::min<size_t>(n / 2, kGridIds) + 1);
        uint32_t any = 0;
        const auto may = [&](size_t i) { // i + 1 <= n / 2 + 1 < n
            return static_cast<uint32_t>(v[i + 1] - v[i] == step) & static_cast<uint32_t>(v[n - 1] - v[n - 1 - i] == v[i] - v[0]);
        };
        for (size_t i = from; i < end; ++i)
            any |= may(i);
        if (!any) continue;
        for (size_t i = from; i < end; ++i) {
            if (!may(i) || n % i != 0) continue;
            if (is_grid(v, n, static_cast<uint32_t>(i), true, v[i] - v[0])) return {static_cast<uint32_t>(i), true};
            if (--looks == 0) return {};
        }
    }
    return {};
}

// The ids of a side, `apart` from each other in `v`, counted from the smallest one (`lowest`, the largest one being `last`), or false if
// they don't fit 16 bits.
static __attribute__((always_inline)) inline bool
take_ids(const uint32_t *v, size_t n_ids, size_t apart, uint16_t *to, uint32_t &lowest, uint32_t &last) {
    uint32_t id[kGridIds]; // read once, whatever becomes of the caller's array
    for (size_t i = 0; i < n_ids; ++i)
        id[i] = v[i * apart];
    uint32_t low = UINT32_MAX, high = 0;
    for (size_t i = 0; i < n_ids; ++i) {
        low = std::min(low, id[i]);
        high = std::max(high, id[i]);
    }
    lowest = low;
    last = high;
    if (high - low > 0xffffu) return false;
    for (size_t i = 0; i < n_ids; ++i)
        to[i] = static_cast<uint16_t>(id[i] - low);
    return true;
}

#if defined(__x86_64__)
__attribute__((target("avx2"))) static bool
take_ids_avx2(const uint32_t *v, size_t n_ids, size_t apart, uint16_t *to, uint32_t &lowest, uint32_t &last) {
    return take_ids(v, n_ids, apart, to, lowest, last);
}

__attribute__((target("avx2"))) static GridShape
find_grid_avx2(const uint32_t *v, size_t n, bool by_row) {
    return find_grid(v, n, by_row);
}

__attribute__((target("avx2"))) static bool
is_grid_avx2(const uint32_t *v, size_t n, uint32_t length, bool by_column, uint32_t step) {
    return is_grid(v, n, length, by_column, step);
}
#endif

// The indices of a request as a grid, if both vectors are consecutive or grids of one shape, one of them listed.  What
// the kernel reads are the ids and steps taken here, and those are what is held against the lists' lengths:
// a request that this turns away is looked at as any other, and told what is wrong with it.
static std::unique_ptr<GridIndices>
take_grid(const nixl_amd_copy_run_t &src_run, const int32_t *src_index, uint64_t src_entries, const nixl_amd_copy_run_t &dst_run,
          const int32_t *dst_index, uint64_t dst_entries, size_t n, uint64_t len) {
#if defined(__x86_64__)
    const bool wide = __builtin_cpu_supports("avx2");
    const auto find = wide ? find_grid_avx2 : [](const uint32_t *v, size_t of, bool by_row) { return find_grid(v, of, by_row); };
    const auto is = wide ? is_grid_avx2 : [](const uint32_t *v, size_t of, uint32_t length, bool by_column, uint32_t step) {
        return is_grid(v, of, length, by_column, step);
    };
    const auto take = wide ? take_ids_avx2 : [](const uint32_t *v, size_t n_ids, size_t apart, uint16_t *to, uint32_t &lowest, uint32_t &last) {
        return take_ids(v, n_ids, apart, to, lowest, last);
    };
    const auto count = wide ? count_consecutive_avx2 : [](const uint32_t *v, uint32_t first, size_t of) { return count_consecutive(v, first, of); };
#else
    const auto find = find_grid;
    const auto is = is_grid;
    const auto take = take_ids;
    const auto count = count_consecutive;
#endif
    const uint32_t *v[2] = {reinterpret_cast<const uint32_t *>(src_index), reinterpret_cast<const uint32_t *>(dst_index)};
    const nixl_amd_copy_run_t *run[2] = {&src_run, &dst_run};
    const uint64_t entries[2] = {src_entries, dst_entries};
    // which are listed is guessed from their start: the shape of one that is decides more cheaply than all of one that is not
    const auto looks_listed = [&](int side) { return count(v[side], v[side][0], std::min<size_t>(n, 1024)) < std::min<size_t>(n, 1024); };
    const bool listed[2] = {looks_listed(0), looks_listed(1)};
    if (!listed[0] && !listed[1]) return nullptr;
    const GridShape shape = find(v[listed[0] ? 0 : 1], n, len <= kMaxRowBlock || n * len <= kMaxRowBytes);
    if (shape.length == 0) return nullptr;
    const size_t rows = n / shape.length, n_ids = shape.by_column ? shape.length : rows, others = shape.by_column ? rows : shape.length;
    if (rows > kMaxGridRows) return nullptr;
    std::unique_ptr<GridIndices> g(new GridIndices); // not cleared
    g->row_length = FastDiv(shape.length);
    g->by_column = shape.by_column ? ~0u : 0;
    size_t place = 0;
    for (int side = 0; side < 2; ++side) {
        GridIndices::Side &s = side ? g->dst : g->src;
        s = {run[side]->base, run[side]->stride, v[side][0], 0, 0, 0};
        uint64_t highest = static_cast<uint64_t>(s.first) + (n - 1);
        if (listed[side]) {
            s.step = shape.by_column ? v[side][shape.length] - v[side][0] : v[side][1] - v[side][0];
            if (place + n_ids > kGridIds || s.step > INT32_MAX) return nullptr;
            if (side == 1 && listed[0] && !is(v[1], n, shape.length, shape.by_column, s.step)) return nullptr;
            uint32_t lowest, last;
            if (!take(v[side], n_ids, shape.by_column ? 1 : shape.length, g->ids + place, lowest, last)) return nullptr;
            s.first = lowest;
            s.listed = ~0u;
            s.place = static_cast<uint32_t>(place);
            place += n_ids;
            highest = static_cast<uint64_t>(last) + static_cast<uint64_t>(others - 1) * s.step;
        } else if (count(v[side], s.first, n) < n) {
            return nullptr;
        }
        if (highest > INT32_MAX || highest >= entries[side]) return nullptr;
    }
    return g;
}

// Requests of at least so many pairs a run are sent as runs.  Making a request of 65 536 and of 262 144
// pairs, us: vectors 34 and 88, runs of 8 pairs 34 and 86, of 16 pairs 29 and 65, of 64 pairs 26 and 50.
constexpr size_t kMinIndexRun = 8;

#if defined(__x86_64__)
// One bit a pair of the 64 from `i` on: it does not continue the pair before it on both sides.
__attribute__((target("avx2"))) static uint64_t
index_breaks(const int32_t *src, const int32_t *dst, size_t i, size_t n) {
    uint64_t breaks = 0;
    if (i > 0 && i + 64 <= n) {
        const __m256i one = _mm256_set1_epi32(1);
        for (size_t j = 0; j < 64; j += 8) {
            const auto *s = reinterpret_cast<const __m256i_u *>(src + i + j), *s1 = reinterpret_cast<const __m256i_u *>(src + i + j - 1);
            const auto *d = reinterpret_cast<const __m256i_u *>(dst + i + j), *d1 = reinterpret_cast<const __m256i_u *>(dst + i + j - 1);
            const __m256i follows =
                _mm256_and_si256(_mm256_cmpeq_epi32(_mm256_sub_epi32(_mm256_loadu_si256(s), _mm256_loadu_si256(s1)), one),
                                 _mm256_cmpeq_epi32(_mm256_sub_epi32(_mm256_loadu_si256(d), _mm256_loadu_si256(d1)), one));
            breaks |= static_cast<uint64_t>(~static_cast<uint32_t>(_mm256_movemask_ps(_mm256_castsi256_ps(follows))) & 0xffu) << j;
        }
        return breaks;
    }
    for (size_t j = i; j < std::min(i + 64, n); ++j)
        breaks |= static_cast<uint64_t>(j == 0 || static_cast<uint32_t>(src[j]) - static_cast<uint32_t>(src[j - 1]) != 1u ||
                                        static_cast<uint32_t>(dst[j]) - static_cast<uint32_t>(dst[j - 1]) != 1u)
            << (j - i);
    return breaks;
}
#endif

// Cuts `n` pairs into runs whose indices advance by one on both sides, and notes for every
// kListThreads pairs the run that their first one lies in, and at the end the last run.  False
// when more than a run for every kMinIndexRun pairs comes of it, looked at in stretches (vectors
// that are no runs are found out at their start), or where the pairs cannot be looked at eight at
// a time.  `runs` has room for n / kMinIndexRun + 1.
static bool
index_runs(const int32_t *src, const int32_t *dst, size_t n, IndexRun *runs, uint32_t *run_of) {
#if defined(__x86_64__)
    if (!__builtin_cpu_supports("avx2")) return false;
    constexpr size_t kStretch = 4096;
    static_assert(kListThreads % 64 == 0);
    size_t n_runs = 0;
    for (size_t i = 0; i < n; i += 64) {
        const uint64_t breaks = index_breaks(src, dst, i, n);
        if (i % kListThreads == 0) run_of[i / kListThreads] = static_cast<uint32_t>(n_runs - 1 + (breaks & 1));
        const size_t allowed = std::min(n, (i / kStretch + 1) * kStretch) / kMinIndexRun + 1;
        if (n_runs + static_cast<size_t>(__builtin_popcountll(breaks)) > allowed) return false;
        for (uint64_t left = breaks; left; left &= left - 1) {
            const size_t at = i + static_cast<size_t>(__builtin_ctzll(left));
            runs[n_runs++] = IndexRun{static_cast<uint32_t>(at), static_cast<uint32_t>(src[at]), static_cast<uint32_t>(dst[at]), 0};
        }
    }
    run_of[(n + kListThreads - 1) / kListThreads] = static_cast<uint32_t>(n_runs - 1);
    return true;
#else
    return false;
#endif
}

struct Tuning {
    int upl = 1, nt = 0, waves = 1, swizzle = 0, sort_scatter = 0;
    uint32_t max_wgs = 0;
    hipStream_t stream = nullptr;
};

// Defaults from a sweep on MI355X: the smallest chunk (one 128-bit load and store per lane,
// one wave per workgroup) gave the highest HBM rate; the cache policy follows the
// destination pattern.
static int
parse_tuning(const nixl_amd_copy_tuning_t *tuning, Tuning &t, const char *who) {
    if (tuning) {
        if (tuning->units_per_lane) t.upl = tuning->units_per_lane;
        if (tuning->nontemporal) t.nt = tuning->nontemporal;
        if (tuning->max_workgroups > 0) t.max_wgs = static_cast<uint32_t>(tuning->max_workgroups);
        if (tuning->waves_per_workgroup) t.waves = tuning->waves_per_workgroup;
        if (tuning->xcd_swizzle) t.swizzle = tuning->xcd_swizzle == 1 ? 1 : 0;
        t.sort_scatter = tuning->sort_scatter;
        t.stream = static_cast<hipStream_t>(tuning->stream);
    }
    if (t.upl != 1 && t.upl != 2 && t.upl != 4 && t.upl != 8 && t.upl != 16)
        return nixl_amd_fail(NIXL_AMD_ERR_INVALID, std::string(who) + ": units_per_lane must be 1, 2, 4, 8 or 16");
    if (t.nt < 0 || t.nt > 4) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, std::string(who) + ": nontemporal must be 0 to 4");
    if (t.waves != 1 && t.waves != 2 && t.waves != 4 && t.waves != 8 && t.waves != 16)
        return nixl_amd_fail(NIXL_AMD_ERR_INVALID, std::string(who) + ": waves_per_workgroup must be 1, 2, 4, 8 or 16");
    return NIXL_AMD_OK;
}

// Whether equal blocks of `len` bytes can be a plan of one record per block: whole chunks,
// long enough that a record is small next to its payload.
static bool
block_len_fits(uint64_t len, const Tuning &t) {
    const uint64_t chunk_bytes = static_cast<uint64_t>(kWaveSize) * t.upl * 16u;
    return len >= 8192 && len % chunk_bytes == 0;
}

// Whether a plan that scatters `n` equal blocks out of consecutive memory has its records sorted, unless the caller
// says so or not (tuning field `sort_scatter`).  Sorted, the writes find DRAM pages open; but sorting takes 4 us more in
// front of the copy, and the loads of unsorted records are ordinary ones.  Requests made, moved and waited for, three
// with pools of their own in turn, sorted and not, us: blocks of 8 KiB, 38 MB 32.1 and 27.5, 118 MB 60.6 and 55.8, 354 MB 141 and
// 138, 590 MB 225 and 222; of 9 KiB 18 MB 25.7 and 21.2, 225 MB 98.9 and 94.3, 562 MB 225 and 217; of 16 KiB 34 MB 30.1 and
// 25.6, 168 MB 74.3 and 71.5, 420 MB 157 and 156, 629 MB 226.9 and 229.1, 1049 MB 370.4 and 373.0; of 64 KiB 67 MB 38.8 and 34.2,
// 537 MB 183 and 182, 839 MB 275 and 274.
constexpr uint64_t kSortScatterFrom = 512ull << 20;

// Scatters that are grids listed by column (GridIndices) are sorted if their blocks are as large as this. Sorted and as a grid, us, 734 MB of
// 2 KiB 347 and 281, 940 MB of 4 KiB 382 and 347, 786 MB of 8 KiB 294 and 286, 562 and 956 MB of 9 KiB 245 and 221, 376 and 355, 1180 MB of 12 KiB
// 443 and 438, 787 MB of 14 KiB 309 and 293; of 16 KiB 629 MB 241 and 244, 839 MB 314 and 324, 1074 MB 385 and 418; 1468 MB of 32 KiB 505 and 537.
constexpr uint64_t kSortGridBlock = 16384;

// Of those that are left as they are, the ones of more than this are sorted when they get records (later_records). Up to
// it, unsorted records are loaded ordinarily and find what is in the last-level cache: 128 MiB of 16 KiB
// launched again and again 50.8 sorted and 45.8 not, three with pools of their own in turn 50.7 and 52.0; of 64 KiB 48.9 and 43.9, 48.9 and 49.7.
constexpr uint64_t kSortLaterFrom = 256ull << 20;

static bool
sort_pays(int sort_scatter, size_t n, uint64_t len) {
    if (sort_scatter == 2 || n < kSortWindow) return false;
    return sort_scatter == 1 || n * len > kSortScatterFrom;
}

// Whether a plan of `n` equal blocks can carry its records as kernel arguments: few enough, and
// the launch shape the inline kernel has.
static bool
fits_inline(size_t n, uint64_t len, const Tuning &t, size_t most = kInlineRecs) {
    return n <= most && t.upl == 1 && t.waves == 1 && !t.swizzle && n * (len / (kWaveSize * 16u)) <= kMaxGrid;
}

// The members a plan of `n_recs` equal blocks has wherever its records are.
static void
describe_blocks(nixl_amd_copy_plan &plan, const Tuning &t, size_t n_recs, uint64_t len, size_t n_descs) {
    const uint64_t chunk_bytes = static_cast<uint64_t>(kWaveSize) * t.upl * 16u;
    plan.chunks_per_rec = static_cast<uint32_t>(len / chunk_bytes);
    plan.n_uniform = static_cast<uint32_t>(n_recs * plan.chunks_per_rec);
    plan.uniform_wgs = (plan.n_uniform + static_cast<uint32_t>(t.waves) - 1) / static_cast<uint32_t>(t.waves);
    plan.info.payload_bytes = n_recs * len;
    plan.info.vec_descs = n_descs;
    plan.info.plan_device_bytes = plan.arena_bytes;
    plan.info.vec_chunks = plan.n_uniform;
    plan.info.uniform_chunks = plan.n_uniform;
    plan.info.units_per_lane = static_cast<uint32_t>(t.upl);
    plan.info.uniform_workgroups = plan.uniform_wgs;
}

// The stream a plan's arrays are written on: the one its launches will follow on, if the caller
// named it and it is idle.  A launch right behind the making then needs no event, no wait of one
// stream for another and no recycling in between (20 us of host time between make and kernel
// became 5); behind a transfer that is still running, the library's own stream writes the arrays
// meanwhile.  It does so, too, for a stream under capture (which may not be asked whether it is
// idle, and whose graph these kernels do not belong in), and for requests that are made and kept:
// the pinned buffer of a plan built on the caller's stream waits with the plan for its first
// launch to be seen done, and only kMaxHeldStaging plans may do that.  (1000 requests of 4096
// blocks made, posted and kept, each with a pinned buffer until its end: 204 us a request, 40 with
// buffers that come back.)
static hipError_t
build_stream(nixl_amd_copy_plan *plan, const Tuning &t, hipStream_t *out) {
    if (t.stream) {
        hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
        const bool may_ask = hipStreamIsCapturing(t.stream, &capture) == hipSuccess && capture == hipStreamCaptureStatusNone;
        // The runtime cannot tell of a launch without an event behind it that it has run: asked for the
        // stream it puts a marker there and finds it busy (a request of 15 250 blocks: 68 us became 103).
        // A launch that is watched says it itself, on a stream that carries nothing else: elsewhere the caller's
        // own work may lie behind it, and a request that waits for its verdict would wait for that.
        DoneSlots *const slots = done_slots(plan->device);
        const int ended = may_ask && slots ? slots->last_ended(t.stream) : -1;
        if (may_ask && (ended >= 0 ? ended == 1 : hipStreamQuery(t.stream) == hipSuccess)) {
            if (g_held_staging.fetch_add(1, std::memory_order_relaxed) < kMaxHeldStaging) {
                plan->reserved = true;
                *out = t.stream;
                return hipSuccess;
            }
            g_held_staging.fetch_sub(1, std::memory_order_relaxed);
        }
        (void)hipGetLastError();
    }
    return upload_stream(plan->device, out);
}

// Everything that writes the plan's arrays is queued on `up`: what later launches and the pinned
// buffer's next user wait for.  The buffer is taken over if this succeeds.
static hipError_t
end_build(nixl_amd_copy_plan *plan, hipStream_t up, void *staging, size_t staging_cap) {
    if (plan->reserved) {
        plan->built_on = up;
        plan->staging_cap = staging_cap;
        plan->staging = staging;
        plan->reserved = false; // from here on the buffer stands for it
        return hipSuccess;
    }
    // No wait here: the event goes behind the kernels, launches wait for it on their stream.
    hipError_t e = hipEventCreateWithFlags(&plan->uploaded, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventRecord(plan->uploaded, up);
    if (e == hipSuccess) recycle_after(plan->device, up, false, staging, staging_cap);
    return e;
}

static GenericItem
generic_item(uint64_t src, uint64_t dst, uint64_t len) {
    return GenericItem{src | (len - 1) >> 8 << kPieceUnitsShift, dst | ((len - 1) & 255u) << kPieceUnitsShift};
}

// Records while a plan is made.  Room for all records of a descriptor is made before the first of
// them is written, without a check for each and without touching memory that is not needed.
template<typename Rec>
struct Records {
    Rec *at = nullptr;
    size_t n = 0, cap = 0;

    Rec *
    room(size_t more, size_t expected) {
        if (cap - n < more) grow(more + expected);
        return at + n;
    }

    void
    end_at(const Rec *end) {
        n = static_cast<size_t>(end - at);
    }

    // Memory of somebody else's for the first records, left again when they are more.
    void
    lend(void *memory, size_t bytes) {
        at = static_cast<Rec *>(memory);
        cap = bytes / sizeof(Rec);
    }

private:
    std::unique_ptr<Rec[]> own_;

    __attribute__((noinline)) void
    grow(size_t more) {
        cap = std::max(2 * cap, n + more);
        std::unique_ptr<Rec[]> grown(new Rec[cap]);
        if (n) std::memcpy(grown.get(), at, n * sizeof(Rec));
        own_ = std::move(grown);
        at = own_.get();
    }
};

// A pinned upload buffer that goes back to its cache if nothing takes it over.
struct Staging {
    const int device;
    void *at = nullptr;
    size_t cap = 0;

    explicit Staging(int d) : device(d) {}
    ~Staging() {
        if (at) upload_cache().put(device, at, cap);
    }
    Staging(const Staging &) = delete;
    Staging &
    operator=(const Staging &) = delete;

    hipError_t
    get(size_t bytes) {
        return upload_cache().get(device, bytes, &at, &cap);
    }
};

// Byte descriptors of kSplitFromBytes and more (at least two chunks of the largest size besides a
// first line) are placed when the others are known.  They may become chunks, and beyond
// kLongItemsFrom of them the items take four rounds each, as making four times as many costs more
// than the copy gains (64 MiB in tensors of 1 MiB + 2 B: 24 us to make and 20.6 to copy with short
// items, 10.7 and 22.0 with long).
constexpr uint64_t kSplitFromBytes = 64 * 1024, kSplitFromTotal = 128ull << 20, kLongItemsFrom = 8ull << 20;

// Long descriptors, which become chunks of their own (ChunkRun).
struct LongDescs {
    explicit LongDescs(uint64_t chunk) : chunk_bytes(chunk) {}

    const uint64_t chunk_bytes;
    std::vector<ChunkRun> runs;
    uint64_t n = 0, edges = 0; // chunks, and how many of them are ends
    bool equal = true; // as many chunks in every run, none of them an end
    uint64_t address_bits = 0;

    // len >= chunk_bytes > back, and len + back > chunk_bytes if there is a back
    void
    add(uint64_t src, uint64_t dst, uint64_t len, uint64_t back) {
        const uint64_t reach = len + back;
        address_bits |= (src + len) | (dst + len);
        equal = equal && reach % chunk_bytes == 0 && back == 0 && (runs.empty() || runs[0].len == len);
        edges += static_cast<uint64_t>(back != 0) + static_cast<uint64_t>(reach % chunk_bytes != 0);
        runs.push_back(ChunkRun{src, dst, len, static_cast<uint32_t>(n), static_cast<uint32_t>(back)});
        n += (reach + chunk_bytes - 1) / chunk_bytes;
    }
};

// The descriptors of a request that are not 16-byte aligned.  Their loop is apart from that over
// the others: in one loop, with items appended one by one to a vector, making a plan took 106 us for
// 14 394 descriptors of up to 16 KiB and 24 for 3000 of up to 64 KiB (54 and 18 so), and code
// for items inlined there cost aligned descriptors 0.6 ns each (50 000 of 512 B: 203 us, 166 so).
// Items are written to the buffer that is uploaded, in front of everything else in it (a request of 2000 descriptors of
// 32 to 64 KiB made in 35 us with a copy of them, 27.8 so; of 3000 of up to 64 KiB 28.1 and 26.7).
struct ByteDescs {
    Records<GenericItem> items;
    std::vector<uint32_t> longs;
    uint64_t reach = kGenericRound; // of an item, from the destination line it starts in
    uint64_t n = 0, payload = 0, long_total = 0, splittable_total = 0;

    // Whether the whole chunks of a long one lie alike inside the lines of both sides.
    static bool
    splittable(const nixl_amd_copy_desc_t &d) {
        return ((d.src ^ d.dst) & 127u) == 0;
    }

    // Items of `len` bytes, written to `at`; every one but the first starts on a destination line.
    static GenericItem *
    cut(GenericItem *at, uint64_t src, uint64_t dst, uint64_t len, uint64_t reach) {
        for (uint64_t room = reach - (dst & 127u); len > room; room = reach) {
            *at++ = generic_item(src, dst, room);
            src += room;
            dst += room;
            len -= room;
        }
        *at++ = generic_item(src, dst, len);
        return at;
    }

    void
    add(uint64_t src, uint64_t dst, uint64_t len) {
        if (len == 0) return;
        items.end_at(cut(items.room(len / reach + 2, longs.size()), src, dst, len, reach));
    }

    // Items of one short descriptor at most.
    static constexpr size_t kMost = kSplitFromBytes / kGenericRound + 2;

    // Bytes to have ahead for the items of short descriptors among descs[i .. end), or 0 if they are too many.  The
    // lengths alone decide while they ask for little (3000 descriptors 1.4 us, 2.4 with a look at what is
    // aligned); beyond that only what has items counts.
    static size_t
    ahead(const nixl_amd_copy_desc_t *descs, size_t i, size_t end) {
        constexpr size_t kLittle = 512u << 10, kTooMany = 64u << 20;
        const auto bytes = [](size_t n_items) { return (n_items + kMost) * sizeof(GenericItem); };
        size_t items = 2 * (end - i);
        for (size_t j = i; j < end; ++j)
            items += descs[j].len < kSplitFromBytes ? descs[j].len / kGenericRound : 0;
        if (bytes(items) <= kLittle) return bytes(items);
        items = 0;
        for (size_t j = i; j < end; ++j)
            if (((descs[j].src | descs[j].dst | descs[j].len) & 15u) != 0 && descs[j].len < kSplitFromBytes)
                items += descs[j].len / kGenericRound + 2;
        return bytes(items) <= kTooMany ? bytes(items) : 0;
    }

    // Takes descriptors from `i` on until one that is aligned or that plan_create refuses; returns
    // where it stopped.
    __attribute__((noinline)) size_t
    take(const nixl_amd_copy_desc_t *descs, size_t i, size_t end) {
        GenericItem *at = nullptr, *limit = nullptr;
        uint64_t taken = 0, bytes = 0;
        for (; i < end; ++i) {
            const nixl_amd_copy_desc_t d = descs[i]; // a copy: the items written may not be taken to change it
            if (d.len == 0) continue;
            const uint64_t src_end = d.src + d.len, dst_end = d.dst + d.len;
            if (((d.src | d.dst | d.len) & 15u) == 0 || d.src == 0 || d.dst == 0 || src_end < d.src || dst_end < d.dst ||
                ((src_end | dst_end) >> kPieceUnitsShift) != 0)
                break;
            ++taken;
            bytes += d.len;
            if (d.len >= kSplitFromBytes) {
                longs.push_back(static_cast<uint32_t>(i));
                long_total += d.len;
                if (splittable(d)) splittable_total += d.len;
                continue;
            }
            if (static_cast<size_t>(limit - at) < kMost) {
                if (at) items.end_at(at);
                at = items.room(kMost, 2 * (end - i));
                limit = items.at + items.cap;
            }
            at = cut(at, d.src, d.dst, d.len, kGenericRound);
        }
        if (at) items.end_at(at);
        n += taken;
        payload += bytes;
        return i;
    }
};

constexpr int kNotBlocks = 1; // build_block_plan: the records are not what a block plan takes (no error recorded)

// A plan of `n_recs` equal blocks of `len` bytes whose {src, dst} records the host has written
// to the start of the pinned buffer `staging`.  One vectorisable pass over the records checks
// them (every address on a 128-byte line, none null, no range that wraps) and reads the
// pattern of the destinations (cache policy) and of the sources (record order); the copy to the
// device, the optional sort and the event behind them are queued on the upload stream and not
// waited for.  `staging` is taken over in every case.  Returns kNotBlocks when the records do
// not qualify, so that the caller can lower the request the general way.
static int
build_block_plan(int device, const Tuning &t, void *staging, size_t staging_cap, size_t n_recs, uint64_t len, size_t n_descs,
                 const nixl_amd_copy_record_facts_t *facts, nixl_amd_copy_plan_t **out) {
    const uint64_t chunk_bytes = static_cast<uint64_t>(kWaveSize) * t.upl * 16u;
    const auto *recs = static_cast<const UniformRec *>(staging);
    bool fits = n_recs > 0 && block_len_fits(len, t) && n_recs < (1ull << 31) && n_recs * (len / chunk_bytes) < (1ull << 32);
    uint64_t regular = 0, src_follows = 0, steps = n_recs ? n_recs - 1 : 0;
    if (fits && facts) {
        // the caller looked at every record while it wrote them
        fits = (facts->address_bits & 127u) == 0;
        regular = facts->regular_dst_steps;
        src_follows = facts->following_src_steps;
        steps = facts->steps;
    } else if (fits) {
        uint64_t misfit = 0;
        for (size_t i = 0; i < n_recs; ++i) {
            const uint64_t a = recs[i].src, b = recs[i].dst;
            misfit |= ((a | b) & 127u) | static_cast<uint64_t>(a == 0) | static_cast<uint64_t>(b == 0) |
                static_cast<uint64_t>(a + len < a) | static_cast<uint64_t>(b + len < b);
        }
        fits = misfit == 0;
        // Destination steps that are regular (one block on, or the same step as the one before)
        // and source steps that go one block on; nothing is carried from one iteration to the
        // next, so that the loop vectorises.
        if (n_recs > 1) {
            regular += (recs[1].dst - recs[0].dst) == len;
            src_follows += (recs[1].src - recs[0].src) == len;
        }
        for (size_t i = 2; i < n_recs; ++i) {
            const uint64_t step = recs[i].dst - recs[i - 1].dst, before = recs[i - 1].dst - recs[i - 2].dst;
            regular += static_cast<uint32_t>(step == len) | static_cast<uint32_t>(step == before);
            src_follows += static_cast<uint32_t>((recs[i].src - recs[i - 1].src) == len);
        }
    }
    if (!fits) {
        upload_cache().put(device, staging, staging_cap);
        return kNotBlocks;
    }
    const size_t bytes = n_recs * sizeof(UniformRec);
    auto *plan = new nixl_amd_copy_plan();
    plan->device = device;
    plan->upl = t.upl;
    plan->waves = t.waves;
    plan->swizzle = t.swizzle;
    plan->max_wgs = t.max_wgs;
    // cache policy by destination pattern, as in the general lowering
    const bool scattered = !(steps == 0 || 2 * regular >= steps);
    // a scatter out of consecutive memory is put into ascending destination order, window by window
    const bool sort = scattered && sort_pays(t.sort_scatter, n_recs, len) && 2 * src_follows >= steps;
    plan->policy = t.nt ? t.nt : copy_policy(n_recs * len, !scattered || sort, 2 * src_follows >= steps);
    if (fits_inline(n_recs, len, t)) {
        plan->inline_recs = std::make_unique<InlineRecs>();
        std::memcpy(plan->inline_recs->rec, recs, bytes);
        upload_cache().put(device, staging, staging_cap);
        describe_blocks(*plan, t, n_recs, len, n_descs);
        *out = plan;
        return NIXL_AMD_OK;
    }
    hipStream_t up = nullptr;
    hipError_t e = arena_cache().get(device, bytes, &plan->arena, &plan->arena_cap);
    if (e == hipSuccess) e = build_stream(plan, t, &up);
    if (e == hipSuccess) e = upload(up, plan->arena, staging, bytes);
    if (e == hipSuccess && sort) {
        hipLaunchKernelGGL(sort_records_kernel, dim3(static_cast<uint32_t>((n_recs + kSortWindow - 1) / kSortWindow)),
                           dim3(kSortWindow), 0, up, static_cast<UniformRec *>(plan->arena), static_cast<uint32_t>(n_recs));
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = end_build(plan, up, staging, staging_cap);
    if (e != hipSuccess) {
        if (up) (void)hipStreamSynchronize(up); // whatever was queued reads the buffers given back below
        if (plan->uploaded) (void)hipEventDestroy(plan->uploaded);
        upload_cache().put(device, staging, staging_cap);
        if (plan->arena) arena_cache().put(device, plan->arena, plan->arena_cap);
        delete plan;
        return nixl_amd_fail(NIXL_AMD_ERR_HIP, std::string("plan upload: ") + hipGetErrorString(e));
    }
    plan->arena_bytes = bytes;
    plan->uniform_recs = static_cast<const UniformRec *>(plan->arena);
    describe_blocks(*plan, t, n_recs, len, n_descs);
    *out = plan;
    return NIXL_AMD_OK;
}

// A pinned upload buffer that its caller fills with block records (nixl_amd_copy_records_begin).
struct nixl_amd_copy_records {
    void *staging = nullptr;
    size_t staging_cap = 0;
    size_t max_records = 0;
};

extern "C" {

int
nixl_amd_copy_plan_create(const nixl_amd_copy_desc_t *descs,
                          size_t n,
                          int device,
                          const nixl_amd_copy_tuning_t *tuning,
                          nixl_amd_copy_plan_t **out) {
    if (!out) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "plan_create: out is null");
    *out = nullptr;
    if (!descs && n) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "plan_create: descs is null");
    if (n >= (1ull << 32)) return nixl_amd_fail(NIXL_AMD_ERR_TOO_LARGE, "plan_create: more than 2^32-1 descriptors");

    Tuning t;
    if (const int rc = parse_tuning(tuning, t, "plan_create")) return rc;
    const int upl = t.upl, waves = t.waves, swizzle = t.swizzle;
    int nt = t.nt;
    const uint32_t max_wgs = t.max_wgs;

    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0)
        return nixl_amd_fail(NIXL_AMD_ERR_NO_DEVICE, "plan_create: no HIP device");
    if (device < 0 || device >= ndev) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "plan_create: bad device index");
    const DeviceScope on_device(device);
    HIP_TRY(on_device.status());

    const uint64_t chunk_units = static_cast<uint64_t>(kWaveSize) * upl, chunk_bytes = chunk_units * 16u;

    // ---- fast path: equal-length, line-aligned descriptors of whole chunks (KV blocks) ----
    // One pass over the descriptors writes the {src, dst} records straight into the pinned
    // upload buffer; nothing else is built.
    if (n > 0 && block_len_fits(descs[0].len, t)) {
        // Descriptors whose length is a multiple of the first one's (neighbouring blocks that
        // the caller merged) become that many records; room for twice as many records as
        // descriptors, beyond that the general lowering takes over.
        const uint64_t len0 = descs[0].len;
        const size_t cap = 2 * n;
        void *staging = nullptr;
        size_t staging_cap = 0;
        reap_uploads(device);
        const hipError_t e = upload_cache().get(device, cap * sizeof(UniformRec), &staging, &staging_cap);
        if (e != hipSuccess)
            return nixl_amd_fail(NIXL_AMD_ERR_HIP, std::string("hipHostMalloc(plan upload buffer): ") + hipGetErrorString(e));
        auto *recs = static_cast<UniformRec *>(staging);
        bool misfit = false;
        size_t n_recs = 0;
        for (size_t i = 0; i < n; ++i) {
            const nixl_amd_copy_desc_t &d = descs[i];
            if (d.len == len0) {
                recs[n_recs++] = UniformRec{d.src, d.dst};
                continue;
            }
            const uint64_t k = d.len / len0;
            if (k == 0 || d.len != k * len0 || k > cap - n_recs || d.src + d.len < d.src || d.dst + d.len < d.dst) {
                misfit = true;
                break;
            }
            for (uint64_t j = 0; j < k; ++j)
                recs[n_recs++] = UniformRec{d.src + j * len0, d.dst + j * len0};
            if (n_recs + (n - 1 - i) > cap) { // the rest must still fit one record each
                misfit = true;
                break;
            }
        }
        if (misfit) {
            upload_cache().put(device, staging, staging_cap); // something else: the general lowering decides
        } else {
            const int rc = build_block_plan(device, t, staging, staging_cap, n_recs, len0, n, nullptr, out);
            if (rc != kNotBlocks) return rc;
        }
    }

    // ---- host-side lowering ------------------------------------------------------
    std::vector<uint64_t> vsrc, vdst, vprefix;
    Records<PieceRec> pieces;
    // Descriptors of 256 B to 8 KiB, and longer ones whose source or destination does not
    // start on a 128-byte line, go to the piece kernel: measured faster there (fewer lines
    // split between wavefronts); line-aligned long descriptors stream best in 1 KiB chunks.
    constexpr uint64_t kPieceMinUnits = 16, kPieceMaxDescUnits = 512;
    vsrc.reserve(n);
    vdst.reserve(n);
    vprefix.reserve(n + 1);
    uint64_t units = 0, payload = 0, n_piece_descs = 0;
    LongDescs chunks(chunk_bytes);
    ByteDescs bytes;
    Staging buffer(device); // what is uploaded; items are written there at once
    bool asked_ahead = false; // for that buffer: once, as it takes a look at the whole list
    bool whole_chunks = false; // there are chunks of some aligned descriptor whatever becomes of those
    for (size_t i = 0; i < n; ++i) {
        const nixl_amd_copy_desc_t &d = descs[i];
        if (d.len == 0) continue;
        if (d.src == 0 || d.dst == 0)
            return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "plan_create: null address in descriptor " + std::to_string(i));
        if (d.src + d.len < d.src || d.dst + d.len < d.dst)
            return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "plan_create: address range wraps in descriptor " + std::to_string(i));
        if (((d.src | d.dst | d.len) & 15u) != 0) {
            if (((d.src + d.len) | (d.dst + d.len)) >> kPieceUnitsShift)
                return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "plan_create: address beyond 2^56");
            if (!asked_ahead) {
                asked_ahead = true;
                const size_t ahead = ByteDescs::ahead(descs, i, n);
                reap_uploads(device);
                if (ahead != 0) {
                    if (buffer.get(ahead) == hipSuccess)
                        bytes.items.lend(buffer.at, buffer.cap);
                    else
                        (void)hipGetLastError();
                }
            }
            i = bytes.take(descs, i, n) - 1; // this one, and the ones behind it as far as they are like it
            continue;
        }
        payload += d.len;
        const uint64_t du = d.len / 16u;
        if (du >= kPieceMinUnits && (du < kPieceMaxDescUnits || ((d.src | d.dst) & 127u) != 0)) {
            // Pieces of at most kPieceUnits units, one wavefront each.  The first piece is
            // cut so that every later one starts on a 128-byte line of the destination: no
            // line is then written by two wavefronts.
            if ((d.dst + d.len) >> kPieceUnitsShift)
                return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "plan_create: destination address beyond 2^56");
            const uint64_t head = kPieceUnits - ((d.dst >> 4) & 7u);
            PieceRec *at = pieces.room(du / kPieceUnits + 2, n);
            uint64_t src = d.src, dst = d.dst, left = du;
            for (uint64_t room = head; left > room; room = kPieceUnits) {
                *at++ = PieceRec{src, dst | ((room - 1) << kPieceUnitsShift)};
                src += room * 16u;
                dst += room * 16u;
                left -= room;
            }
            *at++ = PieceRec{src, dst | ((left - 1) << kPieceUnitsShift)};
            pieces.end_at(at);
            ++n_piece_descs;
        } else {
            whole_chunks |= du >= kPieceMaxDescUnits;
            if (du >= std::max(kPieceMaxDescUnits, chunk_units)) {
                chunks.add(d.src, d.dst, d.len, 0);
                continue;
            }
            vsrc.push_back(d.src);
            vdst.push_back(d.dst);
            vprefix.push_back(units);
            units += du;
        }
    }
    payload += bytes.payload;
    // A long byte descriptor whose two ends lie at the same place inside their lines (tensors whose
    // size is no multiple of 16) is chunks, the first and the last of them ends (whose lanes' 16
    // bytes start anywhere).  Alone and up to kSplitFromTotal the byte kernel has the shorter way: its
    // items are fewer than the chunks' records and need no kernel to write them.  Made, launched and
    // waited for, by the byte kernel and as chunks, us: 15 tensors of 1 MiB + 2 B 21.2 and 24.0, 15 of
    // 4 MiB + 6 B 38.0 and 40.9, 126 of 1 MiB + 2 B 63.7 and 60.9, 2031 of 64 KiB + 2 B 74.9 and 76.7; 255
    // of 1 MiB + 2 B 114 and 101, 4 of 120 MiB 233 and 174.
    const bool join = whole_chunks || bytes.splittable_total >= kSplitFromTotal;
    if (bytes.long_total - (join ? bytes.splittable_total : 0) > kLongItemsFrom) bytes.reach = kGenericItemBytes;
    const size_t n_aligned_runs = chunks.runs.size(), n_aligned_edges = chunks.edges;
    for (const uint32_t i : bytes.longs) {
        const nixl_amd_copy_desc_t &d = descs[i];
        if (!join || !ByteDescs::splittable(d)) {
            bytes.add(d.src, d.dst, d.len);
            continue;
        }
        // the chunks between the ends start on a line
        chunks.add(d.src, d.dst, d.len, (0 - ((0 - d.dst) & 127u)) % chunk_bytes);
    }
    vprefix.push_back(units);
    const size_t nv = vsrc.size();
    const uint64_t n_stream64 = (units + chunk_units - 1) / chunk_units;
    if (n_stream64 + chunks.n >= (1ull << 32) || bytes.items.n >= (1ull << 32) || pieces.n >= (1ull << 31))
        return nixl_amd_fail(NIXL_AMD_ERR_TOO_LARGE, "plan_create: request too large for 32-bit chunk index");
    const uint32_t n_stream = static_cast<uint32_t>(n_stream64), n_uniform_chunks = static_cast<uint32_t>(chunks.n);

    // The stream: descriptors shorter than a chunk.  Every chunk of it remembers the first and the
    // last descriptor that it touches.
    std::vector<uint2> span(n_stream);
    for (size_t c = 0, j = 0; c < n_stream; ++c) {
        const uint64_t first = c * chunk_units, last = std::min(units, first + chunk_units) - 1;
        while (vprefix[j + 1] <= first)
            ++j;
        size_t jl = j;
        while (vprefix[jl + 1] <= last)
            ++jl;
        span[c] = make_uint2(static_cast<uint32_t>(j), static_cast<uint32_t>(jl));
    }
    // Runs of the same whole number of chunks share a record each; else every chunk gets its own,
    // written on the device from the runs.
    const bool expand = !chunks.equal;
    const uint32_t chunks_per_rec = expand || chunks.runs.empty() ? 1 : static_cast<uint32_t>(chunks.runs[0].len / chunk_bytes);
    const size_t n_uniform_recs = expand ? n_uniform_chunks : chunks.runs.size();

    // ---- one device arena for all plan arrays --------------------------------------
    auto align256 = [](size_t x) { return (x + 255) & ~size_t(255); };
    const bool need_desc_arrays = n_stream != 0;
    // The arena ends with the records of chunks.  When they are expanded on the device, that stretch is not uploaded.
    const size_t off_items = 0;
    const size_t off_src = off_items + align256(bytes.items.n * sizeof(GenericItem));
    const size_t off_dst = off_src + (need_desc_arrays ? align256(nv * 8) : 0);
    const size_t off_prefix = off_dst + (need_desc_arrays ? align256(nv * 8) : 0);
    const size_t off_span = off_prefix + (need_desc_arrays ? align256((nv + 1) * 8) : 0);
    const size_t off_pieces = off_span + (need_desc_arrays ? align256(span.size() * sizeof(uint2)) : 0);
    const size_t off_runs = off_pieces + align256(pieces.n * sizeof(PieceRec));
    const size_t off_uni = off_runs + (expand ? align256(chunks.runs.size() * sizeof(ChunkRun)) : 0);
    const size_t total = off_uni + align256(n_uniform_recs * sizeof(UniformRec));
    const size_t uploaded = expand ? off_uni : total;

    auto *plan = new nixl_amd_copy_plan();
    plan->device = device;
    plan->upl = upl;
    if (nt == 0) {
        // Destinations that adjoin (a gather into staging, one long copy) or advance by a
        // constant step (the same block of every layer of a pool) take non-temporal loads where they
        // are long; destinations without such a pattern (a scatter over a pool) take plain loads.
        uint64_t pairs = 0, regular = 0, following = 0, prev_dst = 0, prev_end = 0, prev_step = 0, prev_src_end = 0;
        const bool matters = copy_policy(payload, true, true) != copy_policy(payload, false, false);
        for (size_t i = 0; matters && i < n; ++i) {
            if (descs[i].len == 0) continue;
            if (prev_end) {
                const uint64_t step = descs[i].dst - prev_dst;
                ++pairs;
                regular += (descs[i].dst == prev_end || step == prev_step);
                following += descs[i].src == prev_src_end;
                prev_step = step;
            }
            prev_dst = descs[i].dst;
            prev_end = descs[i].dst + descs[i].len;
            prev_src_end = descs[i].src + descs[i].len;
        }
        nt = copy_policy(payload, 2 * regular >= pairs, 2 * following >= pairs);
    }
    plan->policy = nt;
    plan->piece_policy = tuning && tuning->nontemporal ? tuning->nontemporal : copy_policy(payload, true, false);
    plan->waves = waves;
    plan->swizzle = swizzle;
    plan->max_wgs = max_wgs;

    if (total > 0) {
        Staging larger(device);
        hipError_t e = hipSuccess;
        if (buffer.cap < std::max<size_t>(uploaded, 256)) {
            reap_uploads(device);
            e = larger.get(std::max<size_t>(uploaded, 256));
            if (e != hipSuccess) {
                delete plan;
                return nixl_amd_fail(NIXL_AMD_ERR_HIP, std::string("hipHostMalloc(plan upload buffer): ") + hipGetErrorString(e));
            }
        }
        // the pinned buffer mirrors the arena; this function or the plan gives it back from here on
        Staging &from = larger.at ? larger : buffer;
        void *const staging = from.at;
        const size_t staging_cap = from.cap;
        const auto host = [&](size_t arena_offset) { return static_cast<uint8_t *>(staging) + arena_offset; };
        if (expand) {
            std::memcpy(host(off_runs), chunks.runs.data(), chunks.runs.size() * sizeof(ChunkRun));
        } else {
            auto *recs = reinterpret_cast<UniformRec *>(host(off_uni));
            for (const ChunkRun &run : chunks.runs)
                *recs++ = UniformRec{run.src, run.dst};
        }
        if (need_desc_arrays) {
            std::memcpy(host(off_src), vsrc.data(), nv * 8);
            std::memcpy(host(off_dst), vdst.data(), nv * 8);
            std::memcpy(host(off_prefix), vprefix.data(), (nv + 1) * 8);
            std::memcpy(host(off_span), span.data(), span.size() * sizeof(uint2));
        }
        if (pieces.n) std::memcpy(host(off_pieces), pieces.at, pieces.n * sizeof(PieceRec));
        if (bytes.items.n && bytes.items.at != staging) std::memcpy(host(off_items), bytes.items.at, bytes.items.n * sizeof(GenericItem));
        from.at = nullptr;
        e = arena_cache().get(device, total, &plan->arena, &plan->arena_cap);
        if (e != hipSuccess) {
            upload_cache().put(device, staging, staging_cap);
            delete plan;
            return nixl_amd_fail(NIXL_AMD_ERR_HIP, std::string("hipMalloc(plan arena): ") + hipGetErrorString(e));
        }
        hipStream_t up = nullptr;
        e = build_stream(plan, t, &up);
        auto *arena = static_cast<uint8_t *>(plan->arena);
        if (e == hipSuccess) e = upload(up, arena, staging, uploaded);
        if (e == hipSuccess && expand) {
            const uint32_t wgs = static_cast<uint32_t>(std::min<uint64_t>((static_cast<uint64_t>(n_uniform_chunks) + 255) / 256, 1u << 20));
            hipLaunchKernelGGL(expand_runs_kernel, dim3(wgs), dim3(256), 0, up, reinterpret_cast<UniformRec *>(arena + off_uni),
                               reinterpret_cast<const ChunkRun *>(arena + off_runs), static_cast<uint32_t>(chunks.runs.size()),
                               n_uniform_chunks, static_cast<uint32_t>(chunk_bytes),
                               static_cast<int>((chunks.address_bits >> kPieceUnitsShift) == 0));
            e = hipGetLastError();
        }
        if (e == hipSuccess) e = end_build(plan, up, staging, staging_cap);
        if (e != hipSuccess) {
            if (up) (void)hipStreamSynchronize(up); // a queued copy still reads the buffer given back below
            if (plan->uploaded) (void)hipEventDestroy(plan->uploaded);
            upload_cache().put(device, staging, staging_cap);
            arena_cache().put(device, plan->arena, plan->arena_cap);
            delete plan;
            return nixl_amd_fail(NIXL_AMD_ERR_HIP, std::string("hipMemcpy(plan arena): ") + hipGetErrorString(e));
        }
        plan->arena_bytes = total;
        auto *base = static_cast<uint8_t *>(plan->arena);
        plan->uniform_recs = reinterpret_cast<const UniformRec *>(base + off_uni);
        plan->mixed_args.src = reinterpret_cast<const uint64_t *>(base + off_src);
        plan->mixed_args.dst = reinterpret_cast<const uint64_t *>(base + off_dst);
        plan->mixed_args.prefix = reinterpret_cast<const uint64_t *>(base + off_prefix);
        plan->mixed_args.span = reinterpret_cast<const uint2 *>(base + off_span);
        plan->piece_recs = reinterpret_cast<const PieceRec *>(base + off_pieces);
        plan->generic_items = reinterpret_cast<const GenericItem *>(base + off_items);
    }
    plan->n_pieces = static_cast<uint32_t>(pieces.n);
    plan->n_uniform = n_uniform_chunks;
    plan->chunks_per_rec = chunks_per_rec;
    plan->mixed_args.total_units = units;
    plan->mixed_args.n_mixed = n_stream;
    plan->n_generic = static_cast<uint32_t>(bytes.items.n);

    auto wgs_for = [&](uint32_t n_waves, uint32_t waves_per_wg, bool cap) {
        uint32_t w = (n_waves + waves_per_wg - 1) / waves_per_wg;
        if (cap && plan->max_wgs && w > plan->max_wgs) w = plan->max_wgs;
        if (cap && w > kMaxGrid) w = kMaxGrid; // those kernels loop over their work items
        return w;
    };
    plan->uniform_wgs = wgs_for(plan->n_uniform, static_cast<uint32_t>(waves), false);
    plan->mixed_wgs = wgs_for(plan->mixed_args.n_mixed, kMixedWaves, true);
    plan->generic_wgs = wgs_for(plan->n_generic, kMixedWaves, true);

    plan->info.payload_bytes = payload;
    plan->info.vec_descs = nv + n_aligned_runs + n_piece_descs;
    plan->info.generic_descs = bytes.n;
    plan->info.plan_device_bytes = plan->arena_bytes;
    plan->info.vec_chunks = n_stream + n_uniform_chunks;
    // whole chunks, and the ends of aligned descriptors and the chunks of tiny ones
    plan->info.uniform_chunks = static_cast<uint32_t>(chunks.n - chunks.edges);
    plan->info.mixed_chunks = n_stream + static_cast<uint32_t>(n_aligned_edges);
    plan->info.generic_items = plan->n_generic;
    plan->info.piece_items = plan->n_pieces;
    plan->info.units_per_lane = static_cast<uint32_t>(upl);
    plan->info.uniform_workgroups = plan->uniform_wgs;
    *out = plan;
    return NIXL_AMD_OK;
}

int
nixl_amd_copy_block_len_fits(uint64_t len, const nixl_amd_copy_tuning_t *tuning) {
    Tuning t;
    if (parse_tuning(tuning, t, "block_len_fits")) return 0;
    return block_len_fits(len, t) ? 1 : 0;
}

int
nixl_amd_copy_records_begin(size_t max_records, nixl_amd_copy_records_t **out, nixl_amd_copy_record_t **records) {
    static_assert(sizeof(nixl_amd_copy_record_t) == sizeof(UniformRec));
    if (!out || !records) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "records_begin: null argument");
    *out = nullptr;
    *records = nullptr;
    if (max_records == 0 || max_records >= (1ull << 31))
        return nixl_amd_fail(NIXL_AMD_ERR_TOO_LARGE, "records_begin: between 1 and 2^31-1 records");
    auto *r = new nixl_amd_copy_records();
    r->max_records = max_records;
    const hipError_t e = upload_cache().get(0, max_records * sizeof(UniformRec), &r->staging, &r->staging_cap);
    if (e != hipSuccess) {
        delete r;
        return nixl_amd_fail(NIXL_AMD_ERR_HIP, std::string("hipHostMalloc(plan upload buffer): ") + hipGetErrorString(e));
    }
    *records = static_cast<nixl_amd_copy_record_t *>(r->staging);
    *out = r;
    return NIXL_AMD_OK;
}

int
nixl_amd_copy_records_abandon(nixl_amd_copy_records_t *records) {
    if (!records) return NIXL_AMD_OK;
    upload_cache().put(0, records->staging, records->staging_cap);
    delete records;
    return NIXL_AMD_OK;
}

int
nixl_amd_copy_plan_create_from_records(nixl_amd_copy_records_t *records,
                                       size_t n,
                                       uint64_t len,
                                       int device,
                                       const nixl_amd_copy_tuning_t *tuning,
                                       const nixl_amd_copy_record_facts_t *facts,
                                       nixl_amd_copy_plan_t **out) {
    if (!records) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "plan_create_from_records: records is null");
    // the buffer is taken over whatever happens below
    void *staging = records->staging;
    const size_t staging_cap = records->staging_cap, max_records = records->max_records;
    delete records;
    const auto give_back = [&](int code, const char *why) {
        upload_cache().put(0, staging, staging_cap);
        return nixl_amd_fail(code, why);
    };
    if (!out) return give_back(NIXL_AMD_ERR_INVALID, "plan_create_from_records: out is null");
    *out = nullptr;
    if (n == 0 || n > max_records) return give_back(NIXL_AMD_ERR_INVALID, "plan_create_from_records: record count outside the buffer");
    Tuning t;
    if (const int rc = parse_tuning(tuning, t, "plan_create_from_records")) {
        upload_cache().put(0, staging, staging_cap);
        return rc;
    }
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return give_back(NIXL_AMD_ERR_NO_DEVICE, "plan_create_from_records: no HIP device");
    if (device < 0 || device >= ndev) return give_back(NIXL_AMD_ERR_INVALID, "plan_create_from_records: bad device index");
    const DeviceScope on_device(device);
    if (on_device.status() != hipSuccess) return give_back(NIXL_AMD_ERR_HIP, "plan_create_from_records: hipSetDevice failed");
    reap_uploads(device);
    const int rc = build_block_plan(device, t, staging, staging_cap, n, len, n, facts, out);
    if (rc == kNotBlocks)
        return nixl_amd_fail(NIXL_AMD_ERR_INVALID,
                             "plan_create_from_records: blocks must be whole chunks of at least 8 KiB, start on 128-byte lines and not wrap");
    return rc;
}

int
nixl_amd_copy_plan_create_indexed_lists(const nixl_amd_copy_run_t *src_runs,
                                        size_t n_src_runs,
                                        const int32_t *src_index,
                                        uint64_t src_entries,
                                        const nixl_amd_copy_run_t *dst_runs,
                                        size_t n_dst_runs,
                                        const int32_t *dst_index,
                                        uint64_t dst_entries,
                                        size_t n,
                                        uint64_t len,
                                        int device,
                                        const nixl_amd_copy_tuning_t *tuning,
                                        nixl_amd_copy_plan_t **out) {
    if (!out) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "plan_create_indexed: out is null");
    *out = nullptr;
    if (!src_index || !dst_index || n == 0) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "plan_create_indexed: no indices");
    Tuning t;
    if (const int rc = parse_tuning(tuning, t, "plan_create_indexed")) return rc;
    const int upl = t.upl, nt = t.nt, waves = t.waves, swizzle = t.swizzle, sort_scatter = t.sort_scatter;
    const uint64_t chunk_bytes = static_cast<uint64_t>(kWaveSize) * upl * 16u;
    if (!src_runs || !dst_runs || n_src_runs == 0 || n_dst_runs == 0 || n_src_runs > kMaxIndexRuns || n_dst_runs > kMaxIndexRuns)
        return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "plan_create_indexed: between 1 and 256 runs a side");
    bool src_all_dense = true, dst_all_dense = true;
    for (int side = 0; side < 2; ++side) {
        const nixl_amd_copy_run_t *runs = side ? dst_runs : src_runs;
        const size_t n_runs = side ? n_dst_runs : n_src_runs;
        for (size_t r = 0; r < n_runs; ++r) {
            if (runs[r].base == 0 || ((runs[r].base | runs[r].stride) & 127u) != 0 || len == 0 || len % chunk_bytes != 0)
                return nixl_amd_fail(NIXL_AMD_ERR_INVALID,
                                     "plan_create_indexed: blocks must be whole chunks and start on 128-byte lines");
            if (runs[r].first_index != (r ? runs[r - 1].first_index + runs[r - 1].count : 0))
                return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "plan_create_indexed: runs must follow each other from index 0");
            (side ? dst_all_dense : src_all_dense) &= runs[r].stride == len;
        }
    }
    if (n >= (1ull << 31) || n * (len / chunk_bytes) >= (1ull << 32))
        return nixl_amd_fail(NIXL_AMD_ERR_TOO_LARGE, "plan_create_indexed: request too large for 32-bit chunk index");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0)
        return nixl_amd_fail(NIXL_AMD_ERR_NO_DEVICE, "plan_create_indexed: no HIP device");
    if (device < 0 || device >= ndev) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "plan_create_indexed: bad device index");
    const DeviceScope on_device(device);
    HIP_TRY(on_device.status());

    // The index vectors (and run tables) go into a pinned buffer, where the records kernel reads
    // them: every index is read once, so a copy to the device first would only add its latency.
    // Every workgroup reads the tables, but from the second one on out of the L2 (65 536 pairs with
    // 256 runs a side take 46 us to make, with 4 runs 45, with tables that are moved first 49).
    // The records of a few blocks are made right here instead.
    const size_t index_bytes = n * sizeof(int32_t);
    const bool inlined = fits_inline(n, len, t);
    const bool tables = n_src_runs > 1 || n_dst_runs > 1;
    const bool some = !inlined && !tables && fits_inline(n, len, t, kInlineIndices); // their indices may travel as arguments
    int32_t few[2 * kInlineIndices];
    const auto is_scattered = [](const IndexFacts &dst, size_t of) { return !(of == 1 || 2 * static_cast<uint64_t>(dst.regular) >= of - 1); };
    const auto follows = [&](const IndexFacts &src, size_t of) { return src_all_dense && 2 * static_cast<uint64_t>(src.ones) >= of - 1; };
    const auto is_sorted = [&](bool scattered, const IndexFacts &src, size_t of) {
        return scattered && sort_pays(sort_scatter, n, len) && follows(src, of);
    };
    const auto new_plan = [&](bool scattered, bool sort, bool following) {
        auto *plan = new nixl_amd_copy_plan();
        plan->device = device;
        plan->upl = upl;
        plan->waves = waves;
        plan->swizzle = swizzle;
        plan->policy = nt ? nt : copy_policy(n * len, !scattered || sort, following);
        return plan;
    };
    const auto keep_home = [&](nixl_amd_copy_plan &plan) { // of a plan without records, which may get some
        plan.home = t.stream == hipStreamLegacy || t.stream == hipStreamPerThread ? nullptr : t.stream;
        plan.later_policy = nt == 0 && plan.sort_later ? copy_policy(n * len, true, true) : plan.policy;
    };
    // More indices than an inline plan lists, but a grid.  It repeats itself, so its start says for all of it how regular it is.
    const auto grid_plan = [&](size_t of, const auto &facts) { // of the first `of` indices of both sides
        const auto sorted = [&] { // by the kernel that makes its records
            const auto [src, dst] = facts();
            return is_sorted(is_scattered(dst, of), src, of);
        };
        if ((sort_scatter == 1 || len >= kSortGridBlock) && sort_pays(sort_scatter, n, len) && sorted()) return false;
        auto grid = take_grid(src_runs[0], src_index, src_entries, dst_runs[0], dst_index, dst_entries, n, len);
        if (!grid) return false;
        const auto [src, dst] = facts();
        const bool scattered = is_scattered(dst, of), following = follows(src, of);
        auto *plan = new_plan(scattered, false, following);
        plan->sort_later = grid->by_column && len >= kSortGridBlock && n * len > kSortLaterFrom && sort_scatter == 0 && scattered && following;
        keep_home(*plan);
        plan->inline_grid = std::move(grid);
        describe_blocks(*plan, t, n, len, n);
        *out = plan;
        return true;
    };
    if (!inlined && !some && !tables && fits_inline(n, len, t, n)) {
        const size_t start = std::size(few) / 2;
        if (grid_plan(start, [&] {
                return std::pair(take_indices(src_index, start, few, src_all_dense, true),
                                 take_indices(dst_index, start, few + start, dst_all_dense, true));
            }))
            return NIXL_AMD_OK;
    }
    void *staging = nullptr;
    size_t staging_cap = 0;
    const size_t table_at = (2 * index_bytes + 15) & ~size_t(15); // the run tables follow the index vectors
    const size_t table_bytes = tables ? (n_src_runs + n_dst_runs) * sizeof(nixl_amd_copy_run_t) : 0;
    hipError_t e = hipSuccess;
    const auto take_staging = [&] {
        reap_uploads(device);
        e = upload_cache().get(device, table_at + table_bytes, &staging, &staging_cap);
        return e == hipSuccess ?
            NIXL_AMD_OK :
            nixl_amd_fail(NIXL_AMD_ERR_HIP, std::string("hipHostMalloc(plan upload buffer): ") + hipGetErrorString(e));
    };
    if (!inlined && !some)
        if (const int rc = take_staging()) return rc;
    // One pass over each vector on its way there: bounds, and the patterns that decide cache policy and
    // record order.  A request of 65 536 blocks made, one of whose vectors is consecutive: 51 us with a
    // pass each for a copy, bounds, the pinned copy and the pattern, 23 in one, 16 with the consecutive
    // one left where it is.
    int32_t *si = staging ? static_cast<int32_t *>(staging) : few, *di = si + n;
    const IndexFacts src_facts = take_indices(src_index, n, si, src_all_dense, inlined),
                     dst_facts = take_indices(dst_index, n, di, dst_all_dense, inlined);
    if (src_facts.highest >= src_entries || dst_facts.highest >= dst_entries) {
        if (staging) upload_cache().put(device, staging, staging_cap);
        return nixl_amd_fail(NIXL_AMD_ERR_INDEX, "plan_create_indexed: an index names no entry of its list");
    }
    const bool scattered = is_scattered(dst_facts, n), sort = is_sorted(scattered, src_facts, n);
    if (tables && !inlined) {
        auto *up_runs = reinterpret_cast<nixl_amd_copy_run_t *>(static_cast<uint8_t *>(staging) + table_at);
        std::memcpy(up_runs, src_runs, n_src_runs * sizeof(nixl_amd_copy_run_t));
        std::memcpy(up_runs + n_src_runs, dst_runs, n_dst_runs * sizeof(nixl_amd_copy_run_t));
    }
    auto *plan = new_plan(scattered, sort, follows(src_facts, n));
    if (inlined) {
        const auto address = [](const nixl_amd_copy_run_t *runs, size_t n_runs, uint64_t index) {
            const auto *run = std::upper_bound(runs, runs + n_runs, index, [](uint64_t i, const nixl_amd_copy_run_t &r) { return i < r.first_index; }) - 1;
            return run->base + (index - run->first_index) * run->stride;
        };
        plan->inline_recs = std::make_unique<InlineRecs>();
        for (size_t i = 0; i < n; ++i)
            plan->inline_recs->rec[i] = UniformRec{address(src_runs, n_src_runs, static_cast<uint64_t>(si[i])),
                                                   address(dst_runs, n_dst_runs, static_cast<uint64_t>(di[i]))};
        describe_blocks(*plan, t, n, len, n);
        *out = plan;
        return NIXL_AMD_OK;
    }
    const bool src_follows = src_facts.ones == n - 1, dst_follows = dst_facts.ones == n - 1;
    if (some) {
        const size_t words = (src_follows ? 0 : n) + (dst_follows ? 0 : n);
        if (words <= kInlineIndices) {
            std::unique_ptr<InlineIndices> in(new InlineIndices); // not cleared
            uint32_t place = 0;
            const auto side = [&](const nixl_amd_copy_run_t &run, const int32_t *index, bool follows) {
                InlineIndices::Side s{run.base, run.stride, static_cast<uint32_t>(index[0]), follows ? 0 : ~0u, follows ? 0 : place};
                if (!follows) {
                    std::memcpy(in->index + place, index, index_bytes);
                    place += static_cast<uint32_t>(n);
                }
                return s;
            };
            in->src = side(src_runs[0], si, src_follows);
            in->dst = side(dst_runs[0], di, dst_follows);
            keep_home(*plan);
            plan->inline_indices = std::move(in);
            describe_blocks(*plan, t, n, len, n);
            *out = plan;
            return NIXL_AMD_OK;
        }
        if (grid_plan(n, [&] { return std::pair(src_facts, dst_facts); })) {
            delete plan;
            return NIXL_AMD_OK;
        }
        if (const int rc = take_staging()) {
            delete plan;
            return rc;
        }
        std::memcpy(staging, few, 2 * index_bytes);
        si = static_cast<int32_t *>(staging);
        di = si + n;
    }
    const size_t rec_bytes = n * sizeof(UniformRec);
    hipStream_t up = nullptr;
    e = arena_cache().get(device, rec_bytes, &plan->arena, &plan->arena_cap);
    if (e == hipSuccess) e = build_stream(plan, t, &up);
    auto *recs = static_cast<UniformRec *>(plan->arena);
    if (e == hipSuccess) {
        const IndexVector src_at{src_follows ? nullptr : si, si[0]}, dst_at{dst_follows ? nullptr : di, di[0]};
        const auto launch = [&]<bool SORTED>() {
            const dim3 block(kIndexThreads<SORTED>), grid(static_cast<uint32_t>((n + block.x - 1) / block.x));
            if (tables) {
                const auto *runs = reinterpret_cast<const nixl_amd_copy_run_t *>(static_cast<const uint8_t *>(staging) + table_at);
                hipLaunchKernelGGL(index_records_runs_kernel<SORTED>, grid, block, 0, up, recs, src_at, dst_at, static_cast<uint32_t>(n),
                                   runs, static_cast<uint32_t>(n_src_runs), runs + n_src_runs, static_cast<uint32_t>(n_dst_runs));
            } else {
                hipLaunchKernelGGL(index_records_kernel<SORTED>, grid, block, 0, up, recs, src_at, dst_at, static_cast<uint32_t>(n),
                                   src_runs[0].base, src_runs[0].stride, dst_runs[0].base, dst_runs[0].stride);
            }
        };
        if (sort)
            launch.template operator()<true>();
        else
            launch.template operator()<false>();
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = end_build(plan, up, staging, staging_cap);
    if (e != hipSuccess) {
        if (up) (void)hipStreamSynchronize(up); // whatever was queued reads the buffers given back below
        if (plan->uploaded) (void)hipEventDestroy(plan->uploaded);
        upload_cache().put(device, staging, staging_cap);
        if (plan->arena) arena_cache().put(device, plan->arena, plan->arena_cap);
        delete plan;
        return nixl_amd_fail(NIXL_AMD_ERR_HIP, std::string("plan upload: ") + hipGetErrorString(e));
    }
    plan->arena_bytes = rec_bytes;
    plan->uniform_recs = recs;
    describe_blocks(*plan, t, n, len, n);
    *out = plan;
    return NIXL_AMD_OK;
}

int
nixl_amd_copy_plan_create_indexed_runs(const nixl_amd_copy_run_t *src_runs,
                                       size_t n_src_runs,
                                       const int32_t *src_index,
                                       const nixl_amd_copy_run_t *dst_runs,
                                       size_t n_dst_runs,
                                       const int32_t *dst_index,
                                       size_t n,
                                       uint64_t len,
                                       int device,
                                       const nixl_amd_copy_tuning_t *tuning,
                                       nixl_amd_copy_plan_t **out) {
    return nixl_amd_copy_plan_create_indexed_lists(src_runs, n_src_runs, src_index, UINT64_MAX, dst_runs, n_dst_runs, dst_index, UINT64_MAX,
                                                   n, len, device, tuning, out);
}

int
nixl_amd_copy_plan_create_indexed(uint64_t src_base,
                                  uint64_t src_stride,
                                  const int32_t *src_index,
                                  uint64_t dst_base,
                                  uint64_t dst_stride,
                                  const int32_t *dst_index,
                                  size_t n,
                                  uint64_t len,
                                  int device,
                                  const nixl_amd_copy_tuning_t *tuning,
                                  nixl_amd_copy_plan_t **out) {
    const nixl_amd_copy_run_t src{src_base, src_stride, 0, 0}, dst{dst_base, dst_stride, 0, 0};
    return nixl_amd_copy_plan_create_indexed_runs(&src, 1, src_index, &dst, 1, dst_index, n, len, device, tuning, out);
}

// A prepared list on the device, see nixl_amd_copy_list_create.
struct nixl_amd_copy_list {
    int device = 0;
    nixl_amd_copy_list_entry_t *entries = nullptr;
    size_t cap = 0; // size of the block the entries lie in
    uint32_t n = 0;
    uint32_t max_len = 0;
};

int
nixl_amd_copy_list_create(const nixl_amd_copy_list_entry_t *entries, size_t n, int device, nixl_amd_copy_list_t **out) {
    if (!out) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "list_create: out is null");
    *out = nullptr;
    if (!entries || n == 0) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "list_create: no entries");
    if (n >= (1ull << 30)) return nixl_amd_fail(NIXL_AMD_ERR_TOO_LARGE, "list_create: more than 2^30 entries");
    uint64_t address_bits = 0;
    uint32_t len_bits = 0, min_len = ~0u, max_len = 0, wraps = 0;
    for (size_t i = 0; i < n; ++i) {
        const nixl_amd_copy_list_entry_t &e = entries[i];
        address_bits |= e.addr;
        len_bits |= e.len;
        min_len = std::min(min_len, e.len);
        max_len = std::max(max_len, e.len);
        wraps |= static_cast<uint32_t>(e.addr == 0) | static_cast<uint32_t>(((e.addr + e.len) >> kPieceUnitsShift) != 0);
    }
    if (((address_bits | len_bits) & 15u) || min_len < kListMinBytes || max_len > kListMaxBytes || wraps)
        return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "list_create: entries must be 16-byte aligned and 128 to 8176 bytes long");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return nixl_amd_fail(NIXL_AMD_ERR_NO_DEVICE, "list_create: no HIP device");
    if (device < 0 || device >= ndev) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "list_create: bad device index");
    const DeviceScope on_device(device);
    HIP_TRY(on_device.status());
    void *mem = nullptr;
    size_t cap = 0;
    HIP_TRY(list_cache().get(device, n * sizeof(nixl_amd_copy_list_entry_t), &mem, &cap));
    // waits for the copy: the caller's array may go away, and the first request finds the table there
    hipStream_t up = nullptr;
    hipError_t e = upload_stream(device, &up);
    if (e == hipSuccess) e = hipMemcpyAsync(mem, entries, n * sizeof(nixl_amd_copy_list_entry_t), hipMemcpyHostToDevice, up);
    if (e == hipSuccess) e = hipStreamSynchronize(up);
    if (e != hipSuccess) {
        if (up) (void)hipStreamSynchronize(up);
        list_cache().put(device, mem, cap);
        return nixl_amd_fail(NIXL_AMD_ERR_HIP, std::string("list_create: ") + hipGetErrorString(e));
    }
    auto *list = new nixl_amd_copy_list();
    list->device = device;
    list->entries = static_cast<nixl_amd_copy_list_entry_t *>(mem);
    list->cap = cap;
    list->n = static_cast<uint32_t>(n);
    list->max_len = max_len;
    *out = list;
    return NIXL_AMD_OK;
}

int
nixl_amd_copy_list_destroy(nixl_amd_copy_list_t *list) {
    if (!list) return NIXL_AMD_OK;
    // nothing on the device reads a list once plan_create_listed has returned
    list_cache().put(list->device, list->entries, list->cap);
    delete list;
    return NIXL_AMD_OK;
}

int
nixl_amd_copy_list_device(const nixl_amd_copy_list_t *list) {
    return list ? list->device : nixl_amd_fail(NIXL_AMD_ERR_INVALID, "list_device: list is null");
}

static int
create_listed(const nixl_amd_copy_list_t *src,
              const int32_t *src_index,
              const nixl_amd_copy_list_t *dst,
              const int32_t *dst_index,
              size_t n,
              const nixl_amd_copy_tuning_t *tuning,
              bool on_stream,
              size_t *n_continued,
              nixl_amd_copy_plan_t **out) {
    if (!out) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "plan_create_listed: out is null");
    *out = nullptr;
    if (!src || !dst || !src_index || !dst_index || n == 0) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "plan_create_listed: null argument");
    if (src->device != dst->device) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "plan_create_listed: lists on different devices");
    Tuning t;
    if (const int rc = parse_tuning(tuning, t, "plan_create_listed")) return rc;
    if (!on_stream) t.stream = nullptr;
    // pieces a descriptor can have: its first line may hold back seven units of the first one
    const size_t max_units = std::min(src->max_len, dst->max_len) / 16u;
    const size_t per_desc = 1 + (max_units + 6) / kPieceUnits;
    if (n > (1ull << 31) / per_desc - 1) return nixl_amd_fail(NIXL_AMD_ERR_TOO_LARGE, "plan_create_listed: too many pairs");
    const int device = src->device;
    const DeviceScope on_device(device);
    HIP_TRY(on_device.status());

    const size_t index_bytes = n * sizeof(int32_t);
    const uint32_t workgroups = static_cast<uint32_t>((n + kListThreads - 1) / kListThreads);
    // The two vectors, each starting on a line as every slice of them does (no line is written by the
    // host after a kernel has read it), or in their place the runs and the run of every workgroup
    // (which take less: 16 bytes for kMinIndexRun pairs and more); then the verdict.
    const size_t dst_at = (index_bytes + 127) & ~size_t(127);
    const size_t verdict_at = 2 * dst_at + 128;
    static_assert(sizeof(IndexRun) <= kMinIndexRun * sizeof(int32_t) && kListThreads >= 64);
    void *staging = nullptr;
    size_t staging_cap = 0;
    reap_uploads(device);
    hipError_t e = upload_cache().get(device, verdict_at + sizeof(ListVerdict), &staging, &staging_cap);
    if (e != hipSuccess)
        return nixl_amd_fail(NIXL_AMD_ERR_HIP, std::string("hipHostMalloc(plan upload buffer): ") + hipGetErrorString(e));
    auto *up_src = static_cast<int32_t *>(staging), *up_dst = up_src + dst_at / sizeof(int32_t);
    auto *up_runs = static_cast<IndexRun *>(staging);
    auto *up_run_of = reinterpret_cast<uint32_t *>(up_dst);
    auto *verdict = reinterpret_cast<ListVerdict *>(static_cast<uint8_t *>(staging) + verdict_at);
    *verdict = ListVerdict{};

    auto *plan = new nixl_amd_copy_plan();
    plan->device = device;
    plan->upl = t.upl;
    plan->waves = t.waves;
    plan->swizzle = t.swizzle;
    plan->max_wgs = t.max_wgs;
    plan->policy = t.nt ? t.nt : kPolNtSc1Nt;
    // one arena: the totals, then the records
    constexpr size_t kRecsAt = 256;
    static_assert(sizeof(ListTotals) <= kRecsAt);
    hipStream_t up = nullptr;
    e = arena_cache().get(device, kRecsAt + n * per_desc * sizeof(PieceRec), &plan->arena, &plan->arena_cap);
    if (e == hipSuccess) e = build_stream(plan, t, &up);
    auto *recs = reinterpret_cast<PieceRec *>(static_cast<uint8_t *>(plan->arena) + kRecsAt);
    ListTotals *const slot = e == hipSuccess && device < kMaxDevices ? list_slots(device).take() : nullptr;
    ListTotals *const totals = slot ? slot : static_cast<ListTotals *>(plan->arena);
    bool queued = false; // something that adds to the totals
    if (e == hipSuccess && !slot) {
        hipLaunchKernelGGL(clear_totals_kernel, dim3(1), dim3(kWaveSize), 0, up, totals);
        e = hipGetLastError();
    }
    if (e == hipSuccess) {
        ListArgs a{recs, src->entries, dst->entries, src->n,  dst->n,
                   up_src, up_dst,      up_runs,      up_run_of, 0,
                   static_cast<uint32_t>(n), workgroups, totals, verdict};
        if (index_runs(src_index, dst_index, n, up_runs, up_run_of)) {
            hipLaunchKernelGGL(list_records_kernel<true>, dim3(workgroups), dim3(kListThreads), 0, up, a);
            e = hipGetLastError();
            queued = e == hipSuccess;
        } else {
            for (size_t at = 0; at < n && e == hipSuccess; at += kListSlice) {
                const size_t count = std::min(kListSlice, n - at);
                std::memcpy(up_src + at, src_index + at, count * sizeof(int32_t));
                std::memcpy(up_dst + at, dst_index + at, count * sizeof(int32_t));
                a.first_workgroup = static_cast<uint32_t>(at / kListThreads);
                hipLaunchKernelGGL(list_records_kernel<false>, dim3(static_cast<uint32_t>((count + kListThreads - 1) / kListThreads)),
                                   dim3(kListThreads), 0, up, a);
                e = hipGetLastError();
                queued = queued || e == hipSuccess;
            }
        }
    }
    if (e == hipSuccess) e = await_verdict(*verdict, up);
    const ListVerdict got = *verdict;
    if (slot && e != hipSuccess && queued) { // counted in part, or by nobody knows whom
        hipLaunchKernelGGL(clear_totals_kernel, dim3(1), dim3(kWaveSize), 0, up, totals);
        queued = hipGetLastError() != hipSuccess || hipStreamSynchronize(up) != hipSuccess;
    }
    if (slot && (e == hipSuccess || !queued)) list_slots(device).put(slot);
    // The records are complete when the last kernel ends, which comes behind its verdict: a launch
    // follows on the same stream, or waits for the event; a plan that may be launched anywhere, also into a
    // capture, is complete when the caller has it.
    if (e == hipSuccess && !plan->reserved && !got.bad) {
        e = hipEventCreateWithFlags(&plan->uploaded, hipEventDisableTiming);
        if (e == hipSuccess) e = hipEventRecord(plan->uploaded, up);
        if (e == hipSuccess && !on_stream) e = settle_upload(plan, true);
    }
    if ((e != hipSuccess || got.bad) && up) (void)hipStreamSynchronize(up); // whatever is queued uses the buffers given back below
    // the verdict is the last thing that is written there, and everything else has been read by then
    upload_cache().put(device, staging, staging_cap);
    if (e != hipSuccess || got.bad) {
        if (plan->uploaded) (void)hipEventDestroy(plan->uploaded);
        if (plan->arena) arena_cache().put(device, plan->arena, plan->arena_cap);
        delete plan;
        if (e != hipSuccess) return nixl_amd_fail(NIXL_AMD_ERR_HIP, std::string("plan_create_listed: ") + hipGetErrorString(e));
        return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "plan_create_listed: " + std::to_string(got.bad) +
                                                       " pairs name no entry or join entries of different lengths");
    }
    if (plan->reserved) {
        plan->built_on = up;
        plan->reserved = false; // no buffer waits with the plan
        g_held_staging.fetch_sub(1, std::memory_order_relaxed);
    }
    plan->arena_bytes = kRecsAt + (n + got.extra) * sizeof(PieceRec);
    plan->piece_recs = recs;
    plan->n_pieces = static_cast<uint32_t>(n + got.extra);
    plan->piece_policy = t.nt ? t.nt : copy_policy(got.bytes, true, false);
    plan->info.payload_bytes = got.bytes;
    plan->info.vec_descs = n;
    plan->info.plan_device_bytes = plan->arena_bytes;
    plan->info.piece_items = plan->n_pieces;
    plan->info.units_per_lane = static_cast<uint32_t>(t.upl);
    if (n_continued) *n_continued = got.continued;
    *out = plan;
    return NIXL_AMD_OK;
}

int
nixl_amd_copy_plan_create_listed(const nixl_amd_copy_list_t *src,
                                 const int32_t *src_index,
                                 const nixl_amd_copy_list_t *dst,
                                 const int32_t *dst_index,
                                 size_t n,
                                 const nixl_amd_copy_tuning_t *tuning,
                                 size_t *n_continued,
                                 nixl_amd_copy_plan_t **out) {
    return create_listed(src, src_index, dst, dst_index, n, tuning, false, n_continued, out);
}

int
nixl_amd_copy_plan_create_listed_on(const nixl_amd_copy_list_t *src,
                                    const int32_t *src_index,
                                    const nixl_amd_copy_list_t *dst,
                                    const int32_t *dst_index,
                                    size_t n,
                                    const nixl_amd_copy_tuning_t *tuning,
                                    size_t *n_continued,
                                    nixl_amd_copy_plan_t **out) {
    return create_listed(src, src_index, dst, dst_index, n, tuning, true, n_continued, out);
}

int
nixl_amd_copy_watch_prepare(void) {
    static std::mutex mutex;
    std::lock_guard<std::mutex> lock(mutex);
    if (g_done_slots.load(std::memory_order_relaxed)) return NIXL_AMD_OK;
    constexpr size_t kWords = static_cast<size_t>(kDoneSlots) * DoneSlots::kStride; // of a device
    int n = 0;
    HIP_TRY(hipGetDeviceCount(&n));
    n = std::min(n, kMaxDevices);
    uint32_t *words = nullptr;
    HIP_TRY(hipHostMalloc(reinterpret_cast<void **>(&words), n * kWords * sizeof(uint32_t), hipHostMallocPortable));
    std::memset(words, 0, n * kWords * sizeof(uint32_t));
    auto **all = new DoneSlots *[kMaxDevices]();
    for (int i = 0; i < n; ++i)
        all[i] = new DoneSlots(words + i * kWords);
    g_done_slots.store(all, std::memory_order_release);
    return NIXL_AMD_OK;
}

int
nixl_amd_copy_watch_stream(int device, void *stream, int own) {
    const hipStream_t s = static_cast<hipStream_t>(stream);
    if (!s || s == hipStreamLegacy || s == hipStreamPerThread)
        return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "watch_stream: a default stream is not the caller's alone");
    DoneSlots *const slots = done_slots(device);
    if (!slots) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "watch_stream: no words for this device (nixl_amd_copy_watch_prepare)");
    slots->own_stream(s, own != 0);
    return NIXL_AMD_OK;
}

// The records of a plan that was made without any (InlineIndices, GridIndices), or null if this launch is to go without.
// Making records costs a request that is launched once more than it gives, but one that is launched again and again
// pays for their lack every time: a wave finds its addresses by one more division and multiplication, a launch
// carries 3.7 KiB, and a scatter is not sorted.  Without and with, launch to end, us: 300 blocks of 8 KiB 10.4 and
// 9.5; gathers of grids 4096 of 1 KiB 10.8 and 9.6, 8192 of 16 KiB 51.0 and 50.0, 28 672 157.4 and 155.8; scatters listed by column
// 14 560 of 9 KiB 55.7 and 52.8, 50 944 176 and 166, 28 672 of 16 KiB 172 and 163, 32 640 196 and 182.5, 8160 of 64 KiB 181 and 172.  Hence
// the sixteenth launch on the stream that the plan was made for makes them, in front of its copy.  Only launches on
// that stream, which are behind their making, use them, and none into a capture, whose graph may be replayed
// anywhere: other launches go without, as before.
constexpr uint32_t kRecordsAt = 16;

static const UniformRec *
later_records(nixl_amd_copy_plan *plan, hipStream_t s, bool captured, bool *made) {
    if (!s || s != plan->home || captured) return nullptr;
    if (plan->later) return static_cast<const UniformRec *>(plan->later);
    if (plan->launches_at_home >= kRecordsAt || ++plan->launches_at_home < kRecordsAt) return nullptr; // tried once
    const uint32_t n = plan->n_uniform / plan->chunks_per_rec;
    const size_t bytes = static_cast<size_t>(n) * sizeof(UniformRec);
    // Another stream may be under a capture that allocations in any thread would end, but for those of a thread in this mode.
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    if (hipThreadExchangeStreamCaptureMode(&mode) != hipSuccess) return nullptr;
    const hipError_t had = arena_cache().get(plan->device, bytes, &plan->later, &plan->later_cap);
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (had != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    auto *recs = static_cast<UniformRec *>(plan->later);
    const auto launch = [&]<bool SORTED>(const auto &from) {
        hipLaunchKernelGGL((later_records_kernel<SORTED, std::decay_t<decltype(from)>>), dim3((n + kIndexThreads<SORTED> - 1) / kIndexThreads<SORTED>),
                           dim3(kIndexThreads<SORTED>), 0, s, recs, from, n);
    };
    if (plan->inline_indices)
        launch.template operator()<false>(*plan->inline_indices);
    else if (plan->sort_later)
        launch.template operator()<true>(*plan->inline_grid);
    else
        launch.template operator()<false>(*plan->inline_grid);
    if (hipGetLastError() != hipSuccess) {
        (void)hipStreamSynchronize(s); // unless the error is an earlier one's, and they are being made
        arena_cache().put(plan->device, plan->later, plan->later_cap);
        plan->later = nullptr;
        return nullptr;
    }
    plan->later_bytes.store(bytes, std::memory_order_relaxed);
    *made = true;
    return recs;
}

static int
launch_plan(nixl_amd_copy_plan_t *plan, void *stream, bool watched) {
    if (!plan) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "plan_launch: plan is null");
    const DeviceScope on_device(plan->device);
    HIP_TRY(on_device.status());
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (s && hipStreamIsCapturing(s, &capture) != hipSuccess) (void)hipGetLastError();
    if (plan->built_on && plan->ever_launched) {
        // An earlier launch followed the build: once it has run, so has the build.  Its event lies
        // on built_on: asking for it while that stream is captured would end the capture.
        if (plan->seen_done) {
            plan->built_on = nullptr;
        } else if (capture == hipStreamCaptureStatusNone && ended(plan, false) == hipSuccess) {
            plan->built_on = nullptr;
            give_back_staging(plan);
        }
    }
    if (plan->built_on && s == plan->built_on && capture != hipStreamCaptureStatusNone)
        return nixl_amd_fail(NIXL_AMD_ERR_INVALID,
                             "plan_launch: the stream a plan was made on is under capture and no launch of the plan has been seen "
                             "complete (nixl_amd_copy_plan_status)");
    if (plan->built_on && s != plan->built_on) {
        // not where the caller said: from here on the build is one on a stream of its own
        if (!plan->uploaded) HIP_TRY(hipEventCreateWithFlags(&plan->uploaded, hipEventDisableTiming));
        HIP_TRY(hipEventRecord(plan->uploaded, plan->built_on));
        plan->built_on = nullptr;
    }
    if (plan->uploaded) {
        hipError_t e = settle_upload(plan, false);
        if (e == hipErrorNotReady) {
            // A stream under graph capture must not be made to depend on work outside the
            // graph: the host waits instead, and the graph holds the launch alone.
            e = capture == hipStreamCaptureStatusNone ? hipStreamWaitEvent(s, plan->uploaded, 0) : hipErrorNotReady;
            if (e != hipSuccess) {
                (void)hipGetLastError();
                e = settle_upload(plan, true);
            }
        }
        HIP_TRY(e);
    }
    // The word this launch is watched by.  A plan whose earlier launch is still being watched takes an
    // event for this one: the two may run on different streams, and end in any order.
    // The legacy stream takes one, too: how its launch fares may not be asked while any stream is captured, and
    // without an answer a launch that failed would be waited for without end.  And the per-thread one, which is
    // another stream in the thread that asks.
    Done done{};
    const bool asked = s && s != hipStreamLegacy && s != hipStreamPerThread;
    DoneSlots *const slots = watched && asked && capture == hipStreamCaptureStatusNone ? done_slots(plan->device) : nullptr;
    if (slots && plan->slot.load(std::memory_order_relaxed) >= 0) (void)ended(plan, false);
    const bool failed = plan->watch_failure != hipSuccess;
    int slot = slots && (failed || plan->slot.load(std::memory_order_relaxed) < 0) ? slots->take(&done) : -1;
    bool told = false; // the copy writes the word itself
    bool made = false;
    const UniformRec *const later = later_records(plan, s, capture != hipStreamCaptureStatusNone, &made);
    const auto give_up = [&](hipError_t e) {
        if (made) (void)hipStreamSynchronize(s); // no launch that destroying the plan would wait for is behind the records
        if (slot >= 0) slots->put(slot); // nothing that would write its word is queued
        return nixl_amd_fail(NIXL_AMD_ERR_HIP, std::string("plan_launch: ") + hipGetErrorString(e));
    };
    const auto launch_inline = [&](const auto &recs) {
        using Recs = std::decay_t<decltype(recs)>;
        // The line between the two forms (above): at 4 MiB, 256 workgroups to be counted, 11.0 us and 11.3
        // with a kernel behind, the median of both 10.5; at 8 MiB 11.8 both, the median 11.5 and 10.8.
        constexpr uint32_t kToldChunks = 4096;
        const bool through = plan->policy == kPolPlainSc1Nt || plan->policy == kPolNtSc1Nt;
        if (slot >= 0 && through && plan->n_uniform <= kToldChunks) {
            const dim3 grid((plan->n_uniform + kDoneWaves * kDoneChunks - 1) / (kDoneWaves * kDoneChunks));
            const auto launch = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, grid, dim3(kWaveSize * kDoneWaves), 0, s, recs, FastDiv(plan->chunks_per_rec),
                                   plan->n_uniform, done);
            };
            if (plan->policy == kPolPlainSc1Nt)
                launch(copy_inline_done_kernel<kPolPlainSc1Nt, Recs>);
            else
                launch(copy_inline_done_kernel<kPolNtSc1Nt, Recs>);
            told = true;
        } else {
            with_policy(plan->policy, [&]<int POL>() {
                if constexpr (std::is_same_v<Recs, GridIndices>) {
                    const uint32_t length = recs.row_length.divisor, rows = plan->n_uniform / plan->chunks_per_rec / length;
                    hipLaunchKernelGGL(copy_grid_kernel<POL>, dim3(plan->chunks_per_rec * length, rows), dim3(kWaveSize), 0, s, recs,
                                       FastDiv(plan->chunks_per_rec));
                } else {
                    hipLaunchKernelGGL((copy_inline_kernel<POL, Recs>), dim3(plan->n_uniform), dim3(kWaveSize), 0, s, recs,
                                       FastDiv(plan->chunks_per_rec));
                }
            });
        }
        return hipGetLastError();
    };
    if (plan->inline_recs) {
        if (const hipError_t e = launch_inline(*plan->inline_recs); e != hipSuccess) return give_up(e);
    } else if (plan->inline_indices && !later) {
        if (const hipError_t e = launch_inline(*plan->inline_indices); e != hipSuccess) return give_up(e);
    } else if (plan->inline_grid && !later) {
        if (const hipError_t e = launch_inline(*plan->inline_grid); e != hipSuccess) return give_up(e);
    } else if (plan->uniform_wgs) {
        // One launch per kMaxGrid workgroups.  With the die swizzle each launch's grid is
        // rounded up to a multiple of 8 so that every die owns an equally long slice; surplus
        // workgroups exit at once.
        const uint32_t waves = static_cast<uint32_t>(plan->waves);
        for (uint64_t wg64 = 0; wg64 < plan->uniform_wgs; wg64 += kMaxGrid) {
            const uint32_t wg0 = static_cast<uint32_t>(wg64);
            UniformLaunch u{};
            u.recs = later ? later : plan->uniform_recs;
            u.first_chunk = wg0 * waves;
            u.n_chunks = plan->n_uniform - u.first_chunk;
            u.n_wgs = std::min(kMaxGrid, plan->uniform_wgs - wg0);
            u.chunks_per_rec = plan->chunks_per_rec;
            u.swizzle = plan->swizzle;
            u.grid = dim3(plan->swizzle ? ((u.n_wgs + kNumXcd - 1) / kNumXcd) * kNumXcd : u.n_wgs);
            u.stream = s;
            with_policy(later ? plan->later_policy : plan->policy, [&]<int POL>() { launch_uniform_upl<POL>(plan->upl, plan->waves, u); });
            if (const hipError_t e = hipGetLastError(); e != hipSuccess) return give_up(e);
        }
    }
    if (plan->n_pieces) {
        const uint32_t w = static_cast<uint32_t>(plan->waves > 4 ? 4 : plan->waves);
        const uint32_t per_launch = kMaxGrid * w;
        for (uint32_t p0 = 0; p0 < plan->n_pieces; p0 += per_launch) {
            const uint32_t n = std::min(per_launch, plan->n_pieces - p0);
            with_policy(plan->piece_policy,
                        [&]<int POL>() { launch_pieces<POL>(w, (n + w - 1) / w, s, plan->piece_recs + p0, n); });
            if (const hipError_t e = hipGetLastError(); e != hipSuccess) return give_up(e);
        }
    }
    if (plan->mixed_wgs) {
        with_policy(plan->policy, [&]<int POL>() { launch_mixed_upl<POL>(plan->upl, dim3(plan->mixed_wgs), s, plan->mixed_args); });
        if (const hipError_t e = hipGetLastError(); e != hipSuccess) return give_up(e);
    }
    if (plan->generic_wgs) {
        hipLaunchKernelGGL(copy_generic_kernel, dim3(plan->generic_wgs), dim3(kMixedThreads), 0, s,
                           plan->generic_items, plan->n_generic);
        if (const hipError_t e = hipGetLastError(); e != hipSuccess) return give_up(e);
    }
    // What nixl_amd_copy_plan_destroy looks at.  A stream under graph capture gets no event: the
    // graph's owner keeps the plan alive for as long as the graph may be replayed.
    if (slot >= 0 && !told) {
        hipLaunchKernelGGL(done_kernel, dim3(1), dim3(kWaveSize), 0, s, done.word, done.value);
        if (hipGetLastError() != hipSuccess) {
            slots->put(slot);
            slot = -1;
        }
    }
    if (failed && capture == hipStreamCaptureStatusNone) { // this launch is what the status is about from here on
        plan->slot = -1; // no other launch gets it: who knows whether something still writes there
        plan->watch_failure.store(hipSuccess);
    }
    if (slot >= 0) {
        plan->slot_value = done.value;
        plan->watched_on = s;
        plan->polls.store(0, std::memory_order_relaxed);
        slots->last_on(s, slot, done.value);
        plan->slot.store(slot, std::memory_order_release);
        plan->ever_launched = true;
    } else if (capture == hipStreamCaptureStatusNone) {
        if (DoneSlots *all = done_slots(plan->device)) all->last_on(s, -1, 0);
        if (!plan->launched) HIP_TRY(hipEventCreateWithFlags(&plan->launched, hipEventDisableTiming));
        HIP_TRY(hipEventRecord(plan->launched, s));
        plan->launched_valid = true;
        plan->ever_launched = true;
    }
    return NIXL_AMD_OK;
}

int
nixl_amd_copy_plan_launch(nixl_amd_copy_plan_t *plan, void *stream) {
    return launch_plan(plan, stream, false);
}

int
nixl_amd_copy_plan_launch_watched(nixl_amd_copy_plan_t *plan, void *stream) {
    return launch_plan(plan, stream, true);
}

int
nixl_amd_copy_plan_status(nixl_amd_copy_plan_t *plan, int wait) {
    if (!plan) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "plan_status: plan is null");
    if (!plan->ever_launched) return NIXL_AMD_OK;
    const DeviceScope on_device(plan->device);
    const hipError_t state = ended(plan, wait != 0);
    if (state == hipSuccess) {
        plan->seen_done = true;
        give_back_staging(plan);
        return NIXL_AMD_OK;
    }
    if (state == hipErrorNotReady) return NIXL_AMD_ERR_BUSY; // polled in a loop: no message is made for it
    return nixl_amd_fail(NIXL_AMD_ERR_HIP, std::string("plan_status: ") + hipGetErrorString(state));
}

int
nixl_amd_copy_plan_destroy(nixl_amd_copy_plan_t *plan) {
    if (!plan) return NIXL_AMD_OK;
    const DeviceScope on_device(plan->device);
    // The arena goes back to a pool that the next plan's upload writes into: not while a
    // launch of this plan may still read it.  The plan stays as it is; destroy it later.
    if (plan->ever_launched && ended(plan, false) == hipErrorNotReady)
        return nixl_amd_fail(NIXL_AMD_ERR_BUSY, "plan_destroy: a launch of this plan has not completed");
    if (plan->built_on && !plan->ever_launched) {
        // never launched: the build itself may still run, behind whatever is in front of it
        hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(plan->built_on, &capture) != hipSuccess) (void)hipGetLastError();
        if (capture != hipStreamCaptureStatusNone)
            return nixl_amd_fail(NIXL_AMD_ERR_BUSY, "plan_destroy: the stream the plan was made on is under capture");
        void *staging = plan->staging.exchange(nullptr);
        if (staging) g_held_staging.fetch_sub(1, std::memory_order_relaxed);
        recycle_after(plan->device, plan->built_on, true, staging, plan->staging_cap, plan->arena, plan->arena_cap);
        plan->arena = nullptr;
    }
    (void)settle_upload(plan, true); // the arena and the upload buffer go back only when nothing writes or reads them
    if (plan->launched) (void)hipEventDestroy(plan->launched);
    if (plan->ev0) (void)hipEventDestroy(plan->ev0);
    if (plan->ev1) (void)hipEventDestroy(plan->ev1);
    give_back_staging(plan);
    if (plan->arena) arena_cache().put(plan->device, plan->arena, plan->arena_cap);
    if (plan->later) arena_cache().put(plan->device, plan->later, plan->later_cap);
    delete plan;
    return NIXL_AMD_OK;
}

int
nixl_amd_copy_plan_query(const nixl_amd_copy_plan_t *plan, nixl_amd_copy_plan_info_t *info) {
    if (!plan || !info) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "plan_query: null argument");
    *info = plan->info;
    info->plan_device_bytes += plan->later_bytes.load(std::memory_order_relaxed);
    return NIXL_AMD_OK;
}

int
nixl_amd_copy_plan_time(nixl_amd_copy_plan_t *plan, void *stream, int iters, float *ms_per_launch) {
    if (!plan || !ms_per_launch || iters <= 0)
        return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "plan_time: bad argument");
    const DeviceScope on_device(plan->device);
    HIP_TRY(on_device.status());
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (!plan->ev0) HIP_TRY(hipEventCreate(&plan->ev0));
    if (!plan->ev1) HIP_TRY(hipEventCreate(&plan->ev1));
    HIP_TRY(hipEventRecord(plan->ev0, s));
    for (int i = 0; i < iters; ++i) {
        int rc = nixl_amd_copy_plan_launch(plan, stream);
        if (rc) return rc;
    }
    HIP_TRY(hipEventRecord(plan->ev1, s));
    HIP_TRY(hipEventSynchronize(plan->ev1));
    float ms = 0.f;
    HIP_TRY(hipEventElapsedTime(&ms, plan->ev0, plan->ev1));
    *ms_per_launch = ms / static_cast<float>(iters);
    return NIXL_AMD_OK;
}

} // extern "C"
