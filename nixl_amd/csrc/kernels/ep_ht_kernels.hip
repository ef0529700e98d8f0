// Normal-mode ("high-throughput") expert-parallel kernels and the router, for all virtual
// ranks of one GPU, with their C ABI (declared in include/nixl_amd_ep.h).
//
// The reference streams token rows through RDMA and NVLink ring queues, forwarding them hop
// by hop (kernels/nixl_ep_ht.cu:472-1245).  None of that exists when every rank is a region
// of the same HBM; what remains is the result: destination rows ordered by source rank then
// source token, rebased top-k indices, and the unweighted fp32 reduction on the way back.
// Positions come from prefix sums instead of queue heads:
//   row(r, t, d) = recv_row_offset[d] + recv_rank_prefix[d][r - 1] + send_head[r][t][d].
//
// HBM traffic: dispatch reads every source row once (2H) and writes it once per destination
// rank that holds one of its experts; combine reads those rows once and writes 2H per token.
#include <algorithm>
#include <cstdint>

#include "common.h"
#include "ep_common.h"
#include "nixl_amd_ep.h"

namespace {

constexpr int kScanThreads = 1024;

// Exclusive prefix of `v` over the workgroup (blockDim.x == kScanThreads); `total` gets the sum.
template<typename V>
__device__ __forceinline__ V
block_exclusive_scan(V v, V *wave_sums, V &total) {
    const int lane = threadIdx.x & (kWaveSize - 1), wave = threadIdx.x / kWaveSize;
    V incl = v;
#pragma unroll
    for (int off = 1; off < kWaveSize; off <<= 1) {
        const V up = __shfl_up(incl, off);
        if (lane >= off) incl += up;
    }
    __syncthreads(); // wave_sums may still be read from a previous call
    if (lane == kWaveSize - 1) wave_sums[wave] = incl;
    __syncthreads();
    constexpr int kWaves = kScanThreads / kWaveSize;
    V before = 0, sum = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        const V s = wave_sums[w];
        if (w < wave) before += s;
        sum += s;
    }
    total = sum;
    return before + incl - v;
}

// ---- layout (kernels/layout.cu:31-138) ----------------------------------------------------
// grid = R source ranks x chunks of blockDim.x tokens, one token per thread; LDS: E + R
// counters per workgroup, added to the (zeroed) outputs at the end.  Integer sums: the
// result does not depend on the order of the additions.  A rank of at most kLayoutWhole tokens
// and kLayoutWholeSelections selections is one chunk, whose counters are the result: nothing to
// clear and nothing to add (GPU time, one chunk against several: 8 x 1024 tokens top-4 4.1 and 4.7 us,
// 4 x 512 top-2 2.8 and 4.4, 8 x 512 top-8 4.8 and 5.4; top-6 of 1024 is even, 4.8 and 5.2).  Beyond, the
// LDS atomics of a single workgroup cost more than a second launch: 8 x 1024 top-8 7.6 and 5.5, 8 x 512
// top-16 7.7 and 7.2.  So do the flags of many ranks, R bytes a token by one thread, beyond
// kLayoutWholeFlags a rank: 32 x 768 tokens 5.0 and 5.1 us, 32 x 1024 5.9 and 5.1, 64 x 384 5.5 and 7.0, 64 x 768
// 8.7 and 8.1, 128 x 384 42 and 37; a single chunk of kLayoutTokens tokens is one workgroup either way, and
// from 256 ranks on one workgroup a rank fills the chip (256 x 384 121 and 159, 256 x 1024 327 and 592).
constexpr int kMaxTopk = 16; // check_ht
constexpr int kLayoutTokens = 256;
constexpr int kLayoutWhole = 1024;
constexpr int kLayoutWholeSelections = 4096;
constexpr int kLayoutWholeFlags = 24576;
constexpr int kLayoutWholeRanks = 256;

__global__ void __launch_bounds__(256)
zero_ints_kernel(int *__restrict__ a, size_t na, int *__restrict__ b, size_t nb) {
    const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < na) a[i] = 0;
    if (i < nb) b[i] = 0;
}

__global__ void __launch_bounds__(kLayoutWhole)
layout_kernel(const int32_t *__restrict__ topk_idx,
              int *__restrict__ per_rank,
              int *__restrict__ per_expert,
              uint8_t *__restrict__ in_rank,
              int T,
              int K,
              int R,
              int E,
              FastDiv chunks,
              FastDiv of_rank) { // experts of a rank
    extern __shared__ int counters[]; // [E] experts, then [R] ranks
    uint32_t chunk;
    const int src = chunks.quotient(blockIdx.x, chunk);
    const int t = chunk * blockDim.x + threadIdx.x;
    for (int i = threadIdx.x; i < E + R; i += blockDim.x)
        counters[i] = 0;
    __syncthreads();
    // whether the R flag bytes of a token can be written as one aligned 8-byte word
    const bool word_flags = R == 8 && (reinterpret_cast<uintptr_t>(in_rank) & 7u) == 0;
    if (t < T) {
        const int32_t *sel = topk_idx + (static_cast<size_t>(src) * T + t) * K;
        uint8_t *flags = in_rank + (static_cast<size_t>(src) * T + t) * R;
        if (R <= 64) {
            // destination ranks of the token as a bit mask in a register
            unsigned long long mask = 0;
            for (int k = 0; k < K; ++k) {
                const int e = sel[k];
                if (e < 0 || e >= E) continue;
                atomicAdd(&counters[e], 1);
                mask |= 1ull << of_rank.quotient(e);
            }
            if (word_flags) {
                // bit d to byte d: a copy of the bits in every byte, its own one of them, and that to the last place
                const unsigned long long own = (mask * 0x0101010101010101ull) & 0x8040201008040201ull;
                *reinterpret_cast<unsigned long long *>(flags) = ((own + 0x7f7f7f7f7f7f7f7full) >> 7) & 0x0101010101010101ull;
            } else {
                for (int d = 0; d < R; ++d)
                    flags[d] = static_cast<uint8_t>((mask >> d) & 1ull);
            }
            while (mask) {
                const int d = __builtin_ctzll(mask);
                mask &= mask - 1;
                atomicAdd(&counters[E + d], 1);
            }
        } else {
            for (int d = 0; d < R; ++d)
                flags[d] = 0;
            for (int k = 0; k < K; ++k) {
                const int e = sel[k];
                if (e < 0 || e >= E) continue;
                atomicAdd(&counters[e], 1);
                flags[of_rank.quotient(e)] = 1;
            }
            for (int d = 0; d < R; ++d)
                if (flags[d]) atomicAdd(&counters[E + d], 1);
        }
    }
    __syncthreads();
    if (chunks.divisor == 1) {
        for (int i = threadIdx.x; i < E; i += blockDim.x)
            per_expert[static_cast<size_t>(src) * E + i] = counters[i];
        for (int i = threadIdx.x; i < R; i += blockDim.x)
            per_rank[static_cast<size_t>(src) * R + i] = counters[E + i];
        return;
    }
    for (int i = threadIdx.x; i < E; i += blockDim.x)
        if (counters[i]) atomicAdd(&per_expert[static_cast<size_t>(src) * E + i], counters[i]);
    for (int i = threadIdx.x; i < R; i += blockDim.x)
        if (counters[E + i]) atomicAdd(&per_rank[static_cast<size_t>(src) * R + i], counters[E + i]);
}

// ---- notify, part 1: per (source, destination) pair, positions inside the segment and the
// per-channel prefix (kernels/nixl_ep_ht.cu:324-373).  grid = R * R workgroups. ----------------
__global__ void __launch_bounds__(kScanThreads)
ht_scan_kernel(const uint8_t *__restrict__ in_rank,
               int *__restrict__ send_head,
               int *__restrict__ channel_prefix,
               int T,
               int R,
               int C) {
    __shared__ int wave_sums[kScanThreads / kWaveSize];
    const int src = blockIdx.x / R, d = blockIdx.x % R;
    const int per_thread = (T + kScanThreads - 1) / kScanThreads;
    const int t0 = min(static_cast<int>(threadIdx.x) * per_thread, T), t1 = min(t0 + per_thread, T);
    const int per_channel = (T + C - 1) / C;
    int mine = 0;
    for (int t = t0; t < t1; ++t)
        mine += in_rank[(static_cast<size_t>(src) * T + t) * R + d] != 0;
    int total;
    int pos = block_exclusive_scan(mine, wave_sums, total);
    for (int t = t0; t < t1; ++t) {
        const bool hit = in_rank[(static_cast<size_t>(src) * T + t) * R + d] != 0;
        __builtin_nontemporal_store(hit ? pos : -1, &send_head[(static_cast<size_t>(src) * T + t) * R + d]);
        pos += hit;
        // `pos` is now the number of hits in tokens [0, t]; a channel's inclusive prefix
        // is that number at the channel's last token.
        if ((t + 1) % per_channel == 0 || t + 1 == T) {
            const int c = t / per_channel;
            channel_prefix[(static_cast<size_t>(src) * R + d) * C + c] = pos;
        }
    }
    // channels that start at or beyond T are empty: they repeat the grand total
    if (threadIdx.x == 0)
        for (int c = (T + per_channel - 1) / per_channel; c < C; ++c)
            channel_prefix[(static_cast<size_t>(src) * R + d) * C + c] = total;
}

// The same for up to 8 ranks and fewer than 65 536 tokens, which is every shipping
// configuration.  A workgroup owns one chunk of kScanThreads tokens of one source rank, one
// token per thread, and handles all destinations at once with four 16-bit counters to a
// 64-bit word: it first counts the hits of the chunks before its own (a reduction; chunks do
// not wait for each other), then scans its own.  A thread writes the R positions of its
// token as one run, a wave consecutive runs.  The positions are stored non-temporally: the
// row kernel that follows reads them from every XCD, and lines left dirty in the writer's L2
// made those reads slow (+45 us on 8 x 4096 tokens).  grid = R * ceil(T / kScanThreads), and one
// more workgroup where that also does part 2 (notify_from_flags).
constexpr int kPackedScanRanks = 8;
constexpr int kPackedScanMaxTokens = 65535;

struct PackedCounts {
    unsigned long long lo, hi; // destinations 0..3 and 4..7, 16 bits each
};

__device__ __forceinline__ int
packed_field(const PackedCounts &c, int d) {
    return static_cast<int>(((d < 4 ? c.lo : c.hi) >> (16 * (d & 3))) & 0xffffu);
}

__device__ __forceinline__ PackedCounts
packed_hits(const uint8_t *flags, int t, int R) {
    PackedCounts hit{0, 0};
    if (R == 8) {
        const unsigned long long f = *reinterpret_cast<const unsigned long long *>(flags + static_cast<size_t>(t) * 8);
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            hit.lo |= static_cast<unsigned long long>(((f >> (8 * d)) & 0xffu) != 0) << (16 * d);
            hit.hi |= static_cast<unsigned long long>(((f >> (8 * (d + 4))) & 0xffu) != 0) << (16 * d);
        }
    } else if (R == 4) {
        const uint32_t f = *reinterpret_cast<const uint32_t *>(flags + static_cast<size_t>(t) * 4);
#pragma unroll
        for (int d = 0; d < 4; ++d)
            hit.lo |= static_cast<unsigned long long>(((f >> (8 * d)) & 0xffu) != 0) << (16 * d);
    } else {
        for (int d = 0; d < R; ++d) {
            const unsigned long long bit = flags[static_cast<size_t>(t) * R + d] != 0;
            if (d < 4)
                hit.lo |= bit << (16 * d);
            else
                hit.hi |= bit << (16 * (d - 4));
        }
    }
    return hit;
}

// Four dwords of two fields each; the upper two only where there are more than four ranks.
template<typename Op>
__device__ __forceinline__ PackedCounts
each_half(const PackedCounts &c, bool upper, const Op &op) {
    const auto both = [&](unsigned long long x) {
        return static_cast<unsigned long long>(op(static_cast<uint32_t>(x >> 32))) << 32 | op(static_cast<uint32_t>(x));
    };
    return {both(c.lo), upper ? both(c.hi) : 0ull};
}

// ---- notify, part 2: receive-side prefix over source ranks, aligned per-expert counts
// (kernels/nixl_ep_ht.cu:295-314) and where each destination's rows start in the
// concatenated outputs.  One workgroup; total_of(r, d) = tokens of source r that go to
// destination d. ------------------------------------------------------------------------------
struct HtNotifyOut {
    const int *per_expert;
    int *recv_rank_prefix;
    int *recv_expert_count;
    long long *row_offset;
    int *recv_counter;
    int alignment;
};

__device__ __forceinline__ int
aligned(int n, int alignment) {
    return (n + alignment - 1) / alignment * alignment;
}

// Experts from `first_expert` on: those before it are done.
template<typename TotalOf>
__device__ __forceinline__ void
notify_prefix(const HtNotifyOut &o, int R, int E, int first_expert, const TotalOf &total_of) {
    __shared__ int wave_sums[kScanThreads / kWaveSize];
    const int tid = threadIdx.x;
    // Loads go out eight at a time before anything depends on them: issued one by one, the
    // round trips of this single workgroup add up to most of the kernel's time.
    constexpr int kBatch = 8;
    for (int e = first_expert + tid; e < E; e += kScanThreads) {
        int n = 0;
        for (int r0 = 0; r0 < R; r0 += kBatch) {
            int v[kBatch];
#pragma unroll
            for (int j = 0; j < kBatch; ++j)
                v[j] = r0 + j < R ? o.per_expert[static_cast<size_t>(r0 + j) * E + e] : 0;
#pragma unroll
            for (int j = 0; j < kBatch; ++j)
                n += v[j];
        }
        o.recv_expert_count[e] = aligned(n, o.alignment);
    }
    // R <= kScanThreads: thread d owns destination d
    int total = 0;
    if (tid < R) {
        for (int r0 = 0; r0 < R; r0 += kBatch) {
            int v[kBatch];
#pragma unroll
            for (int j = 0; j < kBatch; ++j)
                v[j] = r0 + j < R ? total_of(r0 + j, tid) : 0;
#pragma unroll
            for (int j = 0; j < kBatch; ++j)
                if (r0 + j < R) {
                    total += v[j];
                    o.recv_rank_prefix[tid * R + r0 + j] = total;
                }
        }
        if (o.recv_counter) o.recv_counter[tid] = total;
    }
    if (o.row_offset) {
        // exclusive prefix of the per-destination totals in 64 bits
        long long incl = total;
        const int lane = tid & (kWaveSize - 1), wave = tid / kWaveSize;
        if (R <= kWaveSize && wave != 0) return; // the first wave has them all
        for (int off = 1; off < min(R, kWaveSize); off <<= 1) {
            const long long up = __shfl_up(incl, off);
            if (lane >= off) incl += up;
        }
        if (R <= kWaveSize) {
            if (tid < R) o.row_offset[tid + 1] = incl;
            if (tid == 0) o.row_offset[0] = 0;
            return;
        }
        // wave totals fit in 32 bits each only if R * T does; check_ht bounds R * T by 2^30
        if (lane == kWaveSize - 1) wave_sums[wave] = static_cast<int>(incl);
        __syncthreads();
        long long before = 0;
        for (int w = 0; w < wave; ++w)
            before += wave_sums[w];
        if (tid < R) o.row_offset[tid + 1] = before + incl;
        if (tid == 0) o.row_offset[0] = 0;
    }
}

__global__ void __launch_bounds__(kScanThreads)
ht_prefix_kernel(const int *__restrict__ channel_prefix, HtNotifyOut o, int R, int E, int C) {
    notify_prefix(o, R, E, 0, [&](int r, int d) { return channel_prefix[(static_cast<size_t>(r) * R + d) * C + (C - 1)]; });
}

// The same without a launch of its own, for up to 8 ranks: one more workgroup behind those of the
// scan counts the flags itself instead of waiting for their counts.  What bounds it is one
// workgroup's way to flags that another kernel has just written, so every wave has a share of a
// rank's tokens, eight loads in flight a lane, and counts bytes (eight destinations an addition)
// that are widened once a step.  Up to so many tokens that the one workgroup is not slower than the
// launch (layout, scan and this behind one another, one launch and two, us): 8 x 1024 tokens 8.0 and
// 10.5, 8 x 5120 13.5 and 14.3, 8 x 6000 14.5 and 13.0; 4 x 12 288 13.9 and 14.6, 4 x 16 384 16.2 and 15.7.
// Where a token's flags are no word that one load takes, the kernels alone are as fast in two launches from some 4000
// flags on (6 x 200 10.2 and 9.2), but the host has a launch more in front of its wait for the counts: whole passes
// of layout, dispatch and combine (hidden 2048) take 38.2 and 39.7 for 6 x 200, 38.8 and 39.1 for 6 x 340, 39.1 and
// 38.2 for 6 x 400; 5 x 491 40.0 and 38.5, 3 x 1365 42.1 and 42.0, 2 x 3072 42.7 and 43.2, 1 x 12 000 51.0 and 52.7.
constexpr int kNotifyTokensOf8 = 40960, kNotifyTokensOf4 = 57344; // R * T
constexpr int kNotifyFlags = 12288; // R * T * R, other numbers of ranks
constexpr int kNotifyPerLane = 8; // tokens a lane counts at a time, their loads together

// The flags of a token, a byte a destination (R <= 8).
template<int RANKS>
__device__ __forceinline__ unsigned long long
token_flags(const uint8_t *flags, int t, int R) {
    const uint8_t *at = flags + static_cast<size_t>(t) * R;
    if constexpr (RANKS == 8) return *reinterpret_cast<const unsigned long long *>(at);
    if constexpr (RANKS == 4) return *reinterpret_cast<const uint32_t *>(at);
    unsigned long long f = 0;
    for (int d = 0; d < R; ++d)
        f |= static_cast<unsigned long long>(at[d]) << (8 * d);
    return f;
}

// One in every byte of `flags` that is not zero.
__device__ __forceinline__ unsigned long long
byte_flags(unsigned long long flags) {
    constexpr unsigned long long kLow7 = 0x7f7f7f7f7f7f7f7full, kOnes = 0x0101010101010101ull;
    return ((((flags & kLow7) + kLow7) | flags) >> 7) & kOnes;
}

// Four bytes as four 16-bit fields.
__device__ __forceinline__ unsigned long long
widen_bytes(uint32_t bytes) {
    unsigned long long x = bytes;
    x = (x | x << 16) & 0x0000ffff0000ffffull;
    return (x | x << 8) & 0x00ff00ff00ff00ffull;
}

// Hits of this thread's share of the tokens before `base` (a multiple of kScanThreads), four loads in flight.
template<int RANKS>
__device__ __forceinline__ PackedCounts
hits_before(const uint8_t *flags, int base, int R) {
    constexpr int kBatch = 4;
    PackedCounts n{0, 0};
    for (int u0 = 0; u0 < base; u0 += kBatch * kScanThreads) {
        unsigned long long f[kBatch], sum = 0;
#pragma unroll
        for (int j = 0; j < kBatch; ++j)
            f[j] = u0 + j * kScanThreads < base ? token_flags<RANKS>(flags, u0 + j * kScanThreads + threadIdx.x, R) : 0;
#pragma unroll
        for (int j = 0; j < kBatch; ++j)
            sum += byte_flags(f[j]);
        n.lo += widen_bytes(static_cast<uint32_t>(sum));
        n.hi += widen_bytes(static_cast<uint32_t>(sum >> 32));
    }
    return n;
}

// RANKS: the number of ranks, or 0 where it is known at run time only.
template<int RANKS>
__device__ __forceinline__ void
notify_from_flags(const uint8_t *in_rank, const HtNotifyOut &o, int T, int n_ranks, int E) {
    const int R = RANKS ? RANKS : n_ranks;
    constexpr int kWaves = kScanThreads / kWaveSize, kUnit = kWaveSize * kNotifyPerLane;
    constexpr unsigned long long kEven = 0x00ff00ff00ff00ffull;
    const int tid = threadIdx.x, lane = tid & (kWaveSize - 1), wave = tid / kWaveSize;
    __shared__ int hits[kWaves][kPackedScanRanks]; // what a wave has counted
    // the counts of the first experts travel while the flags do
    int of_rank[kPackedScanRanks];
#pragma unroll
    for (int r = 0; r < kPackedScanRanks; ++r)
        if (r < R && tid < E) of_rank[r] = o.per_expert[static_cast<size_t>(r) * E + tid];
    // as many waves to a rank as there are; a wave adds up what it counts in 16-bit fields (T < 65 536)
    const int per_rank = kWaves / R, r = wave / per_rank;
    if (r < R) {
        const uint8_t *flags = in_rank + static_cast<size_t>(r) * T * R;
        unsigned long long even = 0, odd = 0; // destinations 0, 2, 4, 6 and 1, 3, 5, 7
        for (int t0 = (wave % per_rank) * kUnit + lane; t0 - lane < T; t0 += per_rank * kUnit) {
            unsigned long long f[kNotifyPerLane], sum = 0;
#pragma unroll
            for (int j = 0; j < kNotifyPerLane; ++j) {
                const int t = t0 + j * kWaveSize;
                f[j] = t < T ? token_flags<RANKS>(flags, t, R) : 0;
            }
#pragma unroll
            for (int j = 0; j < kNotifyPerLane; ++j)
                sum += byte_flags(f[j]);
            even += sum & kEven;
            odd += (sum >> 8) & kEven;
        }
        const PackedCounts sums = each_half(PackedCounts{even, odd}, true, wave_sum_dpp);
        even = sums.lo;
        odd = sums.hi;
        if (lane < R) hits[wave][lane] = static_cast<int>(((lane & 1 ? odd : even) >> (8 * (lane & 6))) & 0xffffu);
    }
    if (tid < E) {
        int n = 0;
#pragma unroll
        for (int r = 0; r < kPackedScanRanks; ++r)
            if (r < R) n += of_rank[r];
        o.recv_expert_count[tid] = aligned(n, o.alignment);
    }
    __syncthreads();
    notify_prefix(o, R, E, kScanThreads, [&](int r, int d) {
        int n = 0;
        for (int w = 0; w < per_rank; ++w)
            n += hits[r * per_rank + w][d];
        return n;
    });
}

// NOTIFY: the launch has that workgroup.
template<bool NOTIFY>
__global__ void __launch_bounds__(kScanThreads)
ht_scan_packed_kernel(const uint8_t *__restrict__ in_rank,
                      int *__restrict__ send_head,
                      int *__restrict__ channel_prefix,
                      int T,
                      int R,
                      int C,
                      int E,
                      HtNotifyOut notify) {
    constexpr int kWaves = kScanThreads / kWaveSize;
    __shared__ PackedCounts wave_sums[kWaves], wave_before[kWaves];
    const int chunks = (T + kScanThreads - 1) / kScanThreads;
    if (NOTIFY && static_cast<int>(blockIdx.x) == R * chunks) {
        if (R == 8)
            notify_from_flags<8>(in_rank, notify, T, R, E);
        else if (R == 4)
            notify_from_flags<4>(in_rank, notify, T, R, E);
        else
            notify_from_flags<0>(in_rank, notify, T, R, E);
        return;
    }
    const int src = blockIdx.x / chunks, base = (blockIdx.x % chunks) * kScanThreads;
    const int tid = threadIdx.x, lane = tid & (kWaveSize - 1), wave = tid / kWaveSize;
    const int per_channel = (T + C - 1) / C;
    const uint8_t *flags = in_rank + static_cast<size_t>(src) * T * R;
    const int t = base + tid;

    // own token first, so that its load overlaps the count of the earlier chunks
    PackedCounts hit{0, 0};
    if (t < T) hit = packed_hits(flags, t, R);
    PackedCounts earlier{0, 0};
    if (base > 0) {
        earlier = R == 8 ? hits_before<8>(flags, base, R) : R == 4 ? hits_before<4>(flags, base, R) : hits_before<0>(flags, base, R);
        earlier = each_half(earlier, R > 4, wave_sum_dpp);
    }
    PackedCounts incl = each_half(hit, R > 4, wave_scan_dpp); // inside the wave
    if (lane == kWaveSize - 1) wave_sums[wave] = incl;
    if (lane == 0) wave_before[wave] = earlier;
    __syncthreads();
    // second level by the first wave: wave_sums[w] becomes the hits before wave w (earlier
    // chunks included), wave_before[0] the grand total up to the end of this chunk
    if (wave == 0) {
        PackedCounts s{0, 0}, e{0, 0};
        if (lane < kWaves) {
            s = wave_sums[lane];
            e = wave_before[lane];
        }
        const PackedCounts run = each_half(s, R > 4, wave_scan_dpp); // lanes beyond the waves add nothing
        e = each_half(e, R > 4, wave_sum_dpp);
        if (lane < kWaves) wave_sums[lane] = PackedCounts{run.lo - s.lo + e.lo, run.hi - s.hi + e.hi};
        if (lane == kWaves - 1) wave_before[0] = PackedCounts{run.lo + e.lo, run.hi + e.hi};
    }
    __syncthreads();
    const PackedCounts before = wave_sums[wave], total = wave_before[0];
    incl.lo += before.lo; // hits in tokens [0, t]
    incl.hi += before.hi;
    if (t < T) {
        int out[kPackedScanRanks];
#pragma unroll
        for (int d = 0; d < kPackedScanRanks; ++d)
            out[d] = packed_field(hit, d) ? packed_field(incl, d) - 1 : -1;
        int *dst = send_head + (static_cast<size_t>(src) * T + t) * R;
        if (R == 8) {
            st16_nt(dst, make_uint4(out[0], out[1], out[2], out[3]));
            st16_nt(dst + 4, make_uint4(out[4], out[5], out[6], out[7]));
        } else {
#pragma unroll
            for (int d = 0; d < kPackedScanRanks; ++d)
                if (d < R) __builtin_nontemporal_store(out[d], dst + d);
        }
        if ((t + 1) % per_channel == 0 || t + 1 == T) {
            const int c = t / per_channel;
            for (int d = 0; d < R; ++d)
                channel_prefix[(static_cast<size_t>(src) * R + d) * C + c] = packed_field(incl, d);
        }
    }
    // channels that start at or beyond T are empty: they repeat the grand total, which the
    // workgroup of the last chunk knows
    if (tid == 0 && base + kScanThreads >= T)
        for (int c = (T + per_channel - 1) / per_channel; c < C; ++c)
            for (int d = 0; d < R; ++d)
                channel_prefix[(static_cast<size_t>(src) * R + d) * C + c] = packed_field(total, d);
}

struct HtDims {
    int R, T, H, K, E;
};

// Rows of the ranks before r in destination dst's segment.  The load is there whatever r is: behind a branch the
// loads around it wait for it, a trip to memory more in front of every row.
__device__ __forceinline__ int
rows_before(const int *prefix, const HtDims &d, int r, int dst) {
    const int n = prefix[dst * d.R + max(r - 1, 0)];
    return r == 0 ? 0 : n;
}

__device__ __forceinline__ long long
recv_row(const int *prefix, const int *send_head, const long long *row_offset, const HtDims &d, int r, int t, int dst) {
    const int seg = r == 0 ? 0 : prefix[dst * d.R + r - 1];
    return row_offset[dst] + seg + send_head[(static_cast<size_t>(r) * d.T + t) * d.R + dst];
}

constexpr int kHtBatch = 8; // row loads a lane keeps in flight in combine

// The rows of token (r, t) at destinations d0 .. d0 + 63, found by one wave, lane = destination
// - d0: no LDS and no barrier, so that waves of a workgroup need not serve the same token.
// EAGER: positions are loaded beside the flags instead of behind them.
struct WaveRows {
    unsigned long long hits; // destinations that hold the token
    long long mine; // the row at this lane's
};

template<bool EAGER>
__device__ __forceinline__ WaveRows
wave_rows(const uint8_t *in_rank,
          const int *prefix,
          const int *send_head,
          const long long *row_offset,
          const HtDims &d,
          int r,
          int t,
          int d0) {
    const int dst = d0 + (threadIdx.x & (kWaveSize - 1));
    const size_t tok = static_cast<size_t>(r) * d.T + t;
    bool hit = false;
    long long row = 0;
    // the handle comes from the caller: a row outside the destination's range is dropped
    if (EAGER) {
        if (dst < d.R) {
            const uint8_t flag = in_rank[tok * d.R + dst];
            const int head = send_head[tok * d.R + dst], seg = rows_before(prefix, d, r, dst);
            const long long lo = row_offset[dst], hi = row_offset[dst + 1];
            row = lo + seg + head;
            hit = flag != 0 && row >= lo && row < hi;
        }
    } else {
        hit = dst < d.R && in_rank[tok * d.R + dst] != 0;
        if (hit) {
            row = recv_row(prefix, send_head, row_offset, d, r, t, dst);
            hit = row >= row_offset[dst] && row < row_offset[dst + 1];
        }
    }
    return {__ballot(hit), row};
}

// Row of the lowest destination in `hits`, which leaves the set.
__device__ __forceinline__ long long
next_row(const WaveRows &w, unsigned long long &hits) {
    const int lane = __builtin_ctzll(hits);
    hits &= hits - 1;
    const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(w.mine), lane);
    const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(w.mine >> 32), lane);
    return static_cast<long long>((static_cast<unsigned long long>(hi) << 32) | lo);
}

// ---- dispatch (result of kernels/nixl_ep_ht.cu:1109-1243) -------------------------------------
// Rows, scales and metadata in one launch (ht_dispatch_kernel below); these are its three parts.
//
// Rows: a wave owns 1 KiB of a row (`parts` waves a row), holds it in registers and stores it to
// every row of the token.  Bound by the writes, which carry device scope.  Inputs of more than
// kHtStreamFrom (half the last-level cache) are loaded non-temporally, smaller ones ordinarily:
// what a large call loads pushes lines out of the cache that the kernel which made the input left
// there.  8 x 4096 x 7168 bf16 with combine, ordinary and non-temporal loads, us a pass: behind an
// element-wise kernel on the input 1159 and 1106, behind a 512 MB fill 1103 and 1068, again and
// again 957 and 979.  8 x 1024 x 4096 (67 MB) is the same either way behind a producer, and a
// dispatch again and again takes 44 and 54.
//
// Positions of rows are loaded beside the flags (EAGER) or behind them, which spares the loads of
// destinations that do not hold the token and is faster for large calls whose tokens go to many.
// Beside, behind, and by the rows, us a pass of 8 x 4096 x 7168 bf16 top-8 with combine: 1006, 960,
// 959 with experts anywhere (5.3 rows a token), 713, 714, 713 with those of four ranks a token
// (3.6 rows), 481, 501, 481 of two.  Beside the flags in any case: the scales of fp8 rows (738
// beside, 769 behind) and inputs up to kHtStreamFrom, which are the same either way.
constexpr long long kHtStreamFrom = 128ll << 20;
constexpr int kHtManyRows = 4; // a token

struct HtRows {
    uint16_t *recv_x;
    const uint16_t *x;
    const uint8_t *in_rank;
    const int *prefix;
    const int *send_head;
    const long long *row_offset;
    HtDims d;
    FastDiv parts, tokens; // workgroups a row, tokens a rank
    int streamed; // rows are loaded non-temporally
};

// BY_ROWS: the number of rows decides when positions are loaded (else beside the flags).  It lies behind the last
// rank's offset, is there as early as the flags, and only the host would have to wait for it.
template<bool BY_ROWS>
__device__ __forceinline__ void
dispatch_piece(const HtRows &a, uint32_t piece) {
    uint32_t part, t_of_rank;
    const uint32_t token = a.parts.quotient(piece, part);
    if (token >= static_cast<uint32_t>(a.d.R) * a.d.T) return;
    const int r = a.tokens.quotient(token, t_of_rank), t = t_of_rank;
    const int col = part * kWaveSize + (threadIdx.x & (kWaveSize - 1));
    const bool active = col < a.d.H / 8;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (active) {
        const uint4 *from = reinterpret_cast<const uint4 *>(a.x + static_cast<size_t>(token) * a.d.H) + col;
        v = a.streamed ? ld16_nt(from) : *from;
    }
    const bool few = !BY_ROWS || a.row_offset[a.d.R] <= static_cast<long long>(kHtManyRows) * a.d.R * a.d.T;
    for (int d0 = 0; d0 < a.d.R; d0 += kWaveSize) {
        const WaveRows w = few ? wave_rows<true>(a.in_rank, a.prefix, a.send_head, a.row_offset, a.d, r, t, d0) :
                                 wave_rows<false>(a.in_rank, a.prefix, a.send_head, a.row_offset, a.d, r, t, d0);
        for (unsigned long long hits = w.hits; hits;) {
            const long long row = next_row(w, hits);
            if (active) st16_stream(reinterpret_cast<uint4 *>(a.recv_x + static_cast<size_t>(row) * a.d.H) + col, v);
        }
    }
}

// Per-row metadata: rebased top-k indices, weights of the local selections, source rank and
// token.  grid = R * R * ceil(T / 256): (source, destination) pairs major, one token per
// thread.  Consecutive tokens that go to the destination occupy consecutive rows,
// so a wave writes a contiguous stretch of each array; written from the row kernel above,
// the same bytes were isolated 32-byte stores and cost several times as long.
constexpr int kHtMetaThreads = 256;

// VEC: selections moved four at a time and the (rank, token) pair in one store; the host
// picks it when K is a multiple of 4 and every pointer is 16-byte aligned.
struct HtMeta {
    int32_t *recv_topk_idx;
    float *recv_topk_weights;
    int32_t *recv_src_meta;
    const int32_t *topk_idx;
    const float *topk_weights;
};

// Up to kMaxTopk values in registers, zeroes where there is nothing to load.
template<bool VEC, typename One, typename Four>
struct Few {
    One one[VEC ? 1 : kMaxTopk];
    Four four[VEC ? kMaxTopk / 4 : 1];

    __device__ __forceinline__ void
    load(const One *from, int n) {
        if constexpr (VEC) {
#pragma unroll
            for (int k = 0; k < kMaxTopk; k += 4)
                four[k / 4] = from && k < n ? *reinterpret_cast<const Four *>(from + k) : Four{};
        } else {
#pragma unroll
            for (int k = 0; k < kMaxTopk; ++k)
                one[k] = from && k < n ? from[k] : One{};
        }
    }
};

template<bool VEC>
__device__ __forceinline__ void
meta_block(const HtMeta &m,
           const uint8_t *__restrict__ in_rank,
           const int *__restrict__ prefix,
           const int *__restrict__ send_head,
           const long long *__restrict__ row_offset,
           const HtDims &d,
           uint32_t block) {
    int32_t *__restrict__ recv_topk_idx = m.recv_topk_idx;
    float *__restrict__ recv_topk_weights = m.recv_topk_weights;
    int32_t *__restrict__ recv_src_meta = m.recv_src_meta;
    const int32_t *__restrict__ topk_idx = m.topk_idx;
    const float *__restrict__ topk_weights = m.topk_weights;
    const int blocks_per_pair = (d.T + kHtMetaThreads - 1) / kHtMetaThreads;
    const int pair = block / blocks_per_pair;
    const int r = pair / d.R, dst = pair % d.R;
    const int t = (block % blocks_per_pair) * kHtMetaThreads + threadIdx.x;
    if (t >= d.T) return;
    const size_t tok = static_cast<size_t>(r) * d.T + t;
    if (!in_rank[tok * d.R + dst]) return;
    // the token's selections travel beside its row's position, all of them before one is looked at
    Few<VEC, int, int4> sel;
    Few<VEC, float, float4> weight;
    if (recv_topk_idx) {
        sel.load(topk_idx + tok * d.K, d.K);
        weight.load(topk_weights ? topk_weights + tok * d.K : nullptr, d.K);
    }
    const long long row = recv_row(prefix, send_head, row_offset, d, r, t, dst);
    if (row < row_offset[dst] || row >= row_offset[dst + 1]) return;
    const int lo = dst * (d.E / d.R), hi = lo + d.E / d.R;
    if (VEC && recv_topk_idx) {
        // four selections a step: 16-byte loads and stores (tok*K and row*K are multiples of 4)
#pragma unroll
        for (int k = 0; k < kMaxTopk; k += 4) {
            if (k >= d.K) break;
            const int4 s = sel.four[k / 4];
            const bool l0 = s.x >= lo && s.x < hi, l1 = s.y >= lo && s.y < hi;
            const bool l2 = s.z >= lo && s.z < hi, l3 = s.w >= lo && s.w < hi;
            *reinterpret_cast<int4 *>(recv_topk_idx + row * d.K + k) =
                make_int4(l0 ? s.x - lo : -1, l1 ? s.y - lo : -1, l2 ? s.z - lo : -1, l3 ? s.w - lo : -1);
            if (recv_topk_weights) {
                const float4 w = weight.four[k / 4];
                *reinterpret_cast<float4 *>(recv_topk_weights + row * d.K + k) =
                    make_float4(l0 ? w.x : 0.f, l1 ? w.y : 0.f, l2 ? w.z : 0.f, l3 ? w.w : 0.f);
            }
        }
    } else if (recv_topk_idx) {
#pragma unroll
        for (int k = 0; k < kMaxTopk; ++k) {
            if (k >= d.K) break;
            const bool local = sel.one[k] >= lo && sel.one[k] < hi;
            recv_topk_idx[row * d.K + k] = local ? sel.one[k] - lo : -1;
            if (recv_topk_weights) recv_topk_weights[row * d.K + k] = local ? weight.one[k] : 0.f;
        }
    }
    if (recv_src_meta) {
        if (VEC) {
            *reinterpret_cast<int2 *>(recv_src_meta + row * 2) = make_int2(r, t);
        } else {
            recv_src_meta[row * 2] = r;
            recv_src_meta[row * 2 + 1] = t;
        }
    }
}

// Per-token scales that travel with the rows (kernels/nixl_ep_ht.cu:729 reads them at
// token * scale_token_stride + i * scale_hidden_stride, :1198-1209 writes them densely per
// received row).  grid = R * R * ceil(T / 64): the first wave resolves the rows of 64
// consecutive tokens of one (source, destination) pair into LDS; the workgroup then moves
// their scales through an LDS tile of 64 tokens x 64 scales.  The tile is filled along
// whichever index is contiguous in the source (tokens, for the transposed storage the
// reference's callers pass; scales otherwise) and drained along the scales, so that a wave
// reads and writes consecutive addresses either way (consecutive tokens that go to the
// destination occupy consecutive rows).  Scales are moved as 32-bit words whatever they
// hold (fp32 or packed UE8M0).
constexpr int kHtScaleTokens = 64;
constexpr int kHtScaleTile = 64;
constexpr int kHtScaleThreads = 256;

struct HtScales {
    uint32_t *recv;
    const uint32_t *scales;
    int S;
    int wide; // S is a multiple of 4 and recv is 16-byte aligned
    long long rank_stride;
    long long token_stride;
    long long scale_stride;
};

__device__ __forceinline__ void
scales_block(const HtScales &a,
             const uint8_t *__restrict__ in_rank,
             const int *__restrict__ prefix,
             const int *__restrict__ send_head,
             const long long *__restrict__ row_offset,
             const HtDims &d,
             uint32_t block) {
    uint32_t *__restrict__ recv_scales = a.recv;
    const uint32_t *__restrict__ scales = a.scales;
    const int S = a.S, wide = a.wide;
    const long long rank_stride = a.rank_stride, token_stride = a.token_stride, scale_stride = a.scale_stride;
    __shared__ long long rows[kHtScaleTokens];
    __shared__ uint32_t tile[kHtScaleTokens][kHtScaleTile + 1]; // odd pitch: no bank conflicts either way
    const int blocks_per_pair = (d.T + kHtScaleTokens - 1) / kHtScaleTokens;
    const int pair = block / blocks_per_pair;
    const int r = pair / d.R, dst = pair % d.R;
    const int t0 = (block % blocks_per_pair) * kHtScaleTokens;
    const int tid = threadIdx.x;
    if (tid < kHtScaleTokens) {
        const int t = min(t0 + tid, d.T - 1);
        const uint8_t flag = in_rank[(static_cast<size_t>(r) * d.T + t) * d.R + dst];
        const long long row = recv_row(prefix, send_head, row_offset, d, r, t, dst);
        rows[tid] = flag && t == t0 + tid && row >= row_offset[dst] && row < row_offset[dst + 1] ? row : -1;
    }
    __syncthreads();
    const uint32_t *__restrict__ src = scales + static_cast<long long>(r) * rank_stride;
    const bool tokens_contiguous = token_stride < scale_stride;
    for (int g0 = 0; g0 < S; g0 += kHtScaleTile) {
        const int gs = min(kHtScaleTile, S - g0);
        // every load of the tile is issued before the first value is used: one load, one
        // LDS write at a time, the round trips of the 16 steps add up
        constexpr int kSteps = kHtScaleTokens * kHtScaleTile / kHtScaleThreads;
        uint32_t v[kSteps];
        int at[kSteps];
#pragma unroll
        for (int k = 0; k < kSteps; ++k) {
            const int i = tid + k * kHtScaleThreads;
            const int j = tokens_contiguous ? i % kHtScaleTokens : i / gs;
            const int g = tokens_contiguous ? i / kHtScaleTokens : i - j * gs;
            at[k] = -1;
            v[k] = 0;
            if (i < kHtScaleTokens * gs && rows[j] >= 0) {
                at[k] = j * (kHtScaleTile + 1) + g;
                v[k] = src[static_cast<long long>(t0 + j) * token_stride + static_cast<long long>(g0 + g) * scale_stride];
            }
        }
#pragma unroll
        for (int k = 0; k < kSteps; ++k)
            if (at[k] >= 0) (&tile[0][0])[at[k]] = v[k];
        __syncthreads();
        if (wide) {
            // four scales a store: the isolated 4-byte stores of the narrow form run at a
            // fraction of the rate
            const int quads = gs / 4;
            for (int i = tid; i < kHtScaleTokens * quads; i += kHtScaleThreads) {
                const int j = i / quads, q = (i - j * quads) * 4;
                const long long row = rows[j];
                if (row >= 0)
                    *reinterpret_cast<uint4 *>(recv_scales + row * S + g0 + q) =
                        make_uint4(tile[j][q], tile[j][q + 1], tile[j][q + 2], tile[j][q + 3]);
            }
        } else {
            for (int i = tid; i < kHtScaleTokens * gs; i += kHtScaleThreads) {
                const int j = i / gs, g = i - j * gs;
                const long long row = rows[j];
                if (row >= 0) recv_scales[row * S + g0 + g] = tile[j][g];
            }
        }
        __syncthreads();
    }
}

// One launch for the three: workgroups of the scales and of the metadata first, whose short
// writes then run beside the rows', four pieces of rows to a workgroup behind them.  Launched one
// after the other, the three took 14.6 us at 4 x 333 x 4096 fp8 (now 6.9), 157 at 8 x 2048 x 7168
// fp8 (145, and 132 with the loads and stores described at the rows), 55.3 at 8 x 1024 x 4096
// bf16 (52.9 and 49.5).  A launch holds fewer than 2^24 such workgroups (2^32 threads); a call of
// more is launched part by part, each part from its workgroup `first` on.
constexpr int kHtThreads = 256;
constexpr int kHtWaves = kHtThreads / kWaveSize;
constexpr long long kHtMaxGrid = (1ll << 24) - 1;
static_assert(kHtThreads == kHtMetaThreads && kHtThreads == kHtScaleThreads);

template<bool VEC, bool SCALES, bool BY_ROWS>
__global__ void __launch_bounds__(kHtThreads)
ht_dispatch_kernel(HtRows a, HtMeta m, HtScales sc, uint32_t scale_blocks, uint32_t meta_blocks, uint32_t first) {
    uint32_t block = blockIdx.x;
    if (SCALES) {
        if (block < scale_blocks) {
            scales_block(sc, a.in_rank, a.prefix, a.send_head, a.row_offset, a.d, first + block);
            return;
        }
        block -= scale_blocks;
    }
    if (block < meta_blocks) {
        meta_block<VEC>(m, a.in_rank, a.prefix, a.send_head, a.row_offset, a.d, first + block);
        return;
    }
    dispatch_piece<BY_ROWS>(a, (first + block - meta_blocks) * kHtWaves + uniform(threadIdx.x / kWaveSize));
}

// From this many ranks on, the metadata has a launch of its own: a workgroup of it finds one token in
// R / K of its own and is soon gone, and the three kinds' arguments and branches in front
// of it cost more than the launch.  Metadata alone at 64 ranks x 4096 tokens, top-4: 79 us by its own
// kernel, 129 by the common one; whole dispatches there, rows loaded ordinarily, 1286 -> 1254 us, 64 x 3000 x 512 fp8
// 1121 -> 1080, 128 x 3000 x 512 4510 -> 4370, 32 x 3000 x 512 325 -> 317; 24 x 4096 256 -> 262,
// 16 x 4096 141 -> 142, 8 x 4096 61 -> 67.
constexpr int kHtMetaApartRanks = 32;

template<bool VEC>
__global__ void __launch_bounds__(kHtMetaThreads)
ht_meta_kernel(HtMeta m,
               const uint8_t *__restrict__ in_rank,
               const int *__restrict__ prefix,
               const int *__restrict__ send_head,
               const long long *__restrict__ row_offset,
               HtDims d,
               uint32_t first) {
    meta_block<VEC>(m, in_rank, prefix, send_head, row_offset, d, first + blockIdx.x);
}

// ---- combine (combine_token, kernels/nixl_ep_ht.cu:1682-1737) -----------------------------------
// grid = R*T*parts; a row is H/8 lanes of 16 bytes and a workgroup covers blockDim.x of them,
// every wave for itself.  Positions are loaded beside the flags (EAGER), which shortens the chain
// of loads, or behind them, which spares loads and is faster for large calls whose tokens gather
// more than four rows: 8 x 4096 x 7168, eager and not, 317 and 337 us with 3.4 rows a token, 363
// and 363 with 3.9, 409 and 397 with 4.4, 481 and 464 with 5.3.  Up to kHtCombineEager values the eager form is
// as fast or faster with any number (8 x 256 x 7168, 5.3 rows, 30.0 and 30.9), and a call that does
// not say how many rows there are is eager up to that size.
// A wave a workgroup, but four where a row is whole workgroups of them and tokens gather few rows:
// 8 x 4096 x 4096 134 and 138 with one at 1.9 rows, 182.5 and 181.9 at 3.4; rows of 7168, which leave
// a fourth of every fourth workgroup idle, 175 and 165 (4 x 4096, 3.6 rows).
// With many ranks a look-up is many loads, the more so an eager one.  From kHtCombineManyRanks on large
// calls are eager up to three rows a token (64 x 512 x 4096, 3.9 rows, eager and not 237 and 232), and up to
// kHtCombineMostRanks, or kHtCombineMostRanksShared where four waves share the look-up (96 x 146 x 7168, 2.0 rows,
// 142 and 156; 256 x 54 x 7168 282 and 184; 128 x 192 x 4096 142 and 162, 256 x 96 x 4096 226 and 191).
// From kHtCombineManyRanksSmall on small ones share it if the row is whole workgroups of four waves
// (four and one: 40 x 194 x 4096, 7.3 rows, 90.2 and 93.6, 96 x 162 x 2048 96.6 and 108.1, 16 x 972 x 2048 82.9 and
// 82.3; 64 x 69 x 7168 39.8 and 37.1), and above kHtCombineMostRanksShared if it is long
// (160 x 38 x 5120, 2.0 rows, 64.0 and 70.0, 160 x 77 x 2560 71.4 and 69.4).
constexpr int kHtCombineEagerLanes = 256;
constexpr long long kHtCombineEager = 1ll << 25;
constexpr int kHtCombineManyRows = 4, kHtCombineFewRows = 3; // a token; few are as many as are not many in a small call
constexpr int kHtCombineManyRanks = 48, kHtCombineManyRanksSmall = 32, kHtCombineMostRanks = 96, kHtCombineMostRanksShared = 128;
constexpr int kHtCombineLongRow = 512; // lanes

template<bool EAGER>
__global__ void __launch_bounds__(kHtCombineEagerLanes)
ht_combine_kernel(uint16_t *__restrict__ combined,
                  float *__restrict__ combined_w,
                  const uint16_t *__restrict__ x,
                  const float *__restrict__ topk_weights,
                  const uint16_t *__restrict__ bias0,
                  const uint16_t *__restrict__ bias1,
                  const uint8_t *__restrict__ in_rank,
                  const int *__restrict__ prefix,
                  const int *__restrict__ send_head,
                  const long long *__restrict__ row_offset,
                  HtDims d,
                  FastDiv parts,
                  FastDiv tokens) {
    const int tid = threadIdx.x;
    uint32_t part, t_of_rank;
    const int token = parts.quotient(blockIdx.x, part), r = tokens.quotient(token, t_of_rank), t = t_of_rank;
    const size_t tok = static_cast<size_t>(r) * d.T + t;
    const int col = part * blockDim.x + tid;
    const bool active = col < d.H / 8;
    const bool weights = part == 0 && tid < d.K;
    uint4 b0 = make_uint4(0, 0, 0, 0), b1 = b0;
    if (active) {
        if (bias0) b0 = ld16_nt(reinterpret_cast<const uint4 *>(bias0 + tok * d.H) + col);
        if (bias1) b1 = ld16_nt(reinterpret_cast<const uint4 *>(bias1 + tok * d.H) + col);
    }
    float acc[8];
    {
        const uint32_t u0[4] = {b0.x, b0.y, b0.z, b0.w}, u1[4] = {b1.x, b1.y, b1.z, b1.w};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            acc[2 * c] = bf16_lo_to_f32(u0[c]) + bf16_lo_to_f32(u1[c]);
            acc[2 * c + 1] = bf16_hi_to_f32(u0[c]) + bf16_hi_to_f32(u1[c]);
        }
    }
    float wsum = 0.f;
    for (int d0 = 0; d0 < d.R; d0 += kWaveSize) {
        const WaveRows w = wave_rows<EAGER>(in_rank, prefix, send_head, row_offset, d, r, t, d0);
        for (unsigned long long hits = w.hits; hits;) {
            // all loads of the batch first, then the additions in ascending rank order
            const int n = __popcll(hits);
            uint4 v[kHtBatch];
            float wv[kHtBatch];
#pragma unroll
            for (int j = 0; j < kHtBatch; ++j) {
                v[j] = make_uint4(0, 0, 0, 0);
                wv[j] = 0.f;
                if (j < n) {
                    const long long row = next_row(w, hits);
                    if (active) v[j] = ld16_nt(reinterpret_cast<const uint4 *>(x + static_cast<size_t>(row) * d.H) + col);
                    if (topk_weights && weights) wv[j] = topk_weights[row * d.K + tid];
                }
            }
#pragma unroll
            for (int j = 0; j < kHtBatch; ++j) {
                if (j >= n) continue;
                const uint32_t u[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    acc[2 * c] += bf16_lo_to_f32(u[c]);
                    acc[2 * c + 1] += bf16_hi_to_f32(u[c]);
                }
                wsum += wv[j];
            }
        }
    }
    if (active) {
        uint4 out;
        out.x = f32_to_bf16_pair(acc[0], acc[1]);
        out.y = f32_to_bf16_pair(acc[2], acc[3]);
        out.z = f32_to_bf16_pair(acc[4], acc[5]);
        out.w = f32_to_bf16_pair(acc[6], acc[7]);
        st16_nt(reinterpret_cast<uint4 *>(combined + tok * d.H) + col, out);
    }
    if (combined_w && weights) combined_w[tok * d.K + tid] = wsum;
}

// ---- router -----------------------------------------------------------------------------------------
// One wave per token; lane l holds experts l, l + 64, ...  K rounds of a wave-wide argmax
// (larger value wins, equal values go to the lower expert index).  The two reductions of a
// round (maximum of the values, then lowest index among the lanes that hold it) run on
// the DPP data path: four steps inside the rows of 16 lanes, two row broadcasts, result in
// lane 63.  Cross-lane permutes through LDS took three times as long.
constexpr int kRouterMaxPerLane = 16; // E <= 1024

// PL = experts a lane holds (a power of two >= ceil(E / 64)): the argmax rounds only walk
// the slots that exist.
template<int PL>
__global__ void __launch_bounds__(256)
router_kernel(const float *__restrict__ logits, int32_t *__restrict__ topk_idx, float *__restrict__ topk_w, int n_tokens, int E, int K) {
    const int lane = threadIdx.x & (kWaveSize - 1);
    const int token = blockIdx.x * (blockDim.x / kWaveSize) + threadIdx.x / kWaveSize;
    if (token >= n_tokens) return; // whole waves leave together: the DPP steps below see full waves
    float v[PL];
    unsigned taken = 0;
#pragma unroll
    for (int j = 0; j < PL; ++j) {
        const int e = j * kWaveSize + lane;
        v[j] = e < E ? logits[static_cast<size_t>(token) * E + e] : 0.f;
        if (e >= E) taken |= 1u << j;
    }
    float mine = 0.f, first = 0.f; // lane k keeps the k-th selected logit
    int mine_i = 0;
    for (int k = 0; k < K; ++k) {
        float top;
        int win;
        router_round<PL>(v, taken, lane, top, win);
        if (k == 0) first = top;
        if (lane == k) {
            mine = top;
            mine_i = win;
        }
    }
    // softmax over the K selected logits; every lane adds them up in selection order
    const float ex = lane < K ? expf(mine - first) : 0.f;
    float sum = 0.f;
    for (int k = 0; k < K; ++k)
        sum += __shfl(ex, k);
    if (lane < K) {
        topk_idx[static_cast<size_t>(token) * K + lane] = mine_i;
        topk_w[static_cast<size_t>(token) * K + lane] = ex / sum;
    }
}

int
round_up_wave(int n) {
    return (n + kWaveSize - 1) / kWaveSize * kWaveSize;
}

int
check_ht(const char *who, int T, int H, int K, int R, int E) {
    auto bad = [&](const std::string &why) { return nixl_amd_fail(NIXL_AMD_ERR_INVALID, std::string(who) + ": " + why); };
    if (R <= 0 || R > 1024) return bad("num_ranks must be in [1, 1024]");
    if (E <= 0 || E % R != 0) return bad("num_experts must be a positive multiple of num_ranks");
    if (T <= 0) return bad("num_tokens must be positive");
    if (K < 0 || K > 16) return bad("num_topk must be at most 16");
    if (H % 8 != 0 || H < 0 || H > 8192) return bad("hidden must be a multiple of 8, at most 8192");
    if (static_cast<long long>(R) * T > (1ll << 30)) return bad("num_ranks * num_tokens too large");
    return NIXL_AMD_OK;
}

} // namespace

extern "C" {

int
nixl_amd_ep_get_dispatch_layout(const int32_t *topk_idx,
                                int *num_tokens_per_rank,
                                int *num_tokens_per_expert,
                                uint8_t *is_token_in_rank,
                                int num_tokens,
                                int num_topk,
                                int num_ranks,
                                int num_experts,
                                void *stream) {
    const int rc = check_ht("get_dispatch_layout", num_tokens, 0, num_topk, num_ranks, num_experts);
    if (rc) return rc;
    if (!topk_idx || !num_tokens_per_rank || !num_tokens_per_expert || !is_token_in_rank)
        return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "get_dispatch_layout: null pointer argument");
    const size_t lds = static_cast<size_t>(num_experts + num_ranks) * sizeof(int);
    if (lds > 48 * 1024) return nixl_amd_fail(NIXL_AMD_ERR_TOO_LARGE, "get_dispatch_layout: too many experts");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool flags_fit = num_tokens <= kLayoutTokens || num_ranks >= kLayoutWholeRanks ||
                           static_cast<long long>(num_tokens) * num_ranks <= kLayoutWholeFlags;
    if (num_tokens <= kLayoutWhole && num_tokens * num_topk <= kLayoutWholeSelections && flags_fit) {
        hipLaunchKernelGGL(layout_kernel, dim3(static_cast<unsigned>(num_ranks)), dim3(round_up_wave(num_tokens)), lds, s, topk_idx,
                           num_tokens_per_rank, num_tokens_per_expert, is_token_in_rank, num_tokens, num_topk, num_ranks,
                           num_experts, FastDiv(1), FastDiv(num_experts / num_ranks));
        HIP_TRY(hipGetLastError());
        return NIXL_AMD_OK;
    }
    // the counts are accumulated with atomics; cleared by a kernel, not a memset, so that a
    // caller may capture the call into a graph
    const size_t n_rank = static_cast<size_t>(num_ranks) * num_ranks, n_expert = static_cast<size_t>(num_ranks) * num_experts;
    hipLaunchKernelGGL(zero_ints_kernel, dim3(static_cast<unsigned>((std::max(n_rank, n_expert) + 255) / 256)), dim3(256), 0, s,
                       num_tokens_per_rank, n_rank, num_tokens_per_expert, n_expert);
    HIP_TRY(hipGetLastError());
    const long long chunks = (num_tokens + kLayoutTokens - 1) / kLayoutTokens;
    hipLaunchKernelGGL(layout_kernel, dim3(static_cast<unsigned>(num_ranks * chunks)), dim3(kLayoutTokens), lds, s, topk_idx,
                       num_tokens_per_rank, num_tokens_per_expert, is_token_in_rank, num_tokens, num_topk, num_ranks,
                       num_experts, FastDiv(static_cast<uint32_t>(chunks)), FastDiv(num_experts / num_ranks));
    HIP_TRY(hipGetLastError());
    return NIXL_AMD_OK;
}

int
nixl_amd_ep_ht_notify_dispatch(const uint8_t *is_token_in_rank,
                               const int *num_tokens_per_expert,
                               int *recv_gbl_rank_prefix_sum,
                               int *recv_expert_count,
                               int *gbl_channel_prefix_matrix,
                               int *send_head,
                               int64_t *recv_row_offset,
                               int *recv_counter,
                               int num_tokens,
                               int num_ranks,
                               int num_experts,
                               int num_channels,
                               int expert_alignment,
                               void *stream) {
    const int rc = check_ht("ht_notify_dispatch", num_tokens, 0, 0, num_ranks, num_experts);
    if (rc) return rc;
    if (num_channels <= 0 || expert_alignment <= 0)
        return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "ht_notify_dispatch: num_channels and expert_alignment must be positive");
    if (!is_token_in_rank || !num_tokens_per_expert || !recv_gbl_rank_prefix_sum || !recv_expert_count ||
        !gbl_channel_prefix_matrix || !send_head)
        return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "ht_notify_dispatch: null pointer argument");
    hipStream_t s = static_cast<hipStream_t>(stream);
    // the packed kernel reads 8 flag bytes and writes 16-byte pieces at a time
    const bool aligned = reinterpret_cast<uintptr_t>(is_token_in_rank) % 8 == 0 && reinterpret_cast<uintptr_t>(send_head) % 16 == 0;
    const HtNotifyOut notify{num_tokens_per_expert, recv_gbl_rank_prefix_sum, recv_expert_count,
                             reinterpret_cast<long long *>(recv_row_offset), recv_counter, expert_alignment};
    if (num_ranks <= kPackedScanRanks && num_tokens <= kPackedScanMaxTokens && aligned) {
        const long long tokens = static_cast<long long>(num_ranks) * num_tokens;
        const bool one_launch = num_ranks == 8 ? tokens <= kNotifyTokensOf8 :
            num_ranks == 4                     ? tokens <= kNotifyTokensOf4 :
                                                 tokens * num_ranks <= kNotifyFlags;
        hipLaunchKernelGGL(one_launch ? ht_scan_packed_kernel<true> : ht_scan_packed_kernel<false>,
                           dim3(static_cast<unsigned>(num_ranks) * ((num_tokens + kScanThreads - 1) / kScanThreads) + one_launch),
                           dim3(kScanThreads), 0, s, is_token_in_rank, send_head, gbl_channel_prefix_matrix, num_tokens, num_ranks,
                           num_channels, num_experts, notify);
        if (one_launch) {
            HIP_TRY(hipGetLastError());
            return NIXL_AMD_OK;
        }
    } else {
        hipLaunchKernelGGL(ht_scan_kernel, dim3(static_cast<unsigned>(num_ranks) * num_ranks), dim3(kScanThreads), 0, s,
                           is_token_in_rank, send_head, gbl_channel_prefix_matrix, num_tokens, num_ranks, num_channels);
    }
    HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(ht_prefix_kernel, dim3(1), dim3(kScanThreads), 0, s, gbl_channel_prefix_matrix, notify, num_ranks, num_experts,
                       num_channels);
    HIP_TRY(hipGetLastError());
    return NIXL_AMD_OK;
}

int
nixl_amd_ep_ht_dispatch_scaled(void *recv_x,
                               void *recv_x_scales,
                               int32_t *recv_topk_idx,
                               float *recv_topk_weights,
                               int32_t *recv_src_meta,
                               const void *x,
                               const void *x_scales,
                               const int32_t *topk_idx,
                               const float *topk_weights,
                               const uint8_t *is_token_in_rank,
                               const int *recv_gbl_rank_prefix_sum,
                               const int *send_head,
                               const int64_t *recv_row_offset,
                               int num_tokens,
                               int hidden,
                               int elem_bytes,
                               int num_scales,
                               int64_t scale_rank_stride,
                               int64_t scale_token_stride,
                               int64_t scale_hidden_stride,
                               int num_topk,
                               int num_ranks,
                               int num_experts,
                               void *stream) {
    if (elem_bytes != 1 && elem_bytes != 2 && elem_bytes != 4)
        return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "ht_dispatch: elem_bytes must be 1, 2 or 4");
    if (hidden <= 0) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "ht_dispatch: hidden must be positive");
    if ((static_cast<long long>(hidden) * elem_bytes) % 16 != 0)
        return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "ht_dispatch: a row must be a multiple of 16 bytes");
    // the row kernels count a row in 2-byte elements, whatever it holds
    const long long row_halves = static_cast<long long>(hidden) * elem_bytes / 2;
    if (row_halves > 8192) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "ht_dispatch: a row may hold at most 16 KiB");
    const int rc = check_ht("ht_dispatch", num_tokens, static_cast<int>(row_halves), num_topk, num_ranks, num_experts);
    if (rc) return rc;
    if (!recv_x || !x || !is_token_in_rank || !recv_gbl_rank_prefix_sum || !send_head || !recv_row_offset)
        return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "ht_dispatch: null pointer argument");
    if (recv_topk_idx && !topk_idx) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "ht_dispatch: recv_topk_idx without topk_idx");
    if (num_scales < 0 || num_scales > 4096) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "ht_dispatch: num_scales must be in [0, 4096]");
    if ((x_scales != nullptr) != (recv_x_scales != nullptr) || (x_scales && num_scales == 0))
        return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "ht_dispatch: x_scales, recv_x_scales and num_scales go together");
    if (x_scales && (scale_rank_stride < 0 || scale_token_stride < 0 || scale_hidden_stride < 0))
        return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "ht_dispatch: negative scale stride");
    const HtDims d{num_ranks, num_tokens, static_cast<int>(row_halves), num_topk, num_experts};
    const int parts = round_up_wave(d.H / 8) / kWaveSize;
    if (static_cast<long long>(num_ranks) * num_tokens * parts >= (1ll << 31))
        return nixl_amd_fail(NIXL_AMD_ERR_TOO_LARGE, "ht_dispatch: too many tokens");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const long long scale_blocks =
        x_scales ? static_cast<long long>(num_ranks) * num_ranks * ((num_tokens + kHtScaleTokens - 1) / kHtScaleTokens) : 0;
    const long long meta_blocks = recv_topk_idx || recv_src_meta ?
        static_cast<long long>(num_ranks) * num_ranks * ((num_tokens + kHtMetaThreads - 1) / kHtMetaThreads) : 0;
    if (scale_blocks >= (1ll << 31) || meta_blocks >= (1ll << 31))
        return nixl_amd_fail(NIXL_AMD_ERR_TOO_LARGE, "ht_dispatch: too many ranks and tokens");
    const long long *offsets = reinterpret_cast<const long long *>(recv_row_offset);
    const int *prefix = recv_gbl_rank_prefix_sum;
    const HtRows rows{static_cast<uint16_t *>(recv_x), static_cast<const uint16_t *>(x), is_token_in_rank, prefix, send_head, offsets, d,
                      FastDiv(parts), FastDiv(num_tokens), static_cast<long long>(num_ranks) * num_tokens * d.H * 2 > kHtStreamFrom};
    const HtMeta meta{recv_topk_idx, recv_topk_weights, recv_src_meta, topk_idx, topk_weights};
    const HtScales sc{static_cast<uint32_t *>(recv_x_scales), static_cast<const uint32_t *>(x_scales), num_scales,
                      num_scales % 4 == 0 && reinterpret_cast<uintptr_t>(recv_x_scales) % 16 == 0, scale_rank_stride,
                      scale_token_stride, scale_hidden_stride};
    const uintptr_t bits = reinterpret_cast<uintptr_t>(recv_topk_idx) | reinterpret_cast<uintptr_t>(recv_topk_weights) |
                           reinterpret_cast<uintptr_t>(recv_src_meta) | reinterpret_cast<uintptr_t>(topk_idx) |
                           reinterpret_cast<uintptr_t>(topk_weights);
    const bool vec = num_topk % 4 == 0 && bits % 16 == 0;
    const long long pieces = static_cast<long long>(num_ranks) * num_tokens * parts;
    const long long row_blocks = (pieces + kHtWaves - 1) / kHtWaves;
    const auto kernel = x_scales ? (vec ? ht_dispatch_kernel<true, true, false> : ht_dispatch_kernel<false, true, false>) :
        rows.streamed            ? (vec ? ht_dispatch_kernel<true, false, true> : ht_dispatch_kernel<false, false, true>) :
                                   (vec ? ht_dispatch_kernel<true, false, false> : ht_dispatch_kernel<false, false, false>);
    const auto launch = [&](long long n_scale, long long n_meta, long long n_row, long long first) -> int {
        const long long blocks = n_scale + n_meta + n_row;
        if (blocks == 0) return NIXL_AMD_OK;
        hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks)), dim3(kHtThreads), 0, s, rows, meta, sc,
                           static_cast<uint32_t>(n_scale), static_cast<uint32_t>(n_meta), static_cast<uint32_t>(first));
        HIP_TRY(hipGetLastError());
        return NIXL_AMD_OK;
    };
    const bool meta_apart = num_ranks >= kHtMetaApartRanks;
    const long long with_rows = meta_apart ? 0 : meta_blocks;
    if (scale_blocks + with_rows + row_blocks <= kHtMaxGrid) {
        if (const int status = launch(scale_blocks, with_rows, row_blocks, 0)) return status;
    } else {
        const long long part_blocks[3] = {row_blocks, scale_blocks, with_rows};
        for (int part = 0; part < 3; ++part)
            for (long long at = 0; at < part_blocks[part]; at += kHtMaxGrid) {
                const long long n = std::min(kHtMaxGrid, part_blocks[part] - at);
                if (const int status = launch(part == 1 ? n : 0, part == 2 ? n : 0, part == 0 ? n : 0, at)) return status;
            }
    }
    for (long long at = 0; at < meta_blocks - with_rows; at += kHtMaxGrid) {
        hipLaunchKernelGGL(vec ? ht_meta_kernel<true> : ht_meta_kernel<false>,
                           dim3(static_cast<unsigned>(std::min(kHtMaxGrid, meta_blocks - at))), dim3(kHtMetaThreads), 0, s, meta,
                           is_token_in_rank, prefix, send_head, offsets, d, static_cast<uint32_t>(at));
        HIP_TRY(hipGetLastError());
    }
    return NIXL_AMD_OK;
}

int
nixl_amd_ep_ht_dispatch_rows(void *recv_x,
                             void *recv_x_scales,
                             int32_t *recv_topk_idx,
                             float *recv_topk_weights,
                             int32_t *recv_src_meta,
                             const void *x,
                             const void *x_scales,
                             const int32_t *topk_idx,
                             const float *topk_weights,
                             const uint8_t *is_token_in_rank,
                             const int *recv_gbl_rank_prefix_sum,
                             const int *send_head,
                             const int64_t *recv_row_offset,
                             int64_t /*num_rows*/,
                             int num_tokens,
                             int hidden,
                             int elem_bytes,
                             int num_scales,
                             int64_t scale_rank_stride,
                             int64_t scale_token_stride,
                             int64_t scale_hidden_stride,
                             int num_topk,
                             int num_ranks,
                             int num_experts,
                             void *stream) {
    return nixl_amd_ep_ht_dispatch_scaled(recv_x, recv_x_scales, recv_topk_idx, recv_topk_weights, recv_src_meta, x, x_scales,
                                          topk_idx, topk_weights, is_token_in_rank, recv_gbl_rank_prefix_sum, send_head,
                                          recv_row_offset, num_tokens, hidden, elem_bytes, num_scales, scale_rank_stride,
                                          scale_token_stride, scale_hidden_stride, num_topk, num_ranks, num_experts, stream);
}

int
nixl_amd_ep_ht_dispatch(void *recv_x,
                        int32_t *recv_topk_idx,
                        float *recv_topk_weights,
                        int32_t *recv_src_meta,
                        const void *x,
                        const int32_t *topk_idx,
                        const float *topk_weights,
                        const uint8_t *is_token_in_rank,
                        const int *recv_gbl_rank_prefix_sum,
                        const int *send_head,
                        const int64_t *recv_row_offset,
                        int num_tokens,
                        int hidden,
                        int num_topk,
                        int num_ranks,
                        int num_experts,
                        void *stream) {
    return nixl_amd_ep_ht_dispatch_scaled(recv_x, nullptr, recv_topk_idx, recv_topk_weights, recv_src_meta, x, nullptr, topk_idx,
                                          topk_weights, is_token_in_rank, recv_gbl_rank_prefix_sum, send_head, recv_row_offset,
                                          num_tokens, hidden, 2, 0, 0, 0, 0, num_topk, num_ranks, num_experts, stream);
}

int
nixl_amd_ep_ht_combine_rows(void *combined_x,
                            float *combined_topk_weights,
                            const void *x,
                            const float *topk_weights,
                            const void *bias_0,
                            const void *bias_1,
                            const uint8_t *is_token_in_rank,
                            const int *recv_gbl_rank_prefix_sum,
                            const int *send_head,
                            const int64_t *recv_row_offset,
                            int64_t num_rows,
                            int num_tokens,
                            int hidden,
                            int num_topk,
                            int num_ranks,
                            void *stream) {
    const int rc = check_ht("ht_combine", num_tokens, hidden, num_topk, num_ranks, num_ranks);
    if (rc) return rc;
    if (hidden == 0) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "ht_combine: hidden must be positive");
    if (!combined_x || !x || !is_token_in_rank || !recv_gbl_rank_prefix_sum || !send_head || !recv_row_offset)
        return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "ht_combine: null pointer argument");
    const HtDims d{num_ranks, num_tokens, hidden, num_topk, num_ranks};
    const long long tokens = static_cast<long long>(num_ranks) * num_tokens;
    const bool large = tokens * hidden > kHtCombineEager;
    const int row_lanes = round_up_wave(hidden / 8);
    const bool whole_wgs = row_lanes % kHtCombineEagerLanes == 0;
    const bool many_ranks = num_ranks >= (large ? kHtCombineManyRanks : kHtCombineManyRanksSmall);
    const bool eager = !large || (num_rows >= 0 && num_rows <= (many_ranks ? kHtCombineFewRows : kHtCombineManyRows) * tokens &&
                                  num_ranks <= (whole_wgs ? kHtCombineMostRanksShared : kHtCombineMostRanks));
    const bool four_waves = !large && many_ranks ?
        whole_wgs || (num_ranks > kHtCombineMostRanksShared && row_lanes > kHtCombineLongRow) :
        eager && whole_wgs && num_rows <= (large ? kHtCombineFewRows : kHtCombineManyRows) * tokens;
    const int most = four_waves ? kHtCombineEagerLanes : kWaveSize;
    const int parts = (row_lanes + most - 1) / most, lanes = round_up_wave((row_lanes + parts - 1) / parts);
    if (static_cast<long long>(num_ranks) * num_tokens * parts >= (1ll << 31))
        return nixl_amd_fail(NIXL_AMD_ERR_TOO_LARGE, "ht_combine: too many tokens");
    hipLaunchKernelGGL(eager ? ht_combine_kernel<true> : ht_combine_kernel<false>,
                       dim3(static_cast<unsigned>(num_ranks) * num_tokens * parts), dim3(lanes), 0, static_cast<hipStream_t>(stream), static_cast<uint16_t *>(combined_x), combined_topk_weights,
                       static_cast<const uint16_t *>(x), topk_weights, static_cast<const uint16_t *>(bias_0),
                       static_cast<const uint16_t *>(bias_1), is_token_in_rank, recv_gbl_rank_prefix_sum, send_head,
                       reinterpret_cast<const long long *>(recv_row_offset), d, FastDiv(parts), FastDiv(num_tokens));
    HIP_TRY(hipGetLastError());
    return NIXL_AMD_OK;
}

int
nixl_amd_ep_ht_combine(void *combined_x,
                       float *combined_topk_weights,
                       const void *x,
                       const float *topk_weights,
                       const void *bias_0,
                       const void *bias_1,
                       const uint8_t *is_token_in_rank,
                       const int *recv_gbl_rank_prefix_sum,
                       const int *send_head,
                       const int64_t *recv_row_offset,
                       int num_tokens,
                       int hidden,
                       int num_topk,
                       int num_ranks,
                       void *stream) {
    return nixl_amd_ep_ht_combine_rows(combined_x, combined_topk_weights, x, topk_weights, bias_0, bias_1, is_token_in_rank,
                                       recv_gbl_rank_prefix_sum, send_head, recv_row_offset, -1, num_tokens, hidden, num_topk,
                                       num_ranks, stream);
}

int
nixl_amd_ep_router_topk(const float *logits,
                        int32_t *topk_idx,
                        float *topk_weights,
                        int num_tokens,
                        int num_experts,
                        int num_topk,
                        void *stream) {
    if (!logits || !topk_idx || !topk_weights) return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "router_topk: null pointer argument");
    if (num_tokens < 0 || num_experts <= 0 || num_experts > kRouterMaxPerLane * kWaveSize)
        return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "router_topk: num_experts must be in [1, 1024]");
    if (num_topk <= 0 || num_topk > 16 || num_topk > num_experts)
        return nixl_amd_fail(NIXL_AMD_ERR_INVALID, "router_topk: num_topk must be in [1, min(16, num_experts)]");
    if (num_tokens == 0) return NIXL_AMD_OK;
    const dim3 grid((num_tokens + 3) / 4), block(256);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int per_lane = (num_experts + kWaveSize - 1) / kWaveSize;
    if (per_lane <= 1)
        hipLaunchKernelGGL(router_kernel<1>, grid, block, 0, s, logits, topk_idx, topk_weights, num_tokens, num_experts, num_topk);
    else if (per_lane <= 2)
        hipLaunchKernelGGL(router_kernel<2>, grid, block, 0, s, logits, topk_idx, topk_weights, num_tokens, num_experts, num_topk);
    else if (per_lane <= 4)
        hipLaunchKernelGGL(router_kernel<4>, grid, block, 0, s, logits, topk_idx, topk_weights, num_tokens, num_experts, num_topk);
    else if (per_lane <= 8)
        hipLaunchKernelGGL(router_kernel<8>, grid, block, 0, s, logits, topk_idx, topk_weights, num_tokens, num_experts, num_topk);
    else
        hipLaunchKernelGGL(router_kernel<16>, grid, block, 0, s, logits, topk_idx, topk_weights, num_tokens, num_experts, num_topk);
    HIP_TRY(hipGetLastError());
    return NIXL_AMD_OK;
}

} // extern "C"
