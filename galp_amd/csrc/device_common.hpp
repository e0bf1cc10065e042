// device_common.hpp -- wave64 helpers shared by the gfx950 LP kernels.
//
// Everything here is written for CDNA wavefronts of 64 lanes: 64-bit ballot
// masks, lane-index shuffles and reductions across full waves or aligned
// power-of-two lane groups.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace galp {

constexpr int kWave = 64;
constexpr uint32_t kEmpty = 0xffffffffu;   // labels are vertex ids < 2^31

// Fibonacci (multiplicative) hashing into a power-of-two table of 2^bits
// slots (Knuth, TAOCP vol. 3, 6.4).  Labels are arbitrary vertex ids, and the
// top bits of the product spread consecutive ids across the table.
__device__ __forceinline__ uint32_t hash_slot(uint32_t key, int bits) {
    return (key * 0x9E3779B1u) >> (32 - bits);
}

// Label partition of a hub's label (P partitions): a multiplicative hash
// scaled to [0, P), so a hub's distinct labels spread evenly over its
// partitions whatever their values.  Both methods' hub paths use it.
__device__ __forceinline__ uint32_t hub_partition(uint32_t L, uint32_t P) {
    return (uint32_t)(((unsigned long long)(L * 0x85EBCA77u) * P) >> 32);
}

// Round of a label when one hub partition is merged in R rounds (R a power
// of two, at most 4096): bits of a third multiplicative hash, so labels
// that share a partition spread over the rounds.
__device__ __forceinline__ uint32_t sub_round(uint32_t L, uint32_t R) {
    return ((L * 0xC2B2AE3Du) >> 20) & (R - 1u);
}

__device__ __forceinline__ int lane_id() { return (int)(threadIdx.x & (kWave - 1)); }

// ---------------------------------------------------------------------------
// Lane moves inside aligned power-of-two lane groups.  Within a DPP row (16
// lanes) they are VALU data-parallel-primitive moves, not LDS permutes:
//   quad_perm [1,0,3,2], [2,3,0,1], [3,2,1,0]: lane i <- i ^ 1, i ^ 2, i ^ 3;
//   row_half_mirror: i <- i ^ 7 (8-lane halves); row_mirror: i <- i ^ 15.
// Lane i ^ 16 comes from ds_swizzle (bit mode: and 31, or 0, xor 16), which
// needs no address register; lane i ^ 32 from a permute.  All lanes of the
// wave must be active (DPP reads the source lane's register).
constexpr int kDppQuadXor1 = 0xB1;
constexpr int kDppQuadXor2 = 0x4E;
constexpr int kDppQuadXor3 = 0x1B;
constexpr int kDppRowMirror = 0x140;
constexpr int kDppRowHalfMirror = 0x141;
constexpr int kSwizzleXor16 = 0x401F;

template <int CTRL>
__device__ __forceinline__ int32_t dpp_mov(int32_t x) {
    return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xF, 0xF, false);
}

// x of lane (lane ^ J), J a power of two below 64.
template <int J>
__device__ __forceinline__ int32_t lane_xor(int32_t x) {
    if constexpr (J == 1) return dpp_mov<kDppQuadXor1>(x);
    else if constexpr (J == 2) return dpp_mov<kDppQuadXor2>(x);
    else if constexpr (J == 4) return dpp_mov<kDppQuadXor3>(dpp_mov<kDppRowHalfMirror>(x));   // ^7 then ^3
    else if constexpr (J == 8) return dpp_mov<kDppRowHalfMirror>(dpp_mov<kDppRowMirror>(x));  // ^15 then ^7
    else if constexpr (J == 16) return __builtin_amdgcn_ds_swizzle(x, kSwizzleXor16);
    else return __shfl_xor(x, J);
}

// Max over an aligned group of G lanes (G a power of two, G <= 64).
template <int G, typename T>
__device__ __forceinline__ T group_max(T x) {
    if constexpr (sizeof(T) == 4) {   // butterfly of lane moves
        auto step = [&](int32_t y) {
            const T o = (T)y;
            x = x > o ? x : o;
        };
        if constexpr (G >= 64) step(lane_xor<32>((int32_t)x));
        if constexpr (G >= 32) step(lane_xor<16>((int32_t)x));
        if constexpr (G >= 16) step(lane_xor<8>((int32_t)x));
        if constexpr (G >= 8) step(lane_xor<4>((int32_t)x));
        if constexpr (G >= 4) step(lane_xor<2>((int32_t)x));
        if constexpr (G >= 2) step(lane_xor<1>((int32_t)x));
        return x;
    } else {
#pragma unroll
        for (int s = G / 2; s > 0; s >>= 1) {
            T y = __shfl_xor(x, s, G);
            x = x > y ? x : y;
        }
        return x;
    }
}

// Min over an aligned group of G <= 32 lanes.
template <int G>
__device__ __forceinline__ int32_t group_min(int32_t x) {
    if constexpr (G >= 32) x = min(x, lane_xor<16>(x));
    if constexpr (G >= 16) x = min(x, lane_xor<8>(x));
    if constexpr (G >= 8) x = min(x, lane_xor<4>(x));
    if constexpr (G >= 4) x = min(x, lane_xor<2>(x));
    if constexpr (G >= 2) x = min(x, lane_xor<1>(x));
    return x;
}

// Lanes i ^ k, k < K (K = 1, 2, 4, 8, 16 within a row), whose y equals x.
template <int K>
__device__ __forceinline__ uint32_t count_eq_row(int32_t x, int32_t y) {
    uint32_t c = (uint32_t)(y == x);
    if constexpr (K >= 2) c += (uint32_t)(dpp_mov<kDppQuadXor1>(y) == x);
    if constexpr (K >= 4) {
        c += (uint32_t)(dpp_mov<kDppQuadXor2>(y) == x);
        c += (uint32_t)(dpp_mov<kDppQuadXor3>(y) == x);
    }
    if constexpr (K >= 8) c += count_eq_row<4>(x, dpp_mov<kDppRowHalfMirror>(y));   // k = 7, 6, 5, 4
    if constexpr (K >= 16) c += count_eq_row<8>(x, dpp_mov<kDppRowMirror>(y));      // k = 15 .. 8
    return c;
}

// Lanes of this lane's aligned group of G <= 32 (itself included) whose x
// equals this lane's.
template <int G>
__device__ __forceinline__ uint32_t group_count_eq(int32_t x) {
    uint32_t c = count_eq_row<(G < 16 ? G : 16)>(x, x);
    if constexpr (G >= 32) c += count_eq_row<16>(x, lane_xor<16>(x));
    return c;
}

// Wave-wide reduction of 32-bit words for an operation with identity 0 (max
// of unsigned, or); uniform result.  Row shifts and row broadcasts fold into
// the operation's own instruction, one per step, where a butterfly needs a
// move or two besides.
template <class Op>
__device__ __forceinline__ uint32_t wave_reduce_u32(uint32_t x, Op op) {
    auto step = [&](auto ctrl, auto rows) {
        x = op(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int32_t)x, decltype(ctrl)::value, decltype(rows)::value,
                                                        0xF, false));
    };
    using all = std::integral_constant<int, 0xF>;
    step(std::integral_constant<int, 0x111>{}, all{});   // row_shr 1, 2, 4, 8: a row's lane 15 holds its total
    step(std::integral_constant<int, 0x112>{}, all{});
    step(std::integral_constant<int, 0x114>{}, all{});
    step(std::integral_constant<int, 0x118>{}, all{});
    step(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xA>{});   // row_bcast 15 into rows 1, 3
    step(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xC>{});   // row_bcast 31 into rows 2, 3
    return (uint32_t)__builtin_amdgcn_readlane((int32_t)x, kWave - 1);
}
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t x) {
    return wave_reduce_u32(x, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
}

// Lanes of `among` (a wave mask that holds this lane) whose x equals this
// lane's; meaningless in other lanes.  The mask is split by one ballot per
// bit, four vector instructions a bit and hardly a scalar one, skipping the
// groups of four bits in which the lanes of `among` agree: about 80 for
// 20-bit labels, where comparing against every lane's value in turn takes
// 192.  With it (and unproductive peel rounds cut short) the 33..64 class,
// which issue of these instructions bounds while labels are diverse, took a
// 512-graph batch's run from 14.8 to 11.2 ms.
__device__ __forceinline__ unsigned long long match_lanes(int32_t x, unsigned long long among) {
    const int32_t first = __builtin_amdgcn_readlane(x, __ffsll((long long)among) - 1);
    const bool in = (among >> lane_id()) & 1ull;
    const uint32_t vary =
        wave_reduce_u32(in ? (uint32_t)(x ^ first) : 0u, [](uint32_t a, uint32_t b) { return a | b; });
    uint32_t lo = (uint32_t)among, hi = (uint32_t)(among >> 32);
#pragma unroll
    for (int nib = 0; nib < 8; ++nib) {
        if (!((vary >> (4 * nib)) & 15u)) continue;   // uniform
#pragma unroll
        for (int bit = 4 * nib; bit < 4 * nib + 4; ++bit) {
            uint32_t m = (uint32_t)__builtin_amdgcn_sbfe(x, bit, 1);   // the bit in every position
            asm("" : "+v"(m));   // else the compare is rebuilt from a shift of x, one instruction more
            const unsigned long long b = __builtin_amdgcn_ballot_w64(m != 0u);
            constexpr int kAndNotXor = 0x90;   // lo & ~(b ^ m)
            lo = __builtin_amdgcn_bitop3_b32(lo, (uint32_t)b, m, kAndNotXor);
            hi = __builtin_amdgcn_bitop3_b32(hi, (uint32_t)(b >> 32), m, kAndNotXor);
        }
    }
    return ((unsigned long long)hi << 32) | lo;
}

template <typename T>
__device__ __forceinline__ T wave_max(T x) { return group_max<kWave, T>(x); }

__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t x) {
#pragma unroll
    for (int s = kWave / 2; s > 0; s >>= 1) x += __shfl_xor(x, s, kWave);
    return x;
}

// Block-wide max over NW waves; every thread gets the result.  The wave
// count is a template argument: blockDim is read from the dispatch packet
// with a vector load, which would drain every load in flight.
// `scratch` holds NW entries.  Contains barriers when NW > 1.
template <int NW, typename T>
__device__ __forceinline__ T block_max(T x, T *scratch) {
    x = wave_max(x);
    if constexpr (NW == 1) {
        return x;
    } else {
        const int w = (int)(threadIdx.x / kWave);
        if (lane_id() == 0) scratch[w] = x;
        __syncthreads();
        T r = scratch[0];
#pragma unroll
        for (int i = 1; i < NW; ++i) r = r > scratch[i] ? r : scratch[i];
        __syncthreads();
        return r;
    }
}

// Block-wide sum over NW waves; every thread gets the result.  Contains
// barriers when NW > 1.
template <int NW>
__device__ __forceinline__ uint32_t block_sum(uint32_t x, uint32_t *scratch) {
    x = wave_sum_u32(x);
    if constexpr (NW == 1) {
        return x;
    } else {
        const int w = (int)(threadIdx.x / kWave);
        if (lane_id() == 0) scratch[w] = x;
        __syncthreads();
        uint32_t r = 0;
#pragma unroll
        for (int i = 0; i < NW; ++i) r += scratch[i];
        __syncthreads();
        return r;
    }
}

// Block-wide exclusive prefix sum of one int per thread (NW waves); `scratch`
// holds NW entries.  Contains barriers.
template <int NW>
__device__ __forceinline__ int block_exclusive_scan(int x, int *scratch) {
    const int lane = lane_id();
    const int w = (int)(threadIdx.x / kWave);
    int inc = x;
#pragma unroll
    for (int s = 1; s < kWave; s <<= 1) {
        const int y = __shfl_up(inc, s);
        if (lane >= s) inc += y;
    }
    if (lane == kWave - 1) scratch[w] = inc;
    __syncthreads();
    int before = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i)
        if (i < w) before += scratch[i];
    __syncthreads();
    return before + inc - x;
}

// The change counter is kept in kCountShards words, one 128-byte line each, and
// a block adds to the shard of its index: atomics on one word serialise at
// the L2 at about 14 ns each, so a 280 K-edge class kernel of 1716 blocks took
// 25 us, nearly all of it its atomics; with the shards its graph's ten
// iterations (PP-16K) went from 399 to 256 us, RMAT-18 from 2503 to 1966 us,
// LFR-1M from 3.67 to 2.79 ms.  The sum is taken once per iteration
// (k_iter_end).
constexpr int kCountShards = 64;
constexpr int kCountStride = 16;
__device__ __forceinline__ unsigned long long *count_shard(unsigned long long *counter) {
    return counter + (blockIdx.x & (kCountShards - 1)) * kCountStride;
}

// Adds a per-thread count into its shard of the change counter with one
// atomic per block of NW waves.
template <int NW>
__device__ __forceinline__ void block_count_add(uint32_t mine, unsigned long long *counter,
                                                uint32_t *scratch) {
    uint32_t s = wave_sum_u32(mine);
    if constexpr (NW == 1) {
        if (lane_id() == 0 && s) atomicAdd(count_shard(counter), (unsigned long long)s);
    } else {
        const int w = (int)(threadIdx.x / kWave);
        __syncthreads();
        if (lane_id() == 0) scratch[w] = s;
        __syncthreads();
        if (threadIdx.x == 0) {
            unsigned long long t = 0;
#pragma unroll
            for (int i = 0; i < NW; ++i) t += scratch[i];
            if (t) atomicAdd(count_shard(counter), t);
        }
    }
}

// The bookkeeping at an iteration's end, done by k_iter_end or by the last
// block of the iteration's last kernel (on != 0).
struct IterEnd {
    int32_t on;
    int32_t it;                 // slot of the iteration
    double thr;                 // stop at or below this many changes
    int32_t *stop;
    int32_t *iters_done;
    long long *iter_counts;
    int64_t *front;             // the frontier's control words, cleared (may be null)
    int32_t *host;              // the control words' copy in pinned host memory
};
constexpr int kEndCount = 4;    // host + kEndCount: the last change count, 64-bit
constexpr int kEndFront = 32;   // words of front

// The control words as the host reads them after a synchronisation: written
// by the iteration's end itself, so no copy is queued behind it.
__device__ __forceinline__ void publish_ctl(int32_t *host, int32_t *stop, int32_t stopped, int32_t done, long long count) {
    host[0] = stopped;
    host[1] = done;
    host[2] = __hip_atomic_load(stop + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // the error word
    *(long long *)(host + kEndCount) = count;
}

// One wave: sums the shards of the change counter and clears them, records
// the iteration and applies the stop rule.
__device__ __forceinline__ void end_iteration(unsigned long long *counter, const IterEnd &e) {
    static_assert(kCountShards == kWave && kEndFront <= kWave, "one lane per shard");
    unsigned long long *shard = counter + lane_id() * kCountStride;
    unsigned long long c = __hip_atomic_load(shard, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    shard[0] = 0ull;
    shard[1] = 0ull;   // tickets
    shard[2] = 0ull;
    if (e.front && lane_id() < kEndFront) e.front[lane_id()] = 0;
#pragma unroll
    for (int s = kWave / 2; s > 0; s >>= 1) c += __shfl_xor(c, s);
    if (lane_id()) return;
    e.iter_counts[e.it] = (long long)c;
    *e.iters_done = e.it + 1;
    const int32_t stopped = (double)c <= e.thr;
    if (stopped) *e.stop = 1;
    publish_ctl(e.host, e.stop, stopped, e.it + 1, (long long)c);
}

// Sets bits in the graph's error word (states the plan rules out: tables that
// overflow, rows of the wrong class) and waits until they are there.  The last
// block of an iteration publishes the word as soon as every block has taken
// its ticket, and a block takes it behind a barrier that all its waves reach:
// an atomic without a result could still be on its way then.
__device__ __forceinline__ void raise_err(int32_t *err, int32_t bits) {
    int32_t was = atomicOr(err, bits);
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(was)::"memory");
}

// block_count_add that ends the iteration when e.on: every block of the grid
// calls it once, and the last one to come does the bookkeeping, which saves
// the small graphs a launch per iteration (5 us between two short kernels).
// Only atomics are ordered here, and each is complete when its result is back,
// so no block fences or flushes a cache: the count goes to the block's shard,
// then a ticket to the shard's line, and the last block of each shard takes
// one of the whole grid.  Errors are set by raise_err, which waits as well.
template <int NW>
__device__ __forceinline__ void block_count_end(uint32_t mine, unsigned long long *counter, uint32_t *scratch,
                                                const IterEnd &e) {
    if (!e.on) {   // uniform
        block_count_add<NW>(mine, counter, scratch);
        return;
    }
    uint32_t s = wave_sum_u32(mine);
    const int w = (int)(threadIdx.x / kWave);
    __syncthreads();
    if (lane_id() == 0) scratch[w] = s;
    __syncthreads();
    if (w) return;
    int last = 0;
    if (lane_id() == 0) {
        unsigned long long t = 0;
#pragma unroll
        for (int i = 0; i < NW; ++i) t += scratch[i];
        unsigned long long *shard = count_shard(counter);
        unsigned long long done = atomicAdd(shard, t);
        asm volatile("s_waitcnt vmcnt(0)" : "+v"(done)::"memory");   // counted before the ticket is taken
        const uint32_t k = blockIdx.x & (kCountShards - 1);
        const uint32_t blocks = (gridDim.x - k + kCountShards - 1) / kCountShards;   // of this shard
        if (atomicAdd(shard + 1, 1ull) + 1ull == blocks) {
            const uint32_t shards = gridDim.x < (uint32_t)kCountShards ? gridDim.x : (uint32_t)kCountShards;
            last = atomicAdd(counter + 2, 1ull) + 1ull == shards;
        }
    }
    if (__builtin_amdgcn_readfirstlane(last)) end_iteration(counter, e);
}

// Loads that bypass the per-CU vector L1, for table words other workgroups
// update with device-scope atomics.
__device__ __forceinline__ uint32_t load_coherent(const uint32_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace galp
