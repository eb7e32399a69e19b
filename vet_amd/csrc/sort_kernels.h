// Per-pixel sort of the fragment lists by the 64-bit key (depth bits << 32 | point id), ascending, with the top-K cut.
//
// A wave owns up to 64 consecutive pixels of a bin, whose lists are one contiguous stretch of the fragment buffer (or of
// the bin's copy in LDS). Lists are grouped by padded power-of-two length m = 2,4,...,64 and 64/m lists are
// sorted at a time by one bitonic network held in registers (one key per lane, partner exchange by lane shuffles).
// Lists longer than 64 keep the K smallest keys with a streaming wave-wide selection, or are sorted in place in
// global memory when no cut applies.
//
// Counterpart of SegmentedSortBitonicHelper2 and its kernels (src/lib/rendering/AlphaListSort.cu:601-703): that one
// buckets lists into <=32 / <=256 / <=1024 / <=4096 with two extra passes and a device->host read of the bucket sizes,
// sorts by depth only and leaves lists beyond 4096 entries partly unsorted (:290). Here the order is total
// (depth, then point id) and exact for every length.
#pragma once
#include "common.h"

namespace vetrast
{
__device__ __forceinline__ uint64_t shfl_u64(uint64_t v, int src)
{
    const uint32_t lo = __shfl((uint32_t)v, src, kWave);
    const uint32_t hi = __shfl((uint32_t)(v >> 32), src, kWave);
    return ((uint64_t)hi << 32) | lo;
}

// Value of lane ^ M where all lanes are active: without lanes to leave out, a row permutation needs no register to start
// from (lane_xor clears one first).
template <int M>
__device__ __forceinline__ uint32_t partner(uint32_t v, int lane)
{
    if constexpr (M == 4)
        return partner<3>(partner<7>(v, lane), lane);  // 7 ^ 3
    else if constexpr (M < 16)
    {
        constexpr int ctrl = M == 1 ? 0xB1 : M == 2 ? 0x4E : M == 3 ? 0x1B : M == 7 ? 0x141 : M == 15 ? 0x140 : 0x128;
        static_assert(M == 1 || M == 2 || M == 3 || M == 7 || M == 8 || M == 15, "no row permutation for this M");
        return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, ctrl, 0xF, 0xF, false);
    }
    else
        return lane_xor<M>(v, lane);
}

// One compare-exchange stage with partner lane ^ M: lanes for which keep_max holds keep the larger key of the pair, the
// others the smaller one. All lanes must call. The networks are bound by their vector instructions, so the choice is one
// comparison whose lane mask is flipped in the scalar unit: 2 moves, a compare and 2 selects. (Written as a choice between
// other < key and other > key it took 13; sorting 64 keys 1009 against 508 cycles of a SIMD, 16 keys 494 against 244.)
template <int M>
__device__ __forceinline__ uint64_t exchange(uint64_t key, int lane, bool keep_max)
{
    const uint32_t lo    = partner<M>((uint32_t)key, lane);
    const uint32_t hi    = partner<M>((uint32_t)(key >> 32), lane);
    const uint64_t other = ((uint64_t)hi << 32) | lo;
    const bool take      = (other < key) != keep_max;  // (equal keys: either one)
    return take ? other : key;
}

template <int K2, int J>
__device__ __forceinline__ uint64_t halving_steps(uint64_t key, int lane)
{
    if constexpr (J >= 1)
    {
        key = exchange<J>(key, lane, (lane & J) != 0);
        key = halving_steps<K2, (J >> 1)>(key, lane);
    }
    return key;
}

template <int K2, int MAXK>
__device__ __forceinline__ uint64_t bitonic_stages(uint64_t key, int lane)
{
    if constexpr (K2 <= MAXK)
    {
        key = exchange<K2 - 1>(key, lane, (lane & (K2 >> 1)) != 0);  // mirror step inside every block of K2 lanes
        key = halving_steps<K2, (K2 >> 2)>(key, lane);
        key = bitonic_stages<K2 * 2, MAXK>(key, lane);
    }
    return key;
}

// Ascending bitonic sort of every aligned group of 2^LOG lanes (all-ascending form: a mirror step, then halving
// steps), LOG = 1..6.
template <int LOG>
__device__ __forceinline__ uint64_t bitonic_sort_groups(uint64_t key, int lane)
{
    return bitonic_stages<2, (1 << LOG)>(key, lane);
}

// Halving steps only: sorts a bitonic sequence held by the 64 lanes.
__device__ __forceinline__ uint64_t bitonic_merge64(uint64_t key, int lane)
{
    return halving_steps<64, 32>(key, lane);
}

// Sort `count` lists of class LOG (2^(LOG-1) < n <= 2^LOG) found in the wave; src_lane[r] is the lane that owns the r-th.
template <int LOG>
__device__ __forceinline__ void sort_class(uint64_t* fragments, const uint8_t* src_lane, int count,
                                           uint32_t off, uint32_t n, int lane, int K)
{
    constexpr int m        = 1 << LOG;
    constexpr int per_pass = kWave >> LOG;
    const int g = lane >> LOG, e = lane & (m - 1);
    for (int first = 0; first < count; first += per_pass)
    {
        const int li     = first + g;
        const bool valid = li < count;
        const int src    = valid ? src_lane[li] : 0;
        const uint32_t o = __shfl(off, src, kWave);
        uint32_t nn      = __shfl(n, src, kWave);
        if (!valid) nn = 0;
        uint64_t key = ((uint32_t)e < nn) ? fragments[o + e] : kInfKey;
        key          = bitonic_sort_groups<LOG>(key, lane);
        const uint32_t keep = (K > 0) ? min(nn, (uint32_t)K) : nn;
        if ((uint32_t)e < keep) fragments[o + e] = key;
    }
}

// K smallest keys (K <= 64) of a list longer than 64, sorted, written to its first K places. The wave keeps the K smallest
// keys seen so far, sorted, in its first lanes. Of every further 64 keys those that beat the K-th gather in the lanes behind,
// in no order; only when they do not fit there any more all 64 lanes are sorted (115 vector instructions), which leaves the K
// smallest in front. Most of a long list never beats the K-th, so that is two or three times where sorting every 64 keys in
// turn and merging them took one of each (ten million points, lists of up to a thousand cut to 16: the list-building pass went
// from 239 to 215 million vector instructions and 540 to 525 us).
__device__ __forceinline__ void select_smallest(uint64_t* list, uint32_t n, int lane, int K)
{
    uint64_t best = bitonic_sort_groups<6>(list[lane], lane);  // n > 64
    uint64_t kth  = shfl_u64(best, K - 1);
    int filled    = K;  // lanes in use
    if (lane >= K) best = kInfKey;
    for (uint32_t base = kWave; base < n; base += kWave)
    {
        const uint64_t v = (base + lane < n) ? list[base + lane] : kInfKey;
        uint64_t m       = __ballot(v < kth);
        if (m == 0ull) continue;
        if (filled + __popcll(m) > kWave && filled > K)
        {
            best   = bitonic_sort_groups<6>(best, lane);
            kth    = shfl_u64(best, K - 1);
            filled = K;
            if (lane >= K) best = kInfKey;
            m = __ballot(v < kth);
        }
        const int more = __popcll(m);
        if (filled + more > kWave)
        {
            // too many at once: 64 smallest of them and of what there is, a bitonic sequence
            const uint64_t sorted = bitonic_sort_groups<6>(v, lane);
            const uint64_t mirror = shfl_u64(sorted, kWave - 1 - lane);
            best                  = bitonic_merge64((mirror < best) ? mirror : best, lane);
            kth                   = shfl_u64(best, K - 1);
            if (lane >= K) best = kInfKey;
            continue;
        }
        // the keys that count go to the lanes from `filled` on; the others to lane 0, which does not look at what it gets
        const int below    = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        const int to       = (m >> lane) & 1ull ? (filled + below) << 2 : 0;
        const uint32_t lo  = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)(uint32_t)v);
        const uint32_t hi  = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)(uint32_t)(v >> 32));
        if (lane >= filled && lane < filled + more) best = ((uint64_t)hi << 32) | lo;
        filled += more;
    }
    if (filled > K) best = bitonic_sort_groups<6>(best, lane);
    if (lane < K) list[lane] = best;
}

// In-place bitonic sort of a list of any length in global memory by one wave; places beyond n act as +infinity and
// are never touched. Slow path: only lists longer than 64 with no usable cut come here.
__device__ __forceinline__ void sort_in_memory(uint64_t* list, uint32_t n, int lane)
{
    uint32_t m = 1;
    while (m < n) m <<= 1;
    const uint32_t half = m >> 1;
    for (uint32_t k = 2; k <= m; k <<= 1)
    {
        const uint32_t hk = k >> 1;
        for (uint32_t p = lane; p < half; p += kWave)
        {
            const uint32_t blk = p / hk, r = p % hk;
            const uint32_t i = blk * k + r, j = blk * k + (k - 1 - r);
            if (j < n)
            {
                const uint64_t a = list[i], b = list[j];
                if (b < a)
                {
                    list[i] = b;
                    list[j] = a;
                }
            }
        }
        __threadfence_block();
        for (uint32_t jj = k >> 2; jj >= 1; jj >>= 1)
        {
            for (uint32_t p = lane; p < half; p += kWave)
            {
                const uint32_t i = (p / jj) * 2 * jj + (p % jj), j = i + jj;
                if (j < n)
                {
                    const uint64_t a = list[i], b = list[j];
                    if (b < a)
                    {
                        list[i] = b;
                        list[j] = a;
                    }
                }
            }
            __threadfence_block();
        }
    }
}

// Sorts a list of 64 < n <= 64 * CH keys by one wave with the keys in registers, CH keys per lane (chunk q holds places
// 64 q .. 64 q + 63; places beyond n act as +infinity). Every chunk is sorted by the 64-lane network, then chunks are
// merged pairwise, level by level, in the all-ascending form of the bitonic network: the mirror step and the halving
// steps over 64 or more places pair whole chunks register against register (the mirror step with the partner chunk
// reversed across the wave), the last six halving steps of a level run inside every chunk. One load and one store per key.
template <int CH>
__device__ __forceinline__ void sort_in_registers(uint64_t* list, uint32_t n, int lane)
{
    uint64_t c[CH];
#pragma unroll
    for (int q = 0; q < CH; ++q)
    {
        const uint32_t idx = q * kWave + lane;
        c[q]               = idx < n ? list[idx] : kInfKey;
    }
#pragma unroll
    for (int q = 0; q < CH; ++q) c[q] = bitonic_sort_groups<6>(c[q], lane);
    auto reversed = [&](uint64_t v) {
        const uint32_t lo = lane_xor<63>((uint32_t)v, lane), hi = lane_xor<63>((uint32_t)(v >> 32), lane);
        return ((uint64_t)hi << 32) | lo;
    };
#pragma unroll
    for (int w = 2; w <= CH; w <<= 1)  // w chunks per block of this level
    {
#pragma unroll
        for (int q = 0; q < CH; ++q)
            if ((q % w) < w / 2)
            {
                const int p        = q - (q % w) + (w - 1 - (q % w));
                const uint64_t r   = reversed(c[p]);
                const uint64_t mn  = r < c[q] ? r : c[q], mx = r < c[q] ? c[q] : r;
                c[q]               = mn;
                c[p]               = reversed(mx);
            }
#pragma unroll
        for (int d = w / 4; d >= 1; d >>= 1)
#pragma unroll
            for (int q = 0; q < CH; ++q)
                if ((q & d) == 0)
                {
                    const uint64_t x = c[q], y = c[q + d];
                    c[q]             = y < x ? y : x;
                    c[q + d]         = y < x ? x : y;
                }
#pragma unroll
        for (int q = 0; q < CH; ++q) c[q] = bitonic_merge64(c[q], lane);
    }
#pragma unroll
    for (int q = 0; q < CH; ++q)
    {
        const uint32_t idx = q * kWave + lane;
        if (idx < n) list[idx] = c[q];
    }
}

// Sorts the lists of one wave: lane i holds the start `off` (an index into `fragments`) and the length `n` of its list
// (n = 0 for lanes without a list). `fragments` may point to global memory or to LDS. Lists that have to be sorted in
// full and hold more than 64 CHUNKS and up to `skip_longer` keys are left alone: the caller sorts them by other means.
template <int CHUNKS = 4>
__device__ __forceinline__ void sort_wave_lists(uint64_t* fragments, uint8_t* src_lane, uint32_t off, uint32_t n,
                                                int lane, int K, uint32_t skip_longer = 0)
{
    // class = ceil(log2(n)) for 2 <= n <= 64, 0 for n <= 1 (nothing to do), 7 for n > 64
    int cls = 0;
    if (n > 64)
        cls = 7;
    else if (n > 1)
        cls = 32 - __clz((int)(n - 1));

    const uint64_t lanes_below = (1ull << lane) - 1ull;
#pragma unroll
    for (int c = 1; c <= 6; ++c)
    {
        const uint64_t mask = __ballot(cls == c);
        if (mask == 0ull) continue;
        if (cls == c) src_lane[__popcll(mask & lanes_below)] = (uint8_t)lane;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const int count = __popcll(mask);
        switch (c)
        {
            case 1: sort_class<1>(fragments, src_lane, count, off, n, lane, K); break;
            case 2: sort_class<2>(fragments, src_lane, count, off, n, lane, K); break;
            case 3: sort_class<3>(fragments, src_lane, count, off, n, lane, K); break;
            case 4: sort_class<4>(fragments, src_lane, count, off, n, lane, K); break;
            case 5: sort_class<5>(fragments, src_lane, count, off, n, lane, K); break;
            default: sort_class<6>(fragments, src_lane, count, off, n, lane, K); break;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }

    uint64_t long_mask = __ballot(cls == 7);
    while (long_mask != 0ull)
    {
        const int src = __ffsll((unsigned long long)long_mask) - 1;
        long_mask &= long_mask - 1ull;
        const uint32_t o  = __shfl(off, src, kWave);
        const uint32_t nn = __shfl(n, src, kWave);
        if (K > 0 && K <= kWave)
            select_smallest(fragments + o, nn, lane, K);
        else if (nn <= 2 * kWave)
            sort_in_registers<2>(fragments + o, nn, lane);
        else if (CHUNKS > 2 && nn <= (uint32_t)(CHUNKS * kWave))
            sort_in_registers<CHUNKS>(fragments + o, nn, lane);
        else if (nn <= skip_longer)
            continue;  // the caller sorts lists of this length with the whole workgroup
        else
            sort_in_memory(fragments + o, nn, lane);
    }
}

}  // namespace vetrast
