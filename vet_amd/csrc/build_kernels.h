// Per-bin list building: the last step of the forward binning (see forward_kernels.h for the whole scheme).
#pragma once
#include "common.h"
#include "forward_kernels.h"
#include "sort_kernels.h"

namespace vetrast
{
// A bin's records become sorted per-pixel lists in LDS: count per pixel and rank inside the pixel with LDS atomics, scan of
// the (at most 256) counts, keys to list start + rank, lists sorted with register networks; the sorted stretch goes out
// coalesced and is blended right there (BlendMulti, src/lib/rendering/RenderForward.cu:1303-1357): a lane gathers the
// descriptor record of one kept fragment into an LDS stage, then the lane that owns a pixel walks its fragments of that
// stretch front to back in exactly the reference's order: out += (T*c)*t, T = (1-c)*T.
//
// What bounds the pass: its steps are memory round trips and LDS accesses one after the other, so that a compute unit has to
// have many bins under way; once it has, vector instructions (two thirds to four fifths of its cycles) and the stores of the
// results. Four ways, by the number of records:
//  * up to kWaveBinCap of them ONE WAVE builds a bin, four to a workgroup, 32 to a compute unit, without a barrier;
//  * up to kBuildCap a workgroup, 8 to a compute unit, whose waves part where every wave has its pixels' keys (bins of
//    few pixels stay together: the walk wants their pixels side by side in one wave);
//  * up to kBuildMaxRuns times that several workgroups, each a stretch of the bin's pixels (parts_of_bin), in runs that fit;
//  * beyond, or with a list that does not fit by itself, or in small bins with cut lists (shared_end) beyond kBuildCap, one workgroup
//    in the fragment buffer.
// Lists that have to be sorted in full are sorted in a wave's registers up to 256 keys (128 in the fragment buffer), by the workgroup
// up to 1024, and by a wave in the fragment buffer beyond.
// The scan of the bin counts writes down the bins with more than kWaveBinCap records; the first crowded_blocks workgroups go
// through that list, the others take four neighbouring bins each. With a workgroup for every bin and everything beyond
// kBuildCap in the fragment buffer, against now (us, kernel traces on one card): two million points at 1080p 89 and 71, with the
// 2x2 splat 288 and 196, four of its 512x512 crops 255 and 87, four town views of 39 records a bin 457 and 236 (of which the
// stores of the results are 75), a million points in 1279x719 with the 2x2 splat 86 and 74, two FUZZY_BLEND views 151 and 111, ten
// million points 667 and 447. A view in which only a few hundred bins hold anything, and those up to 256 records, is the slower for a
// wave's longer chain: 230 thousand points in 1418x834 19 and 22, 120 thousand FUZZY_BLEND in 1471x814 21 and 25. Neither a workgroup
// for each bin there (25 and 31) nor four waves, each a quarter of the pixels (26 and 28), makes up for it.
constexpr int kBuildPerThread = kBuildCap / kBlock;
constexpr int kWavePerLane    = kWaveBinCap / kWave;
static_assert(kPrimaryCapSmall >= kBuildCap, "a bin built in LDS must find all its records in its own room");
constexpr uint32_t kBuildLongest = kBuildCap;  // a bin of more than kBuildCap records with a longer list goes through memory

// Workgroups of a launch that go through the crowded bins, several each where there are more. One that finds no bin costs
// a load, so there are no more of them than of the others, or than bins can be crowded at all; but where there are few bins,
// as many as the compute units hold at a time, since all may be crowded (a hundred points a pixel in 64x64: with a workgroup to four
// bins 84 us, with 1024 workgroups 44, with 2048 42). And at most twice that, so that one that is done early makes room for another.
constexpr uint32_t kCrowdedAtOnce = 2048;
constexpr uint32_t kCrowdedBlocks = 4096;

struct BuildPass
{
    const uint32_t* bin_offsets;  // [bins + 1] exclusive scan of the bin counts
    const uint4* primary;         // the bins' rooms (LayerTable::room_base): the first room_cap[l] records of every bin
    const uint4* binned;          // compact array: record r >= room_cap[l] of a bin sits at bin_offsets[bin] + r
    int compact_records;          // both hold 8-byte records (depth bits, point id << 8 | pixel in bin), see ScatterTargets
    uint32_t* offsets;    // [P + 1] per pixel: start of its list; [P] = fragments of the view
    uint64_t* fragments;
    uint8_t* list_is_cut;   // [P]
    uint64_t* last_key;     // [P] where list_is_cut: key of the last fragment that took part in the blend (0: none did)
    uint32_t* kept;         // [P] fragments of the pixel that took part in the blend
    // blending
    const float2* projected;  // BILINEAR_BLEND only: [N] where a point projects to at layer 0 (the alpha of a fragment
                              // depends on it)
    const int32_t* index;
    const float4* packed;
    const float* background;
    float* transmittance;  // per fragment, null unless the backward pass will run
    float* weight;         // per pixel
    float* out[VETRAST_MAX_LAYERS];       // already offset to this view
    float* out_mask[VETRAST_MAX_LAYERS];  // already offset to this view, or null
    float* out_weight[VETRAST_MAX_LAYERS];  // the same
    LayerTable ly;
    const uint2* crowded;            // bins of more than kWaveBinCap records, see CrowdedBins
    const uint32_t* crowded_counts;
    uint32_t crowded_capacity;
    uint32_t crowded_blocks;         // workgroups at the front of the grid that go through them
    uint32_t blocks_in_runs;         // workgroups behind those that take their bins in runs (in_runs): whole groups of them, or none
    uint32_t num_bins;
    uint32_t shared_end;             // see CrowdedBins
    int N;
    int K;
    int use_environment_map;
    float mask_value;
    float depth_accept;  // FUZZY_BLEND: depth range of a bucket
};

// Alpha of a fragment: the point's confidence, in BILINEAR_BLEND times this, the bilinear weight of the pixel's corner at the
// point's position in layer l (BlendMultiBilinear, src/lib/rendering/RenderForward.cu:1586-1613). The position at layer 0 is
// the projection the scatter pass stored, so the weight is reproduced bit for bit.
__device__ __forceinline__ float corner_weight(float2 position, int l, int corner)
{
    for (int k = 0; k < l; ++k) position.x *= 0.5f, position.y *= 0.5f;
    return bilinear_weight(position.x, position.y, corner);
}

// BILINEAR_BLEND stops a pixel once its transmittance is below 0.001 (src/lib/rendering/RenderForward.cu:1626) and then
// leaves the background out as well (:1633). The reference compares in double; the float nearest to 0.001 is the smallest
// one that isn't below it, so the comparison in float comes out the same for every T.
template <bool BILINEAR>
__device__ __forceinline__ bool blend_is_saturated(float T)
{
    static_assert((double)0.001f >= 0.001, "0.001f must not be below 0.001");
    return BILINEAR && T < 0.001f;
}

// FUZZY_BLEND (BlendMultiFuzzy, src/lib/rendering/RenderForward.cu:1393-1503): fragments are collected while their depth
// stays within depth_accept of the bucket's first one; a bucket is blended as ONE fragment with the mean confidence and
// the mean descriptor of its elements. After the first bucket the reference sets its reference depth to -100000 (:1468)
// instead of the next fragment's depth, so every later fragment closes the bucket in front of it: only the nearest
// bucket ever holds more than one fragment, and a one-element bucket blends exactly like a FULL_BLEND fragment
// (x / 1.0f == x). So the state below only lives until the nearest bucket is closed; from then on the ordinary blend
// step runs. (That needs depth + 100000 >= depth_accept, which the host checks: depth_accept < 10000.)
template <int C>
struct FuzzyBucket
{
    bool open = true;  // the nearest bucket is still collecting
    float first_depth = 0.f, conf = 0.f;
    float t[C];
    int m = 0;
    __device__ __forceinline__ FuzzyBucket()
    {
#pragma unroll
        for (int ci = 0; ci < C; ++ci) t[ci] = 0.f;
    }
    // blends the collected elements into (T, color) as one fragment
    __device__ __forceinline__ void flush(float& T, float (&color)[C])
    {
        const float fm = (float)m;
        const float cf = conf / fm;
        const float Tc = T * cf;
#pragma unroll
        for (int ci = 0; ci < C; ++ci) color[ci] = Tc * (t[ci] / fm) + color[ci];
        T    = (1.f - cf) * T;
        open = false;
    }
    // Fragment at depth d: true if it joined the nearest bucket; false if it lies behind it, in which case the bucket
    // has been blended and the caller blends the fragment by itself.
    __device__ __forceinline__ bool take(float d, float cf, const float (&td)[4], float depth_accept, float& T,
                                         float (&color)[C])
    {
        if (m == 0) first_depth = d;
        if (!(d - first_depth < depth_accept))
        {
            flush(T, color);
            return false;
        }
        conf += cf;
#pragma unroll
        for (int ci = 0; ci < C; ++ci) t[ci] += td[ci];
        ++m;
        return true;
    }
};

// Sorts list[0, n) in LDS, n <= kBuildCap, by the whole workgroup; places beyond n act as +infinity and are never touched. Every
// wave sorts 64-key chunks in registers, then the chunks are merged pairwise, level by level, in the all-ascending form of the
// bitonic network: a mirror step and the halving steps over 64 or more places run on LDS with a barrier each, the last six halving
// steps of every level again in registers. A list of 512 keys takes 13 barriers instead of the 45 of the plain network. Every
// thread of the workgroup must call.
__device__ __forceinline__ void block_sort(uint64_t* list, uint32_t n, int tid)
{
    const int lane = tid & (kWave - 1), wave = tid / kWave;
    uint32_t m = kWave;
    while (m < n) m <<= 1;  // <= kBuildCap
    auto in_chunks = [&](auto sorted) {
        for (uint32_t c = wave; c * kWave < n; c += kBlock / kWave)
        {
            const uint32_t at  = c * kWave + lane;
            const uint64_t key = sorted(at < n ? list[at] : kInfKey);
            if (at < n) list[at] = key;
        }
        __syncthreads();
    };
    auto order = [&](uint32_t i, uint32_t j) {  // i < j: the smaller key to place i
        if (j >= n) return;
        const uint64_t x = list[i], y = list[j];
        if (y < x)
        {
            list[i] = y;
            list[j] = x;
        }
    };
    __syncthreads();
    in_chunks([&](uint64_t key) { return bitonic_sort_groups<6>(key, lane); });
    for (uint32_t k = 2 * kWave; k <= m; k <<= 1)
    {
        const uint32_t hk = k >> 1;
        for (uint32_t p = tid; p < (m >> 1); p += kBlock)  // mirror step inside every block of k places
        {
            const uint32_t blk = p / hk, r = p % hk;
            order(blk * k + r, blk * k + (k - 1 - r));
        }
        __syncthreads();
        for (uint32_t jj = k >> 2; jj >= (uint32_t)kWave; jj >>= 1)
        {
            for (uint32_t p = tid; p < (m >> 1); p += kBlock)
            {
                const uint32_t i = (p / jj) * 2 * jj + (p % jj);
                order(i, i + jj);
            }
            __syncthreads();
        }
        in_chunks([&](uint64_t key) { return bitonic_merge64(key, lane); });
    }
}

// The same for a list in memory, through the LDS room `room` (kBuildCap keys).
__device__ __forceinline__ void block_sort_through_lds(uint64_t* list, uint32_t n, uint64_t* room, int tid)
{
    for (uint32_t k = tid; k < n; k += kBlock) room[k] = list[k];
    block_sort(room, n, tid);
    for (uint32_t k = tid; k < n; k += kBlock) list[k] = room[k];
    __syncthreads();
}

// The arguments of a launch as they lie in the kernel's argument segment. `again` hands them on as something the compiler
// knows nothing about yet, so that what a step of the pass needs of them is loaded there (from the scalar cache) instead of
// being kept in scalar registers since the step before: there are 80 of those for eight waves, and the pass would put off over
// a hundred into vector registers, lane by lane.
using BuildArgs = const __attribute__((address_space(4))) BuildPass;
__device__ __forceinline__ BuildArgs& again(BuildArgs& a)
{
    BuildArgs* p = &a;
    asm volatile("" : "+s"(p));
    return *p;
}

// Where a bin lies; the same for every lane that works on it.
struct BinPlace
{
    int l;
    uint32_t pixels;  // of the bin: 256, 64, 16 or 4
    uint32_t q0;      // first of them
    int x0, y0;       // corner of the tile it lies in
    size_t room;      // first record of its room
};

__device__ __forceinline__ BinPlace place_of_bin(BuildArgs& a, uint32_t bin)
{
    BinPlace p;
    p.l = 0;
#pragma unroll
    for (int k = 1; k < VETRAST_MAX_LAYERS; ++k)
        if (k < a.ly.L && bin >= a.ly.bin_base[k]) p.l = k;
    const int shift = a.ly.bin_shift[p.l];
    p.pixels        = 1u << shift;
    p.q0            = a.ly.base[p.l] + ((bin - a.ly.bin_base[p.l]) << shift);
    p.room          = (size_t)a.ly.room_base[p.l] + (size_t)(bin - a.ly.bin_base[p.l]) * a.ly.room_cap[p.l];  // room_of_bin
    const uint32_t tile = (p.q0 - a.ly.base[p.l]) / kTilePixels;
    const uint32_t ty   = tile / (uint32_t)a.ly.tiles_x[p.l];
    p.x0 = (int)((tile - ty * (uint32_t)a.ly.tiles_x[p.l]) * kTile);
    p.y0 = (int)(ty * kTile);
    return p;
}

// A fragment record as it comes from memory. Taking it apart is a step of its own: the form is the same for all records of a
// call, but the compiler waits at the end of each side of the choice for what is used there, one record after the other.
struct RawRecord
{
    uint32_t x, y, z;
};
struct FragmentRecord
{
    uint64_t key;
    uint32_t pixel;  // inside the bin
};

// N records at once, record k from `at(k)` on in 8-byte or 16-byte units.
template <int N, class At>
__device__ __forceinline__ void load_records(BuildArgs& a, RawRecord (&raw)[N], At at)
{
    if (a.compact_records)
    {
#pragma unroll
        for (int k = 0; k < N; ++k)
        {
            const uint2 v = *at((const uint2*)nullptr, k);
            raw[k]        = {v.x, v.y, 0u};
        }
    }
    else
    {
#pragma unroll
        for (int k = 0; k < N; ++k)
        {
            const uint4 v = *at((const uint4*)nullptr, k);
            raw[k]        = {v.x, v.y, v.z};
        }
    }
}

__device__ __forceinline__ FragmentRecord taken_apart(BuildArgs& a, const RawRecord& r, uint32_t pixels)
{
    const bool compact = a.compact_records != 0;
    const uint32_t low = compact ? r.y >> 8 : r.x, depth = compact ? r.x : r.y, pixel = compact ? r.y & 0xFFu : r.z;
    return {((uint64_t)depth << 32) | low, pixel & (pixels - 1u)};
}

// What a bin (or a run of its pixels) keeps in LDS, for a workgroup or for one wave.
struct BinRoom
{
    uint64_t* keys;
    // per pixel the place of its list among the keys | place among the items << 16, and behind the last pixel the ends, so
    // that the difference of two neighbours holds the length of the list and how many of it the cut leaves (before the
    // scan: the pixel's count)
    uint32_t* places;
    uint8_t* items;  // the pixel of every fragment the cut leaves, pixel after pixel
    // a stage of the blend: descriptor, alpha, and depth (FUZZY_BLEND), in whose place the transmittance in front comes
    float4* t;
    float* alpha;
    float* depth;
};

__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The same number, of which the compiler knows nothing: what follows from a thread's number then isn't worked out ahead of a
// loop and kept in registers for all of it (the pass needs 64 of them at most to have its eight workgroups, and took 139).
__device__ __forceinline__ int opaque(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

__device__ __forceinline__ uint32_t uniform(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }

// Everything the forward pass writes for a pixel once its list is blended.
template <int C, bool BILINEAR>
__device__ __forceinline__ void store_pixel(BuildArgs& args, const BinPlace& bin, uint32_t pixel, uint32_t count, uint32_t used,
                                            uint64_t last, bool saturated, float T, float (&color)[C])
{
    BuildArgs& a     = again(args);
    const int l      = bin.l;
    const uint32_t q = bin.q0 + pixel;
    // How many fragments of the list took part, and one byte that says whether any did not (top-K cut, saturation):
    // the backward per-point kernel only has to look at the last blended key of a pixel where this is set.
    // (FULL_BLEND blends min(count, K) fragments, which the readers work out themselves: the array is not written.)
    if constexpr (BILINEAR) a.kept[q] = used;
    a.list_is_cut[q] = used < count ? 1 : 0;
    if (used < count) a.last_key[q] = last;
    const int x = bin.x0 + (int)(q & (kTile - 1)), y = bin.y0 + (int)((q / kTile) & (kTile - 1));
    if (x < a.ly.w[l] && y < a.ly.h[l])
    {
        const size_t plane   = (size_t)a.ly.w[l] * a.ly.h[l];
        const uint32_t local = (uint32_t)y * (uint32_t)a.ly.w[l] + (uint32_t)x;
        // The background comes from the scalar cache, the same for every pixel: as a vector load it was waited for together with all
        // stores in front of it, for every channel of every 64 pixels.
        if (!a.use_environment_map && !saturated)
        {
            const __attribute__((address_space(4))) float* background = (const __attribute__((address_space(4))) float*)a.background;
#pragma unroll
            for (int ci = 0; ci < C; ++ci) color[ci] = (T * 1.f) * background[ci] + color[ci];
        }
#pragma unroll
        for (int ci = 0; ci < C; ++ci) a.out[l][ci * plane + local] = color[ci];
        a.weight[q] = T;
        if (a.out_mask[l]) a.out_mask[l][local] = (T == 0.f) ? a.mask_value : 1.f;
        if (a.out_weight[l]) a.out_weight[l][local] = T;
    }
}

// Writes out and blends the sorted lists of the pixels [p0, p1) of a bin, which lie in `room` with place 0 of the keys at
// place `begin` of the fragment buffer. TEAM waves work together: 1, whose lanes take 64 pixels after the other, or all 4
// of a workgroup (every thread must call; `me` is the lane or the thread) for at most 64 pixels, which the first wave's
// lanes walk. A step stages 64 TEAM kept fragments, and the records of the next step are under way while the pixels' lanes walk
// this one: the fragments as they lie, pixel after pixel, or (TURNS, up to 16 pixels) as many of every pixel.
template <int C, bool BILINEAR, bool FUZZY, int TEAM, bool TURNS>
__device__ __forceinline__ void blend_steps(BuildArgs& args, const BinPlace& bin, const BinRoom& room, uint32_t begin, uint32_t p0,
                                            uint32_t p1, int me)
{
    BuildArgs& a             = again(args);
    constexpr uint32_t kStep = kWave * TEAM;
    auto sync = [] {
        if constexpr (TEAM == 1)
            wave_sync();
        else
            __syncthreads();
    };
    const uint32_t first = uniform(room.places[p0]), end = uniform(room.places[p1]);
    // Steps go over items; in turns over ranks inside the lists, `turn` of them a step.
    const uint32_t turn = !TURNS ? kStep : (p1 - p0 <= 4u ? kStep / 4u : kStep / 16u);
    uint32_t first_item = first >> 16, last_item = end >> 16;
    if constexpr (TURNS)
    {
        const uint32_t px = p0 + (uint32_t)(me & 15);
        first_item        = 0u;
        last_item         = wave_max(px < p1 ? (room.places[px + 1] - room.places[px]) >> 16 : 0u);
    }
    // the fragment this lane stages next
    float4 t4     = make_float4(0.f, 0.f, 0.f, 0.f);
    float alpha   = 0.f;
    float2 ip     = make_float2(0.f, 0.f);
    uint32_t at   = 0xFFFFFFFFu;  // its place among the keys, or none
    auto fetch = [&](uint32_t base) {
        at = 0xFFFFFFFFu;
        if constexpr (TURNS)
        {
            const uint32_t px = p0 + (uint32_t)me / turn, rank = base + (uint32_t)me % turn;
            if (px >= p1) return;
            const uint32_t places = room.places[px];
            if (rank >= (room.places[px + 1] - places) >> 16) return;
            at = (places & 0xFFFFu) + rank;
        }
        else
        {
            const uint32_t item = base + (uint32_t)me;
            if (item >= last_item) return;
            const uint32_t places = room.places[room.items[item]];
            at                    = (places & 0xFFFFu) + item - (places >> 16);
        }
        const uint64_t key    = room.keys[at];
        const uint32_t low    = (uint32_t)key;
        const int id          = BILINEAR ? (int)(low >> 2) : (int)low;
        // an id or texture index out of range cannot come from a list the scatter pass wrote; such a fragment
        // blends as fully transparent (the reference asserts on the texture index, RenderForward.cu:1335-1336)
        const int ti = texture_row(a.index, id, a.N);
        if (ti < 0)
            t4 = make_float4(0.f, 0.f, 0.f, 0.f), alpha = 0.f;
        else
        {
            t4    = a.packed[2 * (size_t)ti];
            alpha = a.packed[2 * (size_t)ti + 1].x;
            // written by the scatter pass for every point that has fragments
            if constexpr (BILINEAR) ip = a.projected[id];
        }
    };
    fetch(first_item);

    // the 64 pixels being walked, and this lane's
    const bool walks = TEAM == 1 || me < kWave;
    uint32_t p       = p0;
    uint32_t start = 0, count = 0, item = 0, keep = 0, used = 0, items_end = 0;
    bool saturated = false;
    float T        = 1.f;
    float color[C];
    FuzzyBucket<C> fuzzy;  // FUZZY_BLEND only
    auto next_pixels = [&] {
        const uint32_t px = p + (uint32_t)(me & (kWave - 1));
        uint32_t places = 0, length = 0;
        if (px < p1)
        {
            places = room.places[px];
            length = room.places[px + 1] - places;
        }
        start = places & 0xFFFFu, item = places >> 16, count = length & 0xFFFFu, keep = length >> 16;
        items_end = uniform(room.places[min(p + (uint32_t)kWave, p1)]) >> 16;
        used = 0, saturated = false, T = 1.f;
#pragma unroll
        for (int ci = 0; ci < C; ++ci) color[ci] = 0.f;
        if constexpr (FUZZY) fuzzy = FuzzyBucket<C>();
    };
    next_pixels();
    for (uint32_t base = first_item;; base += turn)
    {
        const uint32_t staged = at;
        if (BILINEAR && staged != 0xFFFFFFFFu) alpha = corner_weight(ip, bin.l, (int)((uint32_t)room.keys[staged] & 3u)) * alpha;
        room.t[me]     = t4;
        room.alpha[me] = alpha;
        if (FUZZY && staged != 0xFFFFFFFFu) room.depth[me] = __uint_as_float((uint32_t)(room.keys[staged] >> 32));
        sync();
        const bool more = base + turn < last_item;  // the same for the whole team
        if (more) fetch(base + turn);
        // the keys go out while the first fragments are walked
        if (base == first_item)
            for (uint32_t r = (first & 0xFFFFu) + (uint32_t)me; r < (end & 0xFFFFu); r += kStep) a.fragments[begin + r] = room.keys[r];
        for (;;)
        {
            if (walks)
            {
                // this lane's fragments of the stage: the first of them, behind the last, and what the rank is ahead of them
                const bool some   = TURNS ? keep > base : item + keep > base && item < base + kStep;
                uint32_t r        = TURNS ? (uint32_t)me * turn : max(item, base) - base;
                const uint32_t hi = TURNS ? r + min(keep - base, turn) : min(item + keep, base + kStep) - base;
                const uint32_t ahead = TURNS ? base - r : base - item;
                if (!saturated && some)
                {
                    if constexpr (FUZZY)
                    {
                        // The nearest bucket, in a loop of its own, so that the loop below is FULL_BLEND's. What is stored
                        // is the transmittance in front of the bucket the fragment joins.
                        for (; r < hi && fuzzy.open; ++r)
                        {
                            const float4 t4  = room.t[r];
                            const float cf   = room.alpha[r];
                            const float t[4] = {t4.x, t4.y, t4.z, t4.w};
                            const bool joined = fuzzy.take(room.depth[r], cf, t, a.depth_accept, T, color);
                            room.depth[r]    = T;
                            if (joined) continue;
                            const float Tc = T * cf;
#pragma unroll
                            for (int ci = 0; ci < C; ++ci) color[ci] = Tc * t[ci] + color[ci];
                            T = (1.f - cf) * T;
                        }
                    }
                    for (; r < hi && !saturated; ++r)
                    {
                        const float4 t4  = room.t[r];
                        const float cf   = room.alpha[r];
                        const float t[4] = {t4.x, t4.y, t4.z, t4.w};
                        room.depth[r]    = T;
                        const float Tc   = T * cf;
#pragma unroll
                        for (int ci = 0; ci < C; ++ci) color[ci] = Tc * t[ci] + color[ci];
                        T = (1.f - cf) * T;
                        saturated = blend_is_saturated<BILINEAR>(T);
                    }
                    used = ahead + r;
                }
            }
            if (TURNS ? more : items_end > base + kStep) break;  // these pixels go on in the next step
            if (walks && p + (uint32_t)(me & (kWave - 1)) < p1)
            {
                if constexpr (FUZZY)
                    if (fuzzy.open && fuzzy.m > 0) fuzzy.flush(T, color);
                const uint64_t last = used && used < count ? room.keys[start + used - 1u] : 0ull;
                store_pixel<C, BILINEAR>(a, bin, p + (uint32_t)(me & (kWave - 1)), count, used, last, saturated, T, color);
            }
            p += kWave;
            if (p >= p1) break;
            next_pixels();
        }
        // the next fragments are waited for in front of this store: behind it, they would wait for its end
        asm volatile("" : "+v"(t4.x), "+v"(t4.y), "+v"(t4.z), "+v"(t4.w), "+v"(alpha), "+v"(ip.x), "+v"(ip.y));
        sync();
        // (for fragments behind a saturated pixel's last one this is no transmittance; nobody reads it)
        if (a.transmittance && staged != 0xFFFFFFFFu) a.transmittance[begin + staged] = room.depth[me];
        if (!more) break;
    }
}

// A bin of up to kWaveBinCap records, by one wave.
template <int C, bool BILINEAR, bool FUZZY>
__device__ __forceinline__ void build_by_wave(BuildArgs& args, uint32_t bin, const BinRoom& room, int lane)
{
    BuildArgs& a         = again(args);
    const BinPlace place = place_of_bin(a, bin);
    // the first records are under way before it is known how many there are: a room has memory for more, whatever is in it
    RawRecord raw[kWavePerLane];
    auto in_room = [&](int first) {
        return [&, first](auto type, int k) { return reinterpret_cast<decltype(type)>(a.primary) + place.room + (first + k) * kWave + lane; };
    };
    {
        RawRecord one[1];
        load_records(a, one, in_room(0));
        raw[0] = one[0];
    }
    uint32_t begin = a.bin_offsets[bin], end = a.bin_offsets[bin + 1];
    // (waited for together: else the compiler moves the records behind the test, where they are needed)
    asm volatile("" : "+v"(raw[0].x), "+v"(raw[0].y), "+v"(raw[0].z), "+v"(begin), "+v"(end));
    begin            = uniform(begin);
    const uint32_t n = uniform(end) - begin;
    if (n > (uint32_t)kWaveBinCap) return;  // on the list
    reinterpret_cast<uint4*>(room.places)[lane] = make_uint4(0u, 0u, 0u, 0u);
    if (n > (uint32_t)kWave)
    {
        RawRecord more[kWavePerLane - 1];
        load_records(a, more, in_room(1));
#pragma unroll
        for (int k = 1; k < kWavePerLane; ++k) raw[k] = more[k - 1];
    }
    FragmentRecord rec[kWavePerLane];
    wave_sync();
    uint32_t rank[kWavePerLane];
#pragma unroll
    for (int k = 0; k < kWavePerLane; ++k)
    {
        if ((uint32_t)(k * kWave) >= n) break;
        rec[k] = taken_apart(a, raw[k], place.pixels);
        if ((uint32_t)(k * kWave + lane) < n) rank[k] = atomicAdd(&room.places[rec[k].pixel], 1u);
    }
    wave_sync();
    {
        // lane i has the pixels 4 i .. 4 i + 3
        const uint4 c = reinterpret_cast<const uint4*>(room.places)[lane];
        auto both = [&](uint32_t count) { return count | ((a.K > 0 ? min(count, (uint32_t)a.K) : count) << 16); };
        const uint4 v = make_uint4(both(c.x), both(c.y), both(c.z), both(c.w));
        const uint32_t incl = wave_inclusive_scan((v.x + v.y) + (v.z + v.w), lane);
        uint4 o;
        o.x = incl - ((v.x + v.y) + (v.z + v.w));
        o.y = o.x + v.x;
        o.z = o.y + v.y;
        o.w = o.z + v.z;
        reinterpret_cast<uint4*>(room.places)[lane] = o;
        if (lane == kWave - 1) room.places[kTilePixels] = incl;
        if (4u * (uint32_t)lane < place.pixels)
        {
            // (q0 is a multiple of 4)
            reinterpret_cast<uint4*>(a.offsets + place.q0)[lane] =
                make_uint4(begin + (o.x & 0xFFFFu), begin + (o.y & 0xFFFFu), begin + (o.z & 0xFFFFu), begin + (o.w & 0xFFFFu));
            if (bin == a.num_bins - 1u && 4u * (uint32_t)lane + 4u == place.pixels) a.offsets[place.q0 + place.pixels] = begin + n;
        }
    }
    wave_sync();
#pragma unroll
    for (int k = 0; k < kWavePerLane; ++k)
    {
        if ((uint32_t)(k * kWave) >= n) break;
        if ((uint32_t)(k * kWave + lane) < n)
        {
            const uint32_t places = room.places[rec[k].pixel];
            room.keys[(places & 0xFFFFu) + rank[k]] = rec[k].key;
            if (a.K <= 0 || rank[k] < (uint32_t)a.K) room.items[(places >> 16) + rank[k]] = (uint8_t)rec[k].pixel;
        }
    }
    wave_sync();
    for (uint32_t p = 0; p < place.pixels; p += kWave)
    {
        uint32_t off = 0, length = 0;
        if (p + (uint32_t)lane < place.pixels)
        {
            off    = room.places[p + lane];
            length = (room.places[p + lane + 1] - off) & 0xFFFFu;
        }
        if (__ballot(length > 1u) != 0ull)
            sort_wave_lists(room.keys, reinterpret_cast<uint8_t*>(room.t), off & 0xFFFFu, length, lane, a.K);
    }
    wave_sync();
    // The few lanes that have a pixel of a small bin would walk one list after the other where the lists are long: with more than a
    // step's fragments they take turns (56 thousand points without a cut, 75 fragments a pixel in the coarsest layer: 32 against 23 us
    // of the pass; a workgroup for a bin of more than 64 records, whose steps hold 256, 23 as well, but dense views lose 3 to 8 %).
    if (place.pixels <= 16u && uniform(room.places[kTilePixels]) >> 16 > (uint32_t)kWave)
        blend_steps<C, BILINEAR, FUZZY, 1, true>(a, place, room, begin, 0u, place.pixels, lane);
    else
        blend_steps<C, BILINEAR, FUZZY, 1, false>(a, place, room, begin, 0u, place.pixels, lane);
}


// A bin that cannot be built in LDS, by a workgroup: the keys go to their lists in the fragment buffer, where they are sorted
// and walked. `starts` (of the lists, in the bin) and `cursors` (zeros) are per pixel in LDS.
template <int C, bool BILINEAR, bool FUZZY, class Records>
__device__ __forceinline__ void build_in_memory(BuildArgs& args, const BinPlace& bin, const BinRoom& room, const uint32_t* starts,
                                                uint32_t* cursors, uint64_t* lists_by_block, Records records, uint32_t begin,
                                                uint32_t n)
{
    BuildArgs& a  = again(args);
    const int tid = opaque(threadIdx.x), lane = tid & (kWave - 1), wave = tid / kWave;
    const uint32_t pixels = bin.pixels;
    // wave w sorts the lists of its quarter of the bin's pixels
    const uint32_t per_wave = pixels >> 2;  // >= 1
    uint32_t list_off = 0, list_len = 0;
    if ((uint32_t)lane < per_wave)
    {
        const uint32_t px = wave * per_wave + lane;
        list_off          = starts[px];
        list_len          = (px + 1u < pixels ? starts[px + 1] : n) - list_off;
    }
    // second pass over the records: a fresh cursor per pixel hands out the places inside the list (any order is
    // fine, the lists are sorted afterwards)
    for (uint32_t r0 = 0; r0 < n; r0 += kBlock * 4)
    {
        RawRecord raw[4];
        load_records(a, raw, records(r0));
#pragma unroll
        for (int k = 0; k < 4; ++k)
        {
            if (r0 + k * kBlock + tid >= n) continue;
            const FragmentRecord rec = taken_apart(a, raw[k], pixels);
            const uint32_t rank      = atomicAdd(&cursors[rec.pixel], 1u);
            a.fragments[begin + starts[rec.pixel] + rank] = rec.key;
        }
    }
    __threadfence_block();  // the keys other waves stored are read below
    __syncthreads();
    // Lists that have to be sorted in full and are too long for a wave's registers are sorted by the whole
    // workgroup through the key array in LDS, which is not in use on this path, one list after the other (in global
    // memory every step of the network costs a memory round trip, and such a list needs dozens of steps).
    const bool full_sort = !(a.K > 0 && a.K <= kWave);
    constexpr int kChunks = 2;  // (four of them would not fit the 64 registers here)
    sort_wave_lists<kChunks>(a.fragments + begin, reinterpret_cast<uint8_t*>(room.t) + wave * kWave, list_off, list_len, lane, a.K,
                             /*skip_longer=*/(uint32_t)kBuildCap);
    __threadfence_block();
    __syncthreads();
    if (full_sort)
    {
        const uint32_t c = (uint32_t)tid < pixels ? cursors[tid] : 0u;
        const bool mine  = c > (uint32_t)(kChunks * kWave) && c <= (uint32_t)kBuildCap;  // pixel tid
        const uint64_t wave_mask = __ballot(mine);
        if (lane == 0) lists_by_block[opaque(threadIdx.x) / kWave] = wave_mask;
        __syncthreads();
        for (int w = 0; w < kBlock / kWave; ++w)  // the same trips for every thread
        {
            uint64_t todo = lists_by_block[w];
            while (todo != 0ull)
            {
                const uint32_t px = w * kWave + (__ffsll((unsigned long long)todo) - 1);
                todo &= todo - 1ull;
                block_sort_through_lds(a.fragments + begin + starts[px], cursors[px], room.keys, opaque(threadIdx.x));
            }
        }
    }
    __threadfence_block();
    __syncthreads();
    // this thread's pixel
    const uint32_t start = (uint32_t)tid < pixels ? starts[tid] : n, c = (uint32_t)tid < pixels ? cursors[tid] : 0u;
    const uint32_t keep  = a.K > 0 ? min(c, (uint32_t)a.K) : c;
    uint32_t used  = 0;  // fragments that took part in the blend
    bool saturated = false;
    float T = 1.f;
    float color[C];
#pragma unroll
    for (int ci = 0; ci < C; ++ci) color[ci] = 0.f;
    FuzzyBucket<C> fuzzy;  // FUZZY_BLEND only
    // All threads gather the descriptor records of a stretch of the lists into the stage, then the pixel's thread walks its
    // fragments of that stretch. With a cut the stretches run over K places for every pixel, so that what it leaves out is
    // left out here as well; without one, or with one that cuts little, over the lists as they are.
    const bool by_cut         = a.K > 0 && (uint64_t)a.K * pixels <= n;
    const uint32_t own_places = by_cut ? (uint32_t)tid * (uint32_t)a.K : start;
    const uint32_t all_places = by_cut ? pixels * (uint32_t)a.K : n;
    for (uint32_t base = 0; base < all_places; base += kBlock)
    {
        const uint32_t r = base + tid;
        uint32_t at      = r;
        bool there       = r < all_places;
        if (by_cut && there)
        {
            const uint32_t px = r / (uint32_t)a.K, j = r - px * (uint32_t)a.K;
            at    = starts[px] + j;
            there = at < (px + 1u < pixels ? starts[px + 1] : n);
        }
        if (there)
        {
            const uint64_t key = a.fragments[begin + at];
            const uint32_t low = (uint32_t)key;
            const int id       = BILINEAR ? (int)(low >> 2) : (int)low;
            const int ti = texture_row(a.index, id, a.N);
            float4 t4    = make_float4(0.f, 0.f, 0.f, 0.f);
            float alpha  = 0.f;
            if (ti >= 0)
            {
                t4    = a.packed[2 * (size_t)ti];
                alpha = a.packed[2 * (size_t)ti + 1].x;
                if constexpr (BILINEAR) alpha = corner_weight(a.projected[id], bin.l, (int)(low & 3u)) * alpha;
            }
            room.t[tid]     = t4;
            room.alpha[tid] = alpha;
            if constexpr (FUZZY) room.depth[tid] = __uint_as_float((uint32_t)(key >> 32));
        }
        __syncthreads();
        if ((uint32_t)tid < pixels)
        {
            const uint32_t hi = min(own_places + keep, base + (uint32_t)kBlock);
            for (uint32_t k = max(own_places, base); k < hi && !saturated; ++k)
            {
                const float4 t4  = room.t[k - base];
                const float cf   = room.alpha[k - base];
                const float t[4] = {t4.x, t4.y, t4.z, t4.w};
                bool joined      = false;
                if constexpr (FUZZY) joined = fuzzy.open && fuzzy.take(room.depth[k - base], cf, t, a.depth_accept, T, color);
                if (a.transmittance) a.transmittance[begin + start + used] = T;
                ++used;
                if (joined) continue;
                const float Tc = T * cf;
#pragma unroll
                for (int ci = 0; ci < C; ++ci) color[ci] = Tc * t[ci] + color[ci];
                T         = (1.f - cf) * T;
                saturated = blend_is_saturated<BILINEAR>(T);
            }
        }
        __syncthreads();
    }
    if constexpr (FUZZY)
        if (fuzzy.open && fuzzy.m > 0) fuzzy.flush(T, color);
    if ((uint32_t)tid < pixels)
    {
        // (the sorted keys are in the fragment buffer)
        const uint64_t last = used && used < c ? a.fragments[begin + start + used - 1u] : 0ull;
        store_pixel<C, BILINEAR>(a, bin, (uint32_t)tid, c, used, last, saturated, T, color);
    }
}

// A bin of more than kWaveBinCap records, by a workgroup; or the `part`th of `parts` of it, the pixels whose lists start in
// that part of the bin's fragments.
template <int C, bool BILINEAR, bool FUZZY>
__device__ __forceinline__ void build_by_workgroup(BuildArgs& args, uint32_t bin, uint32_t part, uint32_t parts, const BinRoom& room, uint32_t* cursors,
                                                   uint64_t* lists_by_block, uint32_t* wave_words)
{
    BuildArgs& a  = again(args);
    const int tid = opaque(threadIdx.x), lane = tid & (kWave - 1), wave = tid / kWave;
    const BinPlace place    = place_of_bin(a, bin);
    const uint32_t pixels   = place.pixels;
    const uint32_t begin    = uniform(a.bin_offsets[bin]);
    const uint32_t n        = uniform(a.bin_offsets[bin + 1]) - begin;
    const uint32_t room_cap = a.ly.room_cap[place.l];
    // the four records a thread takes from `first` on (beyond the last one, that one again): the bin's own room first, what
    // did not fit there in the compact array
    auto records = [&](uint32_t first) {
        return [&, first](auto type, int k) {
            const uint32_t r = min(first + (uint32_t)(k * kBlock) + threadIdx.x, n - 1u);
            return r < room_cap ? reinterpret_cast<decltype(type)>(a.primary) + place.room + r
                                : reinterpret_cast<decltype(type)>(a.binned) + begin + r;
        };
    };
    const bool one_run = n <= (uint32_t)kBuildCap;
    room.places[tid]   = 0u;
    __syncthreads();

    // ---- count per pixel; the LDS atomic also hands every record its rank inside the pixel
    FragmentRecord rec[kBuildPerThread];
    uint32_t rank[kBuildPerThread];
    for (uint32_t r0 = 0; r0 < n; r0 += kBuildPerThread * kBlock)  // (one trip where the records fit)
    {
        RawRecord raw[kBuildPerThread];
        load_records(a, raw, records(r0));
#pragma unroll
        for (int k = 0; k < kBuildPerThread; ++k)
        {
            if (r0 + (uint32_t)(k * kBlock) >= n) break;  // uniform
            rec[k] = taken_apart(a, raw[k], pixels);
            if (r0 + (uint32_t)(k * kBlock + tid) < n) rank[k] = atomicAdd(&room.places[rec[k].pixel], 1u);
        }
    }
    __syncthreads();

    // ---- scan of the pixel counts: list starts, and where the fragments the cut leaves start
    const uint32_t c    = room.places[tid];
    const uint32_t keep = a.K > 0 ? min(c, (uint32_t)a.K) : c;
    const uint32_t incl = wave_inclusive_scan(c, lane), incl_keep = wave_inclusive_scan(keep, lane);
    if (lane == kWave - 1) wave_words[wave] = incl, wave_words[4 + wave] = incl_keep;
    if (!one_run)
    {
        const uint64_t long_lists = __ballot(c > kBuildLongest);
        if (lane == 0) wave_words[8 + wave] = long_lists != 0ull ? 1u : 0u;
    }
    __syncthreads();
    uint32_t start = incl - c, start_keep = incl_keep - keep;
    for (int k = 0; k < wave; ++k) start += wave_words[k], start_keep += wave_words[4 + k];
    uint32_t first_pixel = 0, end_pixel = pixels;
    if (!one_run)
    {
        const bool long_lists = (wave_words[8] | wave_words[9] | wave_words[10] | wave_words[11]) != 0u;
        if (long_lists || bin >= a.shared_end || n > (uint32_t)(kBuildMaxRuns * kBuildCap))
        {
            if (part != 0u) return;
            if ((uint32_t)tid < pixels) a.offsets[place.q0 + tid] = begin + start;
            if (bin == a.num_bins - 1u && tid == 0) a.offsets[place.q0 + pixels] = begin + n;
            room.places[tid] = start;
            cursors[tid]     = 0u;
            __syncthreads();
            build_in_memory<C, BILINEAR, FUZZY>(a, place, room, room.places, cursors, lists_by_block, records, begin, n);
            return;
        }
        __syncthreads();
        const uint32_t lies_in = min(start * parts / n, parts - 1u);
        const uint64_t before  = __ballot((uint32_t)tid < pixels && lies_in < part), inside = __ballot((uint32_t)tid < pixels && lies_in == part);
        if (lane == 0) wave_words[wave] = (uint32_t)__popcll(before), wave_words[4 + wave] = (uint32_t)__popcll(inside);
        __syncthreads();
        first_pixel = uniform((wave_words[0] + wave_words[1]) + (wave_words[2] + wave_words[3]));
        end_pixel   = first_pixel + uniform((wave_words[4] + wave_words[5]) + (wave_words[6] + wave_words[7]));
        if (first_pixel == end_pixel) return;
    }
    if ((uint32_t)tid >= first_pixel && (uint32_t)tid < end_pixel) a.offsets[place.q0 + tid] = begin + start;
    if (bin == a.num_bins - 1u && end_pixel == pixels && tid == 0) a.offsets[place.q0 + pixels] = begin + n;

    // (beyond the bin's pixels there are no records: the places are those behind the last one)
    auto put = [&](const FragmentRecord& r, uint32_t rank) {
        const uint32_t places = room.places[r.pixel];
        room.keys[(places & 0xFFFFu) + rank] = r.key;
        if (a.K <= 0 || rank < (uint32_t)a.K) room.items[(places >> 16) + rank] = (uint8_t)r.pixel;
    };
    if (one_run)
    {
        room.places[tid] = start | (start_keep << 16);
        if (tid == kBlock - 1) room.places[kTilePixels] = (start + c) | ((start_keep + keep) << 16);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kBuildPerThread; ++k)
        {
            if ((uint32_t)(k * kBlock) >= n) break;
            if ((uint32_t)(k * kBlock + tid) < n) put(rec[k], rank[k]);
        }
    }

    // ---- runs of pixels whose records fit: one as a rule
    for (uint32_t g0 = first_pixel; g0 < end_pixel;)
    {
        const int tid = opaque(threadIdx.x), lane = tid & (kWave - 1), wave = tid / kWave;
        uint32_t g1 = end_pixel, run_start = 0;
        if (!one_run)
        {
            __syncthreads();
            if ((uint32_t)tid == g0) wave_words[0] = start, wave_words[1] = start_keep;
            __syncthreads();
            run_start               = uniform(wave_words[0]);
            const uint32_t run_keep = uniform(wave_words[1]);
            const uint64_t fits = __ballot((uint32_t)tid >= g0 && (uint32_t)tid < end_pixel && start + c - run_start <= (uint32_t)kBuildCap);
            if (lane == 0) wave_words[4 + wave] = (uint32_t)__popcll(fits);
            cursors[tid] = 0u;
            // (nobody reads the places of a pixel in front of the run or beyond the one behind its end)
            room.places[tid] = (start - run_start) | ((start_keep - run_keep) << 16);
            if (tid == kBlock - 1) room.places[kTilePixels] = (start + c - run_start) | ((start_keep + keep - run_keep) << 16);
            __syncthreads();
            g1 = uniform(g0 + ((wave_words[4] + wave_words[5]) + (wave_words[6] + wave_words[7])));
            for (uint32_t r0 = 0; r0 < n; r0 += kBlock * 4)
            {
                RawRecord raw[4];
                load_records(a, raw, records(r0));
#pragma unroll
                for (int k = 0; k < 4; ++k)
                {
                    if (r0 + (uint32_t)(k * kBlock) >= n) break;
                    const FragmentRecord got = taken_apart(a, raw[k], pixels);
                    if (r0 + k * kBlock + tid < n && got.pixel >= g0 && got.pixel < g1) put(got, atomicAdd(&cursors[got.pixel], 1u));
                }
            }
        }
        __syncthreads();
        // every wave sorts a quarter of the lists
        const uint32_t per_wave = (g1 - g0 + 3u) / 4u;
        const uint32_t p0 = min(g0 + (uint32_t)wave * per_wave, g1), p1 = min(p0 + per_wave, g1);
        BinRoom mine = room;
        mine.t += wave * kWave, mine.alpha += wave * kWave, mine.depth += wave * kWave;
        uint32_t off = 0, length = 0;
        if (p0 + (uint32_t)lane < p1)
        {
            off    = room.places[p0 + lane];
            length = (room.places[p0 + lane + 1] - off) & 0xFFFFu;
        }
        sort_wave_lists(room.keys, reinterpret_cast<uint8_t*>(mine.t), off & 0xFFFFu, length, lane, a.K, /*skip_longer=*/(uint32_t)kBuildCap);
        if (!(a.K > 0 && a.K <= kWave))
        {
            // Lists that have to be sorted in full and are too long for a wave's registers: by the whole workgroup, one after the
            // other. (By the wave that has them, every step of the network in LDS, 300 to 800 fragments a pixel: 201 against 129 us,
            // with the 2x2 splat 113 against 49. From 128 on instead of 256: 134 and 48.)
            const uint64_t longer = __ballot(length > (uint32_t)(4 * kWave));
            if (lane == 0) lists_by_block[wave] = longer;
            __syncthreads();
            for (int w = 0; w < kBlock / kWave; ++w)  // the same trips for every thread
            {
                uint64_t todo = lists_by_block[w];
                while (todo != 0ull)
                {
                    const uint32_t px = g0 + (uint32_t)w * per_wave + (uint32_t)(__ffsll((unsigned long long)todo) - 1);
                    todo &= todo - 1ull;
                    const uint32_t at = room.places[px] & 0xFFFFu, behind = room.places[px + 1] & 0xFFFFu;
                    block_sort(room.keys + at, behind - at, opaque(threadIdx.x));
                }
            }
            __syncthreads();  // (the next run writes these masks)
        }
        if (g1 - g0 > (uint32_t)kWave)
        {
            wave_sync();
            if (p0 < p1) blend_steps<C, BILINEAR, FUZZY, 1, false>(a, place, mine, begin + run_start, p0, p1, lane);
        }
        else
        {
            __syncthreads();
            blend_steps<C, BILINEAR, FUZZY, kBlock / kWave, false>(a, place, room, begin + run_start, g0, g1, tid);
        }
        g0 = g1;
    }
}

// Consecutive workgroups run on different XCDs, each of which has its own L2. Turn k of the `all` crowded bins goes to place k of this
// order instead: of every kXcds * run places an XCD has `run` neighbouring ones, as far as whole groups of them go. What neighbouring bins
// share (lines of the images and of the lists, descriptors of one block of points) is then in one L2. Us of the pass, in turn / in
// runs: 2x2 splat at 1080p 223 / 220 (runs of 4: 214 where 16 took 211 on another card), dense cloud in it 451 / 441, ten million
// points 447 / 444, surfaces in 960x540 66 / 65, two views with the 2x2 splat 590 / 575. Uncrowded bins take runs of 8 in launches of more
// than kRunsFrom workgroups for them: 1237x701 (3560 of them) 35.8 / 34.4, with the 2x2 splat in 1279x719 54.9 / 53.7, ten million points
// 444 / 441; with fewer, neighbours that hold much are one XCD's and nobody else's: a town in 640x360 (3080) 19.4 / 20.1, four crops of 512x512 (1024)
// 278 / 281. How many there are comes as an argument: the size of the grid does not lie with the arguments, and waiting for
// it as well cost every launch 0.3 us (480x270 with three layers 16.9 / 17.2).
constexpr uint32_t kWaveBinRun = 8, kCrowdedRun = 16, kRunsFrom = 3200;
__device__ __forceinline__ uint32_t in_runs(uint32_t k, uint32_t all, uint32_t run)
{
    const uint32_t group = kXcds * run, first = k / group * group, in = k - first;
    return first + group <= all ? first + in % kXcds * run + in / kXcds : k;
}

template <int C, bool BILINEAR, bool FUZZY>
__device__ __forceinline__ void bin_build(BuildArgs& a)
{
    static_assert(!(BILINEAR && FUZZY), "one blend rule at a time");
    constexpr int kWaves = kBlock / kWave, kPlaces = kTilePixels + 4;
    static_assert(kWaves * kWaveBinCap <= kBuildCap && kWaves * kPlaces >= kPlaces + kBlock, "the waves share the workgroup's arrays");
    __shared__ uint64_t s_keys[kBuildCap];
    __shared__ float4 s_t[kBlock];
    __shared__ float s_alpha[kBlock];
    __shared__ float s_depth[kBlock];
    __shared__ __align__(16) uint32_t s_places[kWaves * kPlaces];
    __shared__ uint8_t s_items[kBuildCap];
    __shared__ uint32_t s_words[12];
    __shared__ uint64_t s_lists_by_block[kWaves];
    if (blockIdx.x < a.crowded_blocks)
    {
        const BinRoom room = {s_keys, s_places, s_items, s_t, s_alpha, s_depth};
        const uint32_t first = uniform(a.crowded_counts[0]), all = first + uniform(a.crowded_counts[1]);
        for (uint32_t turn = blockIdx.x; turn < all; turn += a.crowded_blocks)
        {
            const uint32_t k     = in_runs(turn, all, kCrowdedRun);
            const uint2 entry    = a.crowded[k < first ? k : a.crowded_capacity - 1u - (k - first)];
            const uint32_t bin   = uniform(entry.x), parts = uniform(entry.y);
            if (bin < a.num_bins)  // guard: never false
                build_by_workgroup<C, BILINEAR, FUZZY>(a, bin, parts & 0xFFFFu, parts >> 16, room, s_places + kPlaces, s_lists_by_block, s_words);
            __syncthreads();
        }
        return;
    }
    const int lane = threadIdx.x & (kWave - 1);
    const uint32_t wave = uniform(threadIdx.x / kWave);
    const BinRoom room  = {s_keys + wave * kWaveBinCap, s_places + wave * kPlaces, s_items + wave * kWaveBinCap,
                           s_t + wave * kWave, s_alpha + wave * kWave, s_depth + wave * kWave};
    const uint32_t bin  = in_runs(blockIdx.x - a.crowded_blocks, a.blocks_in_runs, kWaveBinRun) * kWaves + wave;
    if (bin < a.num_bins) build_by_wave<C, BILINEAR, FUZZY>(a, bin, room, lane);
}

// Waves of a SIMD unit to leave registers for: all the LDS lets in; with the state of a bucket one less.
template <bool FUZZY>
constexpr int kBuildWaves = FUZZY ? 7 : 8;

template <int C, bool BILINEAR, bool FUZZY = false>
__global__ void __launch_bounds__(kBlock, kBuildWaves<FUZZY>) bin_build_kernel(BuildPass)
{
    bin_build<C, BILINEAR, FUZZY>(*(BuildArgs*)__builtin_amdgcn_kernarg_segment_ptr());
}

template <int C, bool BILINEAR, bool FUZZY = false>
__global__ void __launch_bounds__(kBlock, kBuildWaves<FUZZY>) bin_build_views_kernel(PerView<BuildPass>)
{
    bin_build<C, BILINEAR, FUZZY>(((BuildArgs*)__builtin_amdgcn_kernarg_segment_ptr())[blockIdx.y]);
}

}  // namespace vetrast
