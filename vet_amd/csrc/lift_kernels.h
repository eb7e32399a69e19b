// Error lifting: the per-pixel error of one rendered view is added to every cell of the scene grid whose projected box
// covers the pixel (FillSceneGridWithLossRasterize, src/lib/rendering/RenderForward.cu:639-761).
//
// The reference gives every cell a warp that tests every pixel of the cell's box against the 12 face triangles. Most of
// those tests have a foregone answer: in one image row the pixels a cell covers are a run whose ends can be computed.
// So the work here goes by rows instead of pixels:
//   1. lift_prefix_kernel: per image row the running sum (double) of sum_c |loss|, so that the sum over a run of pixels is
//      one difference of two entries. Beside that, workgroups of their own look for the cells whose box the image shows.
//   2. lift_cells_kernel: a workgroup takes 32 of those cells, projects their corners and sets up, per triangle and for the
//      outline of the 8 corners, where their edges cross a row; then every lane takes one ROW of one of the cells. Pixels that
//      lie inside a triangle by more than the rounding error of the test are counted as a run, pixels outside the outline
//      by more than that are left out, and the few in between get the literal test of the reference. The counts are the
//      literal ones, pixel for pixel.
// Measured (146 k cells of 0.25 m, 1080p, 121 M covered pixels, the camera inside the grid): 0.87 ms per call with a test per
// pixel (bound by its ~200 vector instructions per 64 pixels), 0.20 ms by rows.
// Bound by vector instructions (32 M of wave instructions a view of three 1080p views of 176 k cells, 52 of the cells kernel's 86 us)
// and the round trips of a row's two running sums. A third of the cells is in the image: with the others in the workgroups too,
// set up by as many idle lanes, it took 43 M and 103 us, cells of 0.15 m 385 a call (now 259), of 1 m 78 (now 56: there are few of
// them, which are dealt to more workgroups then, kLiftLeast; with 768 or 1792 for it the same). Looking for them costs the running
// sums' kernel 1 us (13.4 and 14.2; 17.2 when every cell of a stretch came from a cache line of its own).
// The LDS of 7 workgroups (a bound is two floats; with three, 6 fit: 99 us). 16 cells to a workgroup 92 us, with 128 threads 112.
#pragma once
#include "common.h"
#include "forward_kernels.h"

namespace vetrast
{
constexpr int kLiftLargeCell    = 4096;  // boxes of more pixels are counted in the header (a diagnostic of the interface)
constexpr int kLiftHeader       = 256;   // bytes: DeviceView (160), the count of large cells at 176, flag word at 192
constexpr int kLiftBlock        = 256;   // threads of a workgroup of the cells kernel
constexpr int kLiftCells        = 32;    // its cells, at most
constexpr uint32_t kLiftLeast   = 1024;  // workgroups that take the cells, if there are so many
constexpr int kLiftSetup        = 4;     // threads that set a cell's triangles up, and as many its outline
constexpr int kLiftSetupAll     = kLiftCells * kLiftSetup;
static_assert(kLiftSetupAll % kWave == 0 && kLiftBlock >= 2 * kLiftSetupAll, "triangles and outlines are set up by different waves");
constexpr int kLiftTriangleMax  = 8;     // triangles that wind one way: three faces of a box, and one seen edge-on
constexpr int kLiftOutlineMax   = 8;     // edges of the outline that are kept: a box shows 6 at most
constexpr int kLiftSliverMax    = 8;     // thin triangles whose lines are looked at (the four side faces of a frontal box)
constexpr int kLiftRows         = 4;     // image rows per group of the running sums: 4 rows of one column share 32 bytes
constexpr float kLiftReach      = 5e4f;  // cells whose corners project further away than this (they all but touch the
                                         // camera plane) are tested pixel by pixel: rounding leaves whole strips open
constexpr int kLiftPlainShare   = 128;   // workgroups that share such a cell
constexpr int kLiftPlainAtOnce  = 8;     // cells in work at a time
constexpr float kLiftThin       = 0.05f; // smallest angle (about) of a triangle that is not a sliver
constexpr int kLiftOpen         = 8;     // open pixels of a row that go to the list; a row with more is left to a wave
constexpr int kLiftOpenPixels   = 128;   // the list of a wave; it is worked off when half full (a lane tests what does not fit)
constexpr uint32_t kLiftNone    = 0x80000000u;  // (there are no more than 2^30 cells)
constexpr uint32_t kLiftRun     = 4;     // neighbouring cells that go to one stretch together
constexpr int kLiftOpenRows     = 128;   // such rows a workgroup keeps (a lane finishes what does not fit)
// A cell whose open rows of more than kLiftWideRow columns add up to more than kLiftWideWork and more than one in
// kLiftWideShare of its box's pixels is tested pixel by pixel by lift_plain_kernel: next to the camera the lines of slivers
// sweep hundreds of columns in hundreds of rows, and the one workgroup that had such a cell held the launch up (three 1080p
// views, one of them like that: 1.61 ms of kernels, now 0.57 ms; with 1 m cells at 3840x2160, two bands of rows, 3.47 ms,
// now 1.92 ms). Limits of 64 and 128 columns a row and 1024 and 8192 in all measure the same within 5 % at 1080p, 32768 in
// all is slower by half there; without the share of the box, 0.25 m cells at 3840x2160 take 1.79 ms instead of 1.49 (a few
// wide rows are less work than all pixels of a large box), shares of 256 to 1024 measure the same.
constexpr int kLiftWideRow      = 256;
constexpr int kLiftWideWork     = 2048;
constexpr int kLiftWideShare    = 512;
constexpr size_t kLiftSums      = (size_t)1 << 22;  // running sums that exist at a time in a caller's workspace, at most
                                                    // (33.5 MB: an image of 4.2 M pixels); taller images take several bands
constexpr size_t kLiftStaticSums = (size_t)1 << 21; // the same in the library's own array (16.8 MB: a 1080p image)
static_assert(sizeof(DeviceView) <= VETRAST_LIFT_QUEUE_LENGTH_OFFSET && VETRAST_LIFT_QUEUE_LENGTH_OFFSET + 4 <= VETRAST_LIFT_FLAGS_OFFSET,
              "the header's three parts must not overlap");

struct LiftPass
{
    const float* bb_min;
    const float* bb_length;
    float* value;
    int32_t* access_count;
    const float* loss;  // [channels][height][width]
    int64_t num_cells;
    int channels, height, width, border;
    int y0, y1;         // image rows of this band (y0 a multiple of kLiftRows)
    int first, last;    // this band is the first / last of the call
    // workspace
    DeviceView* view;
    uint32_t* large_cells;
    uint32_t* flags;
    uint32_t* num_plain;    // cells left to lift_plain_kernel
    uint32_t* plain_cell;   // their numbers
    // [num_cells] each, written for cells left to lift_plain_kernel and, with several bands, for every cell that is seen:
    double* cell_sums;      // sum of the bands so far
    uint32_t* plain_state;  // 0, or first image row that is lift_plain_kernel's + 1 in bits 8.., below them its finished shares
    // Cells the image shows, found by the first band's lift_prefix_kernel. The cells are dealt to stretches, kLiftRun neighbours
    // at a time (lift_cell_of_stretch), and column k of stretch c is the place [k * stretches + c] of this array: the stretch's
    // cells that are seen, and in its last column kLiftNone | how many these are, unless all are.
    uint32_t* seen;         // [num_cells]
    uint32_t stretches;     // a multiple of kWave
    uint32_t prefix_groups; // workgroups of lift_prefix_kernel that add up
    double* sums;       // running sums of the band, see lift_sum_at; null: the image is too wide for one band to hold a row
};

// Workgroups that share the cells of a group of stretches.
__host__ __device__ __forceinline__ uint32_t lift_shares(uint32_t cells, uint32_t groups)
{
    const uint32_t full = (cells + kLiftCells - 1u) / kLiftCells, least = (kLiftLeast + groups - 1u) / groups;
    return full > least ? full : (cells < least ? cells : least);
}

// Where the sum of the pixels [0, x) of image row y is, 0 <= x <= width. The entry of x = 0 is zero, with the sign bit set
// where the row has pixels so dim that rounding may have swallowed them.
__device__ __forceinline__ size_t lift_sum_at(const LiftPass& a, int x, int y)
{
    const uint32_t r = (uint32_t)(y - a.y0);
    return ((size_t)(r / kLiftRows) * (size_t)(a.width + 1) + (size_t)x) * kLiftRows + r % kLiftRows;
}

__device__ __forceinline__ float lift_pixel_error(const LiftPass& a, int x, int y)
{
    float grad         = 0.f;
    const size_t plane = (size_t)a.height * a.width;
    const float* px    = a.loss + (size_t)y * a.width + x;
    for (int c = 0; c < a.channels; ++c) grad += fabsf(px[c * plane]);
    return grad;
}

// One workgroup of kLiftRows waves per group of kLiftRows rows: a wave scans its row 1024 pixels at a time (16 per lane),
// the 1024 x 4 block goes through LDS so that the stores are whole 32-byte groups. The first workgroup of a call also
// writes the camera constants of the view. Bound by the chain of steps along a row (1080p: 254 workgroups of 2
// steps; of 4 steps of 512 pixels three views take 6 us more).
constexpr int kLiftPrefixBlock = kLiftRows * kWave;
constexpr int kLiftPerLane     = 16;
constexpr int kLiftStep        = kLiftPerLane * kWave;

// Cell k of a stretch, or a number beyond the last cell. Neighbours share cache lines; what is left at the end is dealt one by one,
// so that a stretch has no more places than cells.
__device__ __forceinline__ uint32_t lift_cell_of_stretch(uint32_t k, uint32_t stretch, uint32_t stretches, uint32_t cells)
{
    const uint32_t in_runs = cells / (kLiftRun * stretches) * kLiftRun;  // cells of a stretch that come in runs
    return k < in_runs ? (k / kLiftRun * stretches + stretch) * kLiftRun + k % kLiftRun : k * stretches + stretch;
}

// Workgroup c of these takes stretch c of the cells, a thread per cell: is one of its corners behind the camera, or its pixel
// box outside the image (src/lib/rendering/RenderForward.cu:679-728)? The others are written down, turned by a share of their
// number that grows from stretch to stretch: cells of one column then lie all over the grid.
__device__ __forceinline__ void lift_find_cells(const LiftPass& a, const DeviceView& view, uint32_t stretch)
{
    __shared__ uint32_t s_seen[kLiftPrefixBlock / kWave];
    const uint32_t all  = (uint32_t)a.num_cells, cell = lift_cell_of_stretch(threadIdx.x, stretch, a.stretches, all);
    const uint32_t own  = threadIdx.x * a.stretches + stretch;  // the place of column threadIdx.x (these are all below 2^31)
    const int lane      = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    bool seen           = cell < all;
    if (seen)
    {
        const float* mn = a.bb_min + 3 * (size_t)cell;
        const float* ln = a.bb_length + 3 * (size_t)cell;
        const float m[3] = {mn[0], mn[1], mn[2]}, n[3] = {ln[0], ln[1], ln[2]};
        float max_x = -10000000.f, max_y = -10000000.f, min_x = 10000000.f, min_y = 10000000.f;
#pragma unroll
        for (int i = 0; i < 8; ++i)
        {
            float4 p;
            p.x = m[0] + n[0] * (float)(i & 1);
            p.y = m[1] + n[1] * (float)(i >> 1 & 1);
            p.z = m[2] + n[2] * (float)(i >> 2);
            p.w = 0.f;
            Projected o;
            if (!project_point(view, p, o))
            {
                seen = false;
                continue;
            }
            max_x = fmaxf(o.ipx, max_x), max_y = fmaxf(o.ipy, max_y);
            min_x = fminf(o.ipx, min_x), min_y = fminf(o.ipy, min_y);
        }
        const float border = (float)a.border, right = (float)(a.width - a.border), bottom = (float)(a.height - a.border);
        seen = seen && !(max_x < border || min_x >= right || max_y < border || min_y >= bottom);
    }
    const uint64_t here = __ballot(seen);
    if (lane == 0) s_seen[wave] = (uint32_t)__popcll(here);
    __syncthreads();
    uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(here >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)here, 0u)), found = 0;
    for (int w = 0; w < kLiftPrefixBlock / kWave; ++w)
    {
        if (w < wave) rank += s_seen[w];
        found += s_seen[w];
    }
    const uint32_t turn = stretch % kWave * found / kWave;
    if (seen)
    {
        const uint32_t column = rank + turn < found ? rank + turn : rank + turn - found;
        a.seen[column * a.stretches + stretch] = cell;
    }
    if (threadIdx.x >= found && own < all && own + a.stretches >= all) a.seen[own] = kLiftNone | found;
}

__global__ void __launch_bounds__(kLiftPrefixBlock) lift_prefix_kernel(LiftPass a, ViewSource src, const double* __restrict__ poses_se3,
                                                                       const float* __restrict__ intrinsics)
{
    // (a place is left free behind a lane's, or all lanes would store to one bank)
    __shared__ double s_sum[kLiftStep * kLiftRows + kWave];
    if (blockIdx.x >= a.prefix_groups)  // (the first band's only)
    {
        bool distorted = false;
        DeviceView v   = make_device_view(src, poses_se3, intrinsics, distorted);
        v.has_dist     = 0u;
        lift_find_cells(a, v, blockIdx.x - a.prefix_groups);
        return;
    }
    if (a.first && blockIdx.x == a.prefix_groups - 1u && threadIdx.x == kLiftPrefixBlock - 1)
    {
        bool distorted = false;
        DeviceView v   = make_device_view(src, poses_se3, intrinsics, distorted);
        v.has_dist     = 0u;  // cameras with distortion are refused here (the flag below)
        *a.view        = v;
        *a.large_cells = 0u;
        *a.num_plain   = 0u;
        *a.flags       = distorted ? 1u : 0u;
    }
    if (!a.sums) return;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int y      = a.y0 + (int)blockIdx.x * kLiftRows + wave;
    const bool row   = y < a.y1;
    double* group    = a.sums + (size_t)blockIdx.x * (size_t)(a.width + 1) * kLiftRows;
    const size_t plane = (size_t)a.height * a.width;
    const float* line  = a.loss + (size_t)(row ? y : a.y0) * a.width;
    const bool wide    = (a.width & 3) == 0 && (reinterpret_cast<uintptr_t>(a.loss) & 15) == 0;
    auto load = [&](int x, float (&g)[kLiftPerLane]) {
#pragma unroll
        for (int k = 0; k < kLiftPerLane; ++k) g[k] = 0.f;
        if (!row) return;
        for (int c = 0; c < a.channels; ++c)
        {
            if (wide)
            {
#pragma unroll
                for (int k = 0; k < kLiftPerLane; k += 4)
                    if (x + k < a.width)
                    {
                        const float4 v = *reinterpret_cast<const float4*>(line + c * plane + x + k);
                        g[k] += fabsf(v.x), g[k + 1] += fabsf(v.y), g[k + 2] += fabsf(v.z), g[k + 3] += fabsf(v.w);
                    }
            }
            else
            {
#pragma unroll
                for (int k = 0; k < kLiftPerLane; ++k)
                    if (x + k < a.width) g[k] += fabsf(line[c * plane + x + k]);
            }
        }
    };
    double carry     = 0.0;
    uint32_t dimmest = 0xFFFFFFFFu;  // smallest error of the lane's pixels that have one, as its bits less one
    float g[kLiftPerLane];
    load(kLiftPerLane * lane, g);
    for (int x0 = 0; x0 < a.width; x0 += kLiftStep)
    {
        float next[kLiftPerLane];
        load(x0 + kLiftStep + kLiftPerLane * lane, next);
        double p[kLiftPerLane];
        p[0] = (double)g[0];
#pragma unroll
        for (int k = 1; k < kLiftPerLane; ++k) p[k] = p[k - 1] + (double)g[k];
        const double own = p[kLiftPerLane - 1];
        double incl      = own;
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1)
        {
            const double up = __shfl_up(incl, d, kWave);
            if (lane >= d) incl += up;
        }
        const double before = carry + (incl - own);
        carry += __shfl(incl, kWave - 1, kWave);
        __syncthreads();  // the block of the step before has been stored
#pragma unroll
        for (int k = 0; k < kLiftPerLane; ++k)
        {
            s_sum[(kLiftPerLane * lane + k) * kLiftRows + wave + lane] = before + p[k];
            dimmest = min(dimmest, __float_as_uint(g[k]) - 1u);  // (no error: the largest number)
        }
        __syncthreads();
        const int columns = min(kLiftStep, a.width - x0);
        for (int k = threadIdx.x; k < columns * kLiftRows; k += kLiftPrefixBlock) group[(size_t)(x0 + 1) * kLiftRows + k] = s_sum[k + k / (kLiftPerLane * kLiftRows)];
#pragma unroll
        for (int k = 0; k < kLiftPerLane; ++k) g[k] = next[k];
    }
    // The empty run. Neighbouring entries are off by a few units in the last place of the row's sum, so a pixel of at least
    // 2^-48 of it shows in every difference; where one is dimmer, or the sum is not finite, the sign of the entry says that
    // it may not.
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) dimmest = min(dimmest, (uint32_t)__shfl_xor((int)dimmest, d, kWave));
    const bool all_show = dimmest == 0xFFFFFFFFu || (double)__uint_as_float(dimmest + 1u) >= carry * 0x1p-48;
    if (lane == 0) group[wave] = all_show ? 0.0 : -0.0;
}

// tris_indices of the reference (src/lib/rendering/RenderForward.cu:665-666): two triangles per face of the box, corner
// numbers packed 4 bits each, triangle t at bits 4 t.
//   {0,1,4} {0,4,2} {1,5,7} {1,7,4} {5,3,6} {5,6,7} {3,0,6} {0,6,2} {3,0,5} {0,5,1} {2,4,6} {4,6,7}
constexpr uint64_t kLiftFirst = 0x420303551100ull, kLiftSecond = 0x645060637541ull, kLiftThird = 0x761526764724ull;
// Triangles whose corners run the other way round than the rest's, seen from outside the box (one bit each). With those
// turned round, the triangles that wind one way on screen are the box's near (or far) side and cover all of its outline.
constexpr uint32_t kLiftInward = 0x67Fu;
// The 12 edges of the box: 0-1 0-2 0-3 1-4 1-5 2-4 2-6 3-5 3-6 4-7 5-7 6-7.
constexpr uint64_t kLiftEdgeFrom = 0x654332211000ull, kLiftEdgeTo = 0x777656454321ull;
__device__ __forceinline__ int nibble(uint64_t packed, int i) { return (int)(packed >> (4 * i)) & 15; }

// sign() and PointInTriangle() of src/lib/rendering/RenderForward.cu:605-625.
__device__ __forceinline__ float edge_sign(float p1x, float p1y, float p2x, float p2y, float p3x, float p3y)
{
    return (p1x - p3x) * (p2y - p3y) - (p2x - p3x) * (p1y - p3y);
}

__device__ __forceinline__ bool point_in_triangle(float x, float y, float ax, float ay, float bx, float by, float cx,
                                                  float cy)
{
    const float d1     = edge_sign(x, y, ax, ay, bx, by);
    const float d2     = edge_sign(x, y, bx, by, cx, cy);
    const float d3     = edge_sign(x, y, cx, cy, ax, ay);
    // has_neg = one of them < 0, has_pos = one of them > 0; fminf / fmaxf drop a NaN like the comparisons do
    const bool has_neg = fminf(fminf(d1, d2), d3) < 0.f;
    const bool has_pos = fmaxf(fmaxf(d1, d2), d3) > 0.f;
    return !(has_neg && has_pos);
}

// Screen footprint of a cell that is tested pixel by pixel, identical in every lane of the wave that computed it.
struct CellFootprint
{
    float px[8], py[8];  // projected corners
    float min_x, min_y;  // clamped pixel box origin
    int x_size, y_size;
};

// Lanes 0..7 of the calling wave project one corner each (src/lib/rendering/RenderForward.cu:679-704); the pixel box of
// the projections is cut to the image minus the border (:706-728). The cell is known to take part. All lanes must call.
__device__ __forceinline__ void cell_footprint(const LiftPass& a, int64_t cell, int lane, CellFootprint& f)
{
    float ipx = 0.f, ipy = 0.f;
    if (lane < 8)
    {
        const int fx = (0xB2 >> lane) & 1, fy = (0xD4 >> lane) & 1, fz = (0xE8 >> lane) & 1;
        const float* mn = a.bb_min + 3 * cell;
        const float* ln = a.bb_length + 3 * cell;
        float4 p;
        p.x = mn[0] + ln[0] * (float)fx;
        p.y = mn[1] + ln[1] * (float)fy;
        p.z = mn[2] + ln[2] * (float)fz;
        p.w = 0.f;
        Projected o;
        if (project_point(*a.view, p, o)) ipx = o.ipx, ipy = o.ipy;
    }
    float max_x = -10000000.f, max_y = -10000000.f, min_x = 10000000.f, min_y = 10000000.f;
#pragma unroll
    for (int i = 0; i < 8; ++i)
    {
        f.px[i] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, ipx), i));
        f.py[i] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, ipy), i));
        max_x   = fmaxf(f.px[i], max_x);
        max_y   = fmaxf(f.py[i], max_y);
        min_x   = fminf(f.px[i], min_x);
        min_y   = fminf(f.py[i], min_y);
    }
    const float border = (float)a.border;
    f.min_x  = fmaxf(min_x, border);
    f.min_y  = fmaxf(min_y, border);
    f.y_size = (int)(fminf(max_y, (float)(a.height - a.border)) - f.min_y);
    f.x_size = (int)(fminf(max_x, (float)(a.width - a.border)) - f.min_x);
}

// A bound on x in an image row: x >= or <= slope * (row - the cell's first row) + x0.
struct RowBound
{
    float slope, x0;
    __device__ __forceinline__ float at(float row) const { return slope * row + x0; }
};
// The same through a point (x0, y0), as it is set up.
struct LineBound
{
    float slope, y0, x0;
    // Moved to the cell's first row, and by what that and evaluating it there may be off in x, to the larger or the smaller side. That
    // is below 5 units in the last place of slope times the height of the box: as if the edge lay 8 of them, 2^-21 of the height,
    // higher or lower.
    __device__ __forceinline__ float off(float height) const { return fabsf(slope) * (height * 4.7683716e-7f); }
    __device__ __forceinline__ RowBound from(float first_row, float height, bool larger) const
    {
        const float moved = off(height);
        return {slope, (slope * (first_row - y0) + x0) + (larger ? moved : -moved)};
    }
};

struct LiftCell
{
    float px[8], py[8];  // projected corners
    float min_y;         // clamped box origin
    int xs, xe;          // first and last pixel column of the box
    int x_skip;          // a column between them that the reference's rounding of column + origin passes over, or INT_MAX
    RowBound outline[kLiftOutlineMax];
    RowBound tri[kLiftTriangleMax][3];                        // per triangle: a left, a right bound and one of either kind
    RowBound sliver[kLiftSliverMax];     // lines of thin triangles (x0 is the image row of one that is flat), and
    float sliver_width[kLiftSliverMax];  // their half width in columns, or -(half width in rows)
    uint32_t left_mask;                  // bit t: the third bound of triangle t is a left one; bit 8 + k: outline[k] is
    int num_outline, num_tri, num_sliver;
    int wide;      // columns of the wide open rows less the limit; above 0: the cell is lift_plain_kernel's
    int count;
    double sum;
};

// Bounds of the half-plane c1 (x - bx) - dx (y - by) >= e0. False where the edge is so flat that the bound says nothing
// about a single row.
__device__ __forceinline__ bool half_plane(float c1, float dx, float bx, float by, float e0, float flat, LineBound& r,
                                           bool& is_left)
{
    if (fabsf(c1) <= flat) return false;
    r.slope   = dx / c1;
    r.y0      = by;
    r.x0      = bx + e0 / c1;
    is_left = c1 > 0.f;
    return true;
}

// Is pixel (x, y) in one of the 12 triangles? The literal test, for the pixels the bounds leave open.
template <class Corners>
__device__ __forceinline__ bool in_any_triangle(const Corners& f, float x, float y)
{
#pragma unroll 1
    for (int t = 0; t < 12; ++t)
    {
        const int i = nibble(kLiftFirst, t), j = nibble(kLiftSecond, t), k = nibble(kLiftThird, t);
        if (point_in_triangle(x, y, f.px[i], f.py[i], f.px[j], f.py[j], f.px[k], f.py[k])) return true;
    }
    return false;
}

// Sum of the pixels [x0, x1) of row y. The difference of two running sums is taken where it keeps its bits: an entry is
// off by 2^-50 of itself or so, so a run of at least 2^-12 of what lies in front of it is good to 38 bits, 14 more than the
// float it ends in. Dimmer runs (also those behind a pixel that is not finite) are added up pixel by pixel; a difference
// of zero is a run without any error where the row has no pixel that rounding could swallow.
__device__ __forceinline__ double lift_run_sum(const LiftPass& a, int x0, int x1, int y)
{
    if (a.sums)
    {
        const double lo = a.sums[lift_sum_at(a, x0, y)], s = a.sums[lift_sum_at(a, x1, y)] - lo;
        if (s >= lo * 0x1p-12) return s;
        if (s == 0.0 && !__builtin_signbit(a.sums[lift_sum_at(a, 0, y)])) return 0.0;
    }
    double s = 0.0;
    for (int x = x0; x < x1; ++x) s += (double)lift_pixel_error(a, x, y);
    return s;
}

// Leaves the rows of a cell from this band on to lift_plain_kernel (a few cells of a grid, once per call). `sum`: what the
// bands in front of it have added up.
__device__ __forceinline__ void leave_to_plain_kernel(const LiftPass& a, int64_t cell, double sum)
{
    a.plain_cell[atomicAdd(a.num_plain, 1u)] = (uint32_t)cell;
    a.cell_sums[cell]   = sum;
    a.plain_state[cell] = (uint32_t)(a.y0 + 1) << 8;  // (an image has less than 2^24 rows)
}

// The cells of share `part` of a group of kWave neighbouring stretches: their cells that are seen, one stretch's after the
// other's, are dealt to as many shares as they fill, every so many-th of them to one, or to more where there are few cells.
// False if there is no such share. Every thread of the workgroup must call.
__device__ __forceinline__ bool lift_cells_of_share(const LiftPass& a, uint32_t group, uint32_t part, uint32_t (&cells)[kLiftCells])
{
    const uint32_t lane = threadIdx.x & (kWave - 1), all = (uint32_t)a.num_cells, stretch = group * kWave + lane;
    const uint32_t columns = stretch < all ? (all - stretch + a.stretches - 1u) / a.stretches : 0u;
    uint32_t found         = 0u;
    if (columns != 0u)
    {
        const uint32_t last = a.seen[(columns - 1u) * a.stretches + stretch];
        found               = (last & kLiftNone) != 0u ? last & ~kLiftNone : columns;
    }
    const uint32_t behind = wave_inclusive_scan(found, (int)lane);  // place behind the last of the lane's stretch
    const uint32_t total  = (uint32_t)__builtin_amdgcn_readlane((int)behind, kWave - 1);
    const uint32_t shares = lift_shares(total, a.stretches / kWave);
    if (part >= shares) return false;  // (the same for all waves)
    const uint32_t at = part + lane * shares;
    uint32_t of       = 0u;  // stretches that end in front of place `at`
#pragma unroll
    for (uint32_t step = kWave / 2; step >= 1u; step >>= 1)
        if ((uint32_t)__shfl((int)behind, (int)(of + step - 1u), kWave) <= at) of += step;
    const uint32_t column = at - ((uint32_t)__shfl((int)behind, (int)of, kWave) - (uint32_t)__shfl((int)found, (int)of, kWave));
    if (threadIdx.x < kLiftCells) cells[threadIdx.x] = at < total ? a.seen[column * a.stretches + group * kWave + of] : kLiftNone;
    return true;
}

__global__ void __launch_bounds__(kLiftBlock) lift_cells_kernel(LiftPass a)
{
    __shared__ LiftCell s_cell[kLiftCells];
    __shared__ int s_start[kLiftCells + 1];  // rows of the cells in front
    __shared__ int4 s_open[kLiftOpenRows];   // slot, y, columns [z, w)
    __shared__ uint2 s_pixel[kLiftBlock / kWave][kLiftOpenPixels];  // open pixels of a wave: x | slot << 24, y
    __shared__ int s_num_open, s_num_pixels[kLiftBlock / kWave];
    __shared__ uint32_t s_large;
    __shared__ bool s_left[kLiftCells];  // the cell is lift_plain_kernel's
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    __shared__ uint32_t s_cells[kLiftCells];  // cells of the workgroup, or kLiftNone
    const uint32_t groups = a.stretches / kWave;
    if (!lift_cells_of_share(a, blockIdx.x % groups, blockIdx.x / groups, s_cells)) return;
    if (lane == 0) s_num_pixels[wave] = 0;
    if (tid == 0) s_num_open = 0, s_large = 0u;
    __syncthreads();
    // ---- set-up: kLiftSetup threads per cell for its triangles, as many in other waves for its outline; both look at the box
    // first. The workgroup's cells are seen, all of them, and lie far apart in the grid (cells next to the camera cover hundreds of
    // rows and are neighbours in it), so every workgroup gets about the same number of rows.
    const bool outlines = tid >= kLiftSetupAll;  // the same in a wave
    const int slot = tid / kLiftSetup % kLiftCells, part = tid % kLiftSetup;
    bool seen      = false;
    float raw_x0 = 0.f, raw_x1 = 0.f, raw_y0 = 0.f, raw_y1 = 0.f, bottom_y = 0.f, first_x = 0.f, last_x = 0.f;  // of the box
    if (tid < 2 * kLiftSetupAll)
    {
        LiftCell& f        = s_cell[slot];
        const uint32_t cell = s_cells[slot];
        const bool left    = !a.first && cell != kLiftNone && a.plain_state[cell] != 0u;  // by an earlier band
        bool behind        = cell == kLiftNone || left;
        float max_x = -10000000.f, max_y = -10000000.f, min_x = 10000000.f, min_y = 10000000.f;
        float far = 0.f;  // largest coordinate
        if (!behind)
        {
            const float* mn = a.bb_min + 3 * (size_t)cell;
            const float* ln = a.bb_length + 3 * (size_t)cell;
            const float m[3] = {mn[0], mn[1], mn[2]}, n[3] = {ln[0], ln[1], ln[2]};
#pragma unroll
            for (int u = 0; u < 8 / kLiftSetup; ++u)
            {
                const int i = part * (8 / kLiftSetup) + u;
                // corner order of bb_facs: 000 100 010 001 110 101 011 111
                const int fx = (0xB2 >> i) & 1, fy = (0xD4 >> i) & 1, fz = (0xE8 >> i) & 1;
                float4 p;
                p.x = m[0] + n[0] * (float)fx;
                p.y = m[1] + n[1] * (float)fy;
                p.z = m[2] + n[2] * (float)fz;
                p.w = 0.f;
                Projected o;
                if (!project_point(*a.view, p, o))
                {
                    behind = true;
                    continue;
                }
                if (!outlines) f.px[i] = o.ipx, f.py[i] = o.ipy;
                max_x   = fmaxf(o.ipx, max_x);
                max_y   = fmaxf(o.ipy, max_y);
                min_x   = fminf(o.ipx, min_x);
                min_y   = fminf(o.ipy, min_y);
                far     = (fabsf(o.ipx) < kLiftReach && fabsf(o.ipy) < kLiftReach) ? far : 1.f;  // also where one of them is NaN
            }
        }
        static_assert(kLiftSetup == 4, "the exchanges below run over groups of four lanes");
        auto all4 = [&](auto op, float v) {
            v = op(v, __uint_as_float(lane_xor<1>(__float_as_uint(v), lane)));
            return op(v, __uint_as_float(lane_xor<2>(__float_as_uint(v), lane)));
        };
        auto larger  = [](float x, float y) { return fmaxf(x, y); };
        auto smaller = [](float x, float y) { return fminf(x, y); };
        max_x = all4(larger, max_x), max_y = all4(larger, max_y);
        min_x = all4(smaller, min_x), min_y = all4(smaller, min_y);
        const bool plain = all4(larger, far) != 0.f;
        const bool gone  = ((__ballot(behind) >> (lane & ~3)) & 15ull) != 0ull;
        // the pixel box, cut to the image minus the border (src/lib/rendering/RenderForward.cu:706-728)
        const float border = (float)a.border;
        const float right  = (float)(a.width - a.border);
        const float bottom = (float)(a.height - a.border);
        raw_x0 = min_x, raw_x1 = max_x, raw_y0 = min_y, raw_y1 = max_y;
        seen      = !gone && !(max_x < border || min_x >= right || max_y < border || min_y >= bottom);
        min_x     = fmaxf(min_x, border);
        min_y     = fmaxf(min_y, border);
        max_x     = fminf(max_x, right);
        max_y     = fminf(max_y, bottom);
        const int x_size = seen ? (int)(max_x - min_x) : 0, y_size = seen ? (int)(max_y - min_y) : 0;
        seen             = x_size > 0 && y_size > 0;
        const bool large = !outlines && part == 0 && seen && x_size * y_size > kLiftLargeCell;
        const bool leaves = seen && plain;  // (in the first band: the corners say so)
        if (leaves) seen = false;
        bottom_y = max_y;
        if (seen) first_x = (float)(int)min_x, last_x = (float)(int)((float)(x_size - 1) + min_x);
        if (!outlines && part == 0)
        {
            if (leaves) leave_to_plain_kernel(a, cell, 0.0);
            s_left[slot]  = leaves || left;
            s_start[slot] = seen ? y_size : 0;
            f.wide        = -max(kLiftWideWork, x_size * y_size / kLiftWideShare);
            f.count       = 0;
            f.sum         = 0.0;
            f.left_mask = 0u;
            f.num_outline = f.num_tri = f.num_sliver = 0;
            if (seen)
            {
                // column number -> pixel is int(float(column) + min_x). Adding a larger column may round up to the next
                // integer from some column on: then one pixel is passed over.
                f.min_y    = min_y;
                f.xs       = (int)min_x;
                f.xe       = (int)((float)(x_size - 1) + min_x);
                int x_skip = 0x7FFFFFFF;
                if (f.xe - f.xs != x_size - 1)
                {
                    int lo = 0, hi = x_size - 1;  // column lo lands on xs + lo, column hi does not
                    while (hi - lo > 1)
                    {
                        const int mid = (lo + hi) / 2;
                        if ((int)((float)mid + min_x) == f.xs + mid)
                            lo = mid;
                        else
                            hi = mid;
                    }
                    x_skip = f.xs + hi;
                }
                f.x_skip = x_skip;
            }
        }
        const uint64_t large_here = __ballot(large);
        if (a.first && large_here != 0ull && lane == 0) atomicAdd(&s_large, (uint32_t)__popcll(large_here));
    }
    __syncthreads();
    {
        LiftCell& f = s_cell[slot];
        if (seen)
        {
            // Rounding error of edge_sign at any pixel of the box: four roundings of two products, each bounded by the
            // extents; twice that.
            const float border = (float)a.border;
            const float xs = first_x, xe = last_x, ys = border > raw_y0 ? border : raw_y0;
            const float reach_x = fmaxf(fmaxf(raw_x1, xe) - fminf(raw_x0, xs), 1.f);
            const float reach_y = fmaxf(fmaxf(raw_y1, bottom_y) - fminf(raw_y0, ys), 1.f) + 1.f;
            const float err     = 16.f * 5.9604645e-8f * (2.f * reach_x * reach_y);
            // The same as a distance, and how far beyond a corner rounding can still see a triangle: the test accepts the
            // triangle with its edges moved out by `moved` at most, whose corners lie 2 / angle times as far out. That
            // covers angles down to kLiftThin; thinner triangles have a line of their own (below).
            const float moved   = 8.f * 5.9604645e-8f * fmaxf(reach_x, reach_y);
            const float margin  = 2.4f / kLiftThin * moved;
            const float slack   = 16.f * 5.9604645e-8f * (reach_x + xe);  // of RowBound::at inside the box, in pixels
            const float flat    = 1e-6f * reach_x;
#pragma unroll
            for (int u = 0; u < 12 / kLiftSetup; ++u)
            {
                const int t = part * (12 / kLiftSetup) + u;
                // a triangle that winds one way, by enough: rows of pixels that are inside it whatever the rounding
                if (!outlines)
                {
                    const int swap = (kLiftInward >> t) & 1;
                    const int v[3] = {nibble(kLiftFirst, t), nibble(swap ? kLiftThird : kLiftSecond, t), nibble(swap ? kLiftSecond : kLiftThird, t)};
                    float x[3], y[3];
#pragma unroll
                    for (int k = 0; k < 3; ++k) x[k] = f.px[v[k]], y[k] = f.py[v[k]];
                    const float area = edge_sign(x[0], y[0], x[1], y[1], x[2], y[2]);  // twice the area, signed
                    float longest = 0.f;
                    int at_longest = 0;
#pragma unroll
                    for (int k = 0; k < 3; ++k)
                    {
                        const float ex = x[k] - x[(k + 1) % 3], ey = y[k] - y[(k + 1) % 3], square = ex * ex + ey * ey;
                        at_longest = square > longest ? k : at_longest;
                        longest    = fmaxf(longest, square);
                    }
                    if (!(fabsf(area) >= kLiftThin * longest))
                    {
                        // A sliver may be seen by rounding far beyond its tips, but only on the line of its longest edge.
                        const float bx = at_longest == 0 ? x[1] : at_longest == 1 ? x[2] : x[0];
                        const float by = at_longest == 0 ? y[1] : at_longest == 1 ? y[2] : y[0];
                        const float ax = at_longest == 0 ? x[0] : at_longest == 1 ? x[1] : x[2];
                        const float ay = at_longest == 0 ? y[0] : at_longest == 1 ? y[1] : y[2];
                        LineBound r;
                        RowBound line;
                        bool is_left;
                        float half_width;
                        const float c1 = ay - by, dx = ax - bx;
                        if (half_plane(c1, dx, bx, by, 0.f, flat, r, is_left))
                            half_width = (err / fabsf(c1) + slack) + 2.f * r.off(reach_y), line = r.from(f.min_y, reach_y, true);
                        else
                            line = {0.f, by}, half_width = -(err + flat * reach_x) / fmaxf(fabsf(dx), 1e-12f);
                        const int at = atomicAdd(&f.num_sliver, 1);
                        if (at < kLiftSliverMax) f.sliver[at] = line, f.sliver_width[at] = half_width;
                    }
                    if (area > 4.f * err)
                    {
                        RowBound bound[3];  // a left one, a right one, one of either kind
                        bool have_left = false, have_right = false, third_is_left = true;
                        bound[0] = {0.f, -1e9f};
                        bound[1] = {0.f, 1e9f};
                        bound[2] = {0.f, -1e9f};
#pragma unroll
                        for (int k = 0; k < 3; ++k)
                        {
                            const float bx = x[(k + 1) % 3], by = y[(k + 1) % 3], c1 = y[k] - by, dx = x[k] - bx;
                            LineBound r;
                            bool is_left = true;
                            if (half_plane(c1, dx, bx, by, err, flat, r, is_left))
                                r.x0 += is_left ? slack : -slack;
                            else
                            {
                                // A flat edge: rows beyond it are all right, rows before it are all wrong. It can be a left
                                // or a right bound alike. It takes the first that is free, so that no bound is lost: at most
                                // two of the other edges bound from one side, and only one where there is a flat edge (the
                                // c1 of the three edges sum up to zero, and two of one sign to more than a flat edge has).
                                const float beyond = (err + flat * reach_x) / fmaxf(fabsf(dx), 1e-12f);
                                r.slope   = dx < 0.f ? -1e12f : 1e12f;
                                r.y0      = dx < 0.f ? by + beyond : by - beyond;
                                r.x0      = 1e7f;  // (beyond any column; one part in 1e5 of a row further it is -infinity)
                                is_left   = !have_left || have_right;
                                if (!is_left) r.slope = -r.slope, r.x0 = -r.x0;
                            }
                            const RowBound b = r.from(f.min_y, reach_y, is_left);
                            if (is_left && !have_left)
                                bound[0] = b, have_left = true;
                            else if (!is_left && !have_right)
                                bound[1] = b, have_right = true;
                            else
                                bound[2] = b, third_is_left = is_left;
                        }
                        const int at = atomicAdd(&f.num_tri, 1);
                        if (at < kLiftTriangleMax)
                        {
#pragma unroll
                            for (int k = 0; k < 3; ++k) f.tri[at][k] = bound[k];
                            if (third_is_left) atomicOr(&f.left_mask, 1u << at);
                        }
                    }
                }
                // a box edge with all corners on one side of it: part of the outline, moved out past every corner
                else
                {
                    const int i = nibble(kLiftEdgeFrom, t), j = nibble(kLiftEdgeTo, t);
                    const float bx = f.px[j], by = f.py[j], c1 = f.py[i] - by, dx = f.px[i] - bx;
                    float lowest = 0.f, highest = 0.f;
#pragma unroll
                    for (int k = 0; k < 8; ++k)
                    {
                        const float e = (f.px[k] - bx) * c1 - dx * (f.py[k] - by);
                        lowest        = fminf(lowest, e);
                        highest       = fmaxf(highest, e);
                    }
                    const float near = 8.f * err + 0.01f * (fabsf(c1) + fabsf(dx));
                    const float out  = margin * (fabsf(c1) + fabsf(dx)) + 4.f * err;
                    LineBound r;
                    bool is_left;
                    auto keep = [&]() {
                        r.x0 += is_left ? -slack : slack;
                        const int at = atomicAdd(&f.num_outline, 1);
                        if (at >= kLiftOutlineMax) return;
                        f.outline[at] = r.from(f.min_y, reach_y, !is_left);
                        if (is_left) atomicOr(&f.left_mask, 256u << at);
                    };
                    if (lowest > -near && half_plane(c1, dx, bx, by, lowest - out, flat, r, is_left)) keep();
                    if (highest < near && half_plane(-c1, -dx, bx, by, -highest - out, flat, r, is_left)) keep();
                }
            }
        }
    }
    __syncthreads();
    if (tid == 0 && s_large != 0u) atomicAdd(a.large_cells, s_large);
    if (tid < kWave)
    {
        const uint32_t rows = tid < kLiftCells ? (uint32_t)s_start[tid] : 0u;
        const uint32_t incl = wave_inclusive_scan(rows, tid);
        if (tid < kLiftCells) s_start[tid] = (int)(incl - rows);
        if (tid == kWave - 1) s_start[kLiftCells] = (int)incl;
    }
    __syncthreads();
    // ---- rows: a lane per row of a cell
    const int total = s_start[kLiftCells];
    auto test_pixel = [&](LiftCell& f, int x, int y) {
        if (!in_any_triangle(f, (float)x, (float)y)) return;
        atomicAdd(&f.count, 1);
        atomicAdd(&f.sum, (double)lift_pixel_error(a, x, y));
    };
    auto do_row = [&](int r) {
        int slot = 0;  // last cell that starts at or in front of row r
#pragma unroll
        for (int step = kLiftCells / 2; step >= 1; step >>= 1)
            if (s_start[slot + step] <= r) slot += step;
        LiftCell& f = s_cell[slot];
        const int y = (int)((float)(r - s_start[slot]) + f.min_y);
        // the box lies inside the bordered image by construction; the guard keeps a row outside the band from being read
        if (y < a.y0 || y >= a.y1) return;
        const float fy = (float)y, row = fy - f.min_y;
        // columns that may be covered
        const uint32_t left_mask = f.left_mask;
        float lo = (float)f.xs, hi = (float)f.xe;
        const int edges = f.num_sliver <= kLiftSliverMax ? min(f.num_outline, kLiftOutlineMax) : 0;
        for (int k = 0; k < edges; ++k)
        {
            const float v    = f.outline[k].at(row);
            const bool left  = (left_mask >> (8 + k)) & 1u;
            lo = fmaxf(lo, left ? v : lo);
            hi = fminf(hi, left ? hi : v);
        }
        int x     = (int)ceilf(fminf(lo, 1e8f));
        int x_end = (int)floorf(fmaxf(hi, -1e8f)) + 1;
        for (int k = 0; k < min(f.num_sliver, kLiftSliverMax); ++k)
        {
            const RowBound line = f.sliver[k];
            const float width   = f.sliver_width[k];
            if (width >= 0.f)
            {
                const float v = line.at(row);
                const float c0 = fmaxf(ceilf(v - width), (float)f.xs), c1 = fminf(floorf(v + width), (float)f.xe);
                if (c0 <= c1)  // (an empty range grows to the columns of the line)
                {
                    x_end = x < x_end ? max(x_end, (int)c1 + 1) : (int)c1 + 1;
                    x     = min(x, (int)c0);
                }
            }
            else if (fabsf(fy - line.x0) <= -width)
                x = f.xs, x_end = f.xe + 1;
        }
        if (x >= x_end) return;
        // columns that are covered for certain, triangle by triangle
        int from[kLiftTriangleMax], to[kLiftTriangleMax];
        const int triangles = min(f.num_tri, kLiftTriangleMax);
#pragma unroll
        for (int t = 0; t < kLiftTriangleMax; ++t)
        {
            from[t] = 0x7FFFFFFF, to[t] = 0;
            if (t < triangles)
            {
                const float v = f.tri[t][2].at(row);
                float l = f.tri[t][0].at(row), h = f.tri[t][1].at(row);
                if ((left_mask >> t) & 1u)
                    l = fmaxf(l, v);
                else
                    h = fminf(h, v);
                from[t] = (int)ceilf(fminf(fmaxf(l, -1e8f), 1e8f));
                to[t]   = (int)floorf(fminf(fmaxf(h, -1e8f), 1e8f)) + 1;
            }
        }
        const int x_first = x;
        int open          = 0;  // pixels the bounds leave open
        int count         = 0;
        double sum        = 0.0;
        uint32_t open_x[kLiftOpen];
        while (x < x_end)  // x grows with every turn
        {
            int next = x;
#pragma unroll
            for (int t = 0; t < kLiftTriangleMax; ++t)
                if (from[t] <= x) next = max(next, to[t]);
            next = min(next, x_end);
            if (f.x_skip >= x) next = min(next, f.x_skip);
            if (next > x)
            {
                // (bounds of two triangles often meet without a gap: on to the end of the run)
                int end = next;
                do
                {
                    next = end;
#pragma unroll
                    for (int t = 0; t < kLiftTriangleMax; ++t)
                        if (from[t] <= next) end = max(end, to[t]);
                    end = min(end, x_end);
                    if (f.x_skip >= next) end = min(end, f.x_skip);
                } while (end > next);
                count += next - x;
                sum += lift_run_sum(a, x, next, y);
            }
            else
            {
                if (x != f.x_skip)
                {
#pragma unroll
                    for (int k = 0; k < kLiftOpen; ++k)
                        if (open == k) open_x[k] = (uint32_t)x;
                    if (++open > kLiftOpen) break;
                }
                next = x + 1;
            }
            x = next;
        }
        if (open > kLiftOpen)
        {
            const int width = x_end - x_first;
            if (width > kLiftWideRow && atomicAdd(&f.wide, width) + width > 0) return;
            const int at = atomicAdd(&s_num_open, 1);
            if (at < kLiftOpenRows)
            {
                s_open[at] = make_int4(slot, y, x_first, x_end);  // a wave starts over
                return;
            }
            for (x = x_first; x < x_end; ++x)  // no room: the literal test for all of the row
                if (x != f.x_skip) test_pixel(f, x, y);
            return;
        }
        if (open > 0)
        {
            const int at = atomicAdd(&s_num_pixels[wave], open);
#pragma unroll
            for (int k = 0; k < kLiftOpen; ++k)
                if (k < open)
                {
                    if (at + k < kLiftOpenPixels)
                        s_pixel[wave][at + k] = make_uint2(open_x[k] | ((uint32_t)slot << 24), (uint32_t)y);
                    else
                        test_pixel(f, (int)open_x[k], y);
                }
        }
        if (count > 0)
        {
            atomicAdd(&f.count, count);
            atomicAdd(&f.sum, sum);
        }
    };
    auto wave_sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    for (int r0 = wave * kWave; r0 < total; r0 += kLiftBlock)
    {
        if (r0 + lane < total) do_row(r0 + lane);
        wave_sync();
        const int pixels = s_num_pixels[wave];
        if (pixels >= kLiftOpenPixels / 2 || (r0 + kLiftBlock >= total && pixels > 0))
        {
            for (int k = lane; k < min(pixels, kLiftOpenPixels); k += kWave)
            {
                const uint2 v = s_pixel[wave][k];
                test_pixel(s_cell[v.x >> 24], (int)(v.x & 0xFFFFFFu), (int)v.y);
            }
            wave_sync();
            if (lane == 0) s_num_pixels[wave] = 0;
        }
        wave_sync();
    }
    __syncthreads();
    // ---- rows with many open pixels (next to the line of a face seen edge-on, in cells that touch the camera plane)
    for (int k = wave; k < min(s_num_open, kLiftOpenRows); k += kLiftBlock / kWave)
    {
        const int4 row = s_open[k];
        LiftCell& f    = s_cell[row.x];
        if (f.wide > 0) continue;
        int count      = 0;
        double sum     = 0.0;
        for (int x = row.z + lane; x < row.w; x += kWave)
            if (x != f.x_skip && in_any_triangle(f, (float)x, (float)row.y))
            {
                ++count;
                sum += (double)lift_pixel_error(a, x, row.y);
            }
#pragma unroll
        for (int d = kWave / 2; d >= 1; d >>= 1) count += __shfl_xor(count, d, kWave), sum += __shfl_xor(sum, d, kWave);
        if (lane == 0 && count > 0)
        {
            atomicAdd(&f.count, count);
            atomicAdd(&f.sum, sum);
        }
    }
    __syncthreads();
    if (tid < kLiftCells)
    {
        const uint32_t cell = s_cells[tid];
        if (cell == kLiftNone || s_left[tid]) return;
        const double in_front = a.first ? 0.0 : a.cell_sums[cell];
        if (s_cell[tid].wide > 0)
        {
            leave_to_plain_kernel(a, cell, in_front);
            return;
        }
        const double sum = s_cell[tid].sum + in_front;
        const int count  = s_cell[tid].count;
        if (!a.last) a.cell_sums[cell] = sum;
        if (a.first && !a.last) a.plain_state[cell] = 0u;
        if (count > 0) a.access_count[cell] += count;
        // one rounding per call: the float terms of a cell are summed in double
        if (a.last && (count > 0 || in_front != 0.0)) a.value[cell] = (float)((double)a.value[cell] + sum);
    }
}

// The cells the rows were not made for: kLiftPlainShare workgroups per cell, each every kLiftPlainShare-th row of its box
// (from the band on that left it here), a thread per pixel. The last one to finish adds the cell's sum, with one rounding,
// to its value. The list is empty or a few cells long; the launch is fixed.
__global__ void __launch_bounds__(kBlock) lift_plain_kernel(LiftPass a)
{
    __shared__ double s_sum[kBlock / kWave];
    __shared__ int s_count[kBlock / kWave];
    __shared__ CellFootprint s_f;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const uint32_t cells = *a.num_plain;
    for (uint32_t k = blockIdx.y; k < cells; k += kLiftPlainAtOnce)
    {
        const int64_t cell = (int64_t)a.plain_cell[k];
        const int from     = (int)(a.plain_state[cell] >> 8) - 1;  // the rows in front of it are in the sum
        if (wave == 0)
        {
            CellFootprint f;
            cell_footprint(a, cell, lane, f);
            if (lane == 0) s_f = f;
        }
        __syncthreads();
        int count  = 0;
        double sum = 0.0;
        for (int row = blockIdx.x; row < s_f.y_size; row += kLiftPlainShare)
            for (int col = tid; col < s_f.x_size; col += kBlock)
            {
                const int x = (int)((float)col + s_f.min_x), y = (int)((float)row + s_f.min_y);
                if (x < 0 || x >= a.width || y < from || y >= a.height || !in_any_triangle(s_f, (float)x, (float)y)) continue;
                ++count;
                sum += (double)lift_pixel_error(a, x, y);
            }
#pragma unroll
        for (int d = kWave / 2; d >= 1; d >>= 1) count += __shfl_xor(count, d, kWave), sum += __shfl_xor(sum, d, kWave);
        if (lane == 0) s_sum[wave] = sum, s_count[wave] = count;
        __syncthreads();
        if (tid == 0)
        {
            for (int w = 1; w < kBlock / kWave; ++w) sum += s_sum[w], count += s_count[w];
            if (count > 0)
            {
                atomicAdd(&a.cell_sums[cell], sum);
                atomicAdd(&a.access_count[cell], count);
            }
            __threadfence();
            if ((atomicAdd(&a.plain_state[cell], 1u) & 0xFFu) == (uint32_t)kLiftPlainShare - 1u)
            {
                __threadfence();
                const double all = atomicAdd(&a.cell_sums[cell], 0.0);
                a.value[cell] = (float)((double)a.value[cell] + all);
            }
        }
        __syncthreads();
    }
}

}  // namespace vetrast
