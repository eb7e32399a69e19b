// Which launches of the per-pixel backward kernels cut the regions of the screen into parts for the XCDs (TileMap, common.h). Plain
// host C++: the rule is checked without a GPU.
#pragma once
#include <stdint.h>

#include <algorithm>

namespace vetrast
{
// Region r goes to XCD r % 8, the same one in every view. What parts can gain is that an XCD holds more of a scene than another; what
// they cost is lines of the images in several L2s, the more the smaller a region is. The kernel's us whole / in 16 parts, means over three
// scenes; `list` is what fragments_a_pixel_may_blend says:
// * Regions of 64 pixels and less (up to three layers) cost more than they give: 1080p with three, two and one layers 347 / 365,
//   276 / 296, 164 / 181 (list 9), 256x256 with three 20 / 20 to 26 / 27.5; what gains up to 9 % is 1000x700 and 500x380 with three.
// * Up to about as many regions as there are XCDs leave some of them idle, or one with twice another's: 203x155 (4 regions) 21 / 17, 384x256 (6)
//   15.0 / 14.2, two town views of 384x384 (9) and two crops of that size 13 to 28 % faster with any list, 700x256 (12) 10 to 20 %; the
//   dearest is one 384x384 frame with its scene in the middle, 1 to 4 % slower.
// * Regions of 256 pixels (five layers) are few and large: 1080p 130 / 114, 602x267 43 / 26, 1000x700 38 / 36, two views of it 80 / 71,
//   2560x1440 352 / 336, 1237x701 (15 of them) 39.5 / 39, with any list.
// * Else the lists decide, and from which length on depends on how many regions lie in a row. A multiple of eight gives every XCD whole columns:
//   960x540 28 / 28 with list 0.8, 34.5 / 34.7 with 1.2, 55 / 53 with 1.7, 80 / 74 with 3.3; 1000x700 36 / 38 with 0.9, 47 / 48 with 1.4, 64 / 62
//   with 2, 127 / 113 with 3.8; two town views of 960x540 139 / 120 with 1.1, of 2000x1080 2 to 4 % slower up to 2.8.
// * One, four or seven (modulo 8) give it a diagonal or every other row's half: 1100x600 31 / 33 with 0.8, 102 / 97 with 3.2; 1080p
//   146 / 145 with 1.2, 224 / 220 with 2.4, 192 / 186 with 3.2, 242 / 234 with 4.2, ten million points in it 553 / 530, but four town
//   views with list 1.1 387 / 402. 512x512 26 / 28 with 2.4, 31 / 35 with 3.3; four crops of that size with the 2x2 splat
//   157 / 162 with 3.9, 257 / 254 with 7.8, where many points are dropped by radius 91 / 89; in FULL_BLEND 183 / 176 with 3.9.
// * Two, three, five or six spread whatever lies together by themselves: 700x500 37 / 41 with 3.7, 84 / 83 with 6, 102 / 95 with 10;
//   640x360 31 / 31 with 3.3, 61 / 57 with 8.6; 1237x701 36 / 41 with 0.8, 65 / 69 with 3.1, 167 / 168 with 5.2, 208 / 203 with 8.6.
constexpr int kPartsLayers            = 4;   // at least
constexpr uint32_t kPartsRegions      = 12;  // at most, of a view, with any list
constexpr uint32_t kPartsLargeRegions = 64;  // ... of five layers
constexpr double kPartsList[8]        = {1.0, 3.5, 6.0, 6.0, 3.5, 6.0, 6.0, 3.5};  // for regions in a row, modulo 8

// Fragments a pixel of layer 0 may blend: those of every point, unless the caller knows how many a view leaves there. Then twice that
// number, as for the sizes of bins: in the frames the rule was measured on about half of the points are in view. (A town
// of ten million points at 1080p, of which a fifteenth is: 123 whole, 131 in parts.)
inline double fragments_a_pixel_may_blend(double if_all_visible, float expected, int w, int h, int cut)
{
    double fragments = if_all_visible;
    if (expected > 0.f) fragments = std::min(fragments, 2.0 * (double)expected);
    const double list = fragments / ((double)w * (double)h);
    return cut > 0 ? std::min(list, (double)cut) : list;
}

inline bool regions_in_parts(int layers, uint32_t regions_x, uint32_t regions, double list)
{
    if (layers < kPartsLayers) return false;
    return regions <= (layers == kPartsLayers ? kPartsRegions : kPartsLargeRegions) || list >= kPartsList[regions_x % 8u];
}
}  // namespace vetrast
