// bvh_build.h -- host construction of a scene's tiles (device layout in bvh.h),
// and of a binary tree over the same spheres that the host checks use.  Plain C++ (no HIP types), so that host-side checks can
// build it with any C++ compiler.
#pragma once

#include <stddef.h>
#include <stdint.h>
#include <vector>

namespace atx {

constexpr uint32_t kBvhLayouts = 8;      // maximum number of traversal orders
constexpr uint32_t kBvhLeafMax = 4;      // spheres per leaf (2-bit count field)
constexpr uint32_t kBvhMinSpheres = 16;  // smaller scenes use the flat loop only
constexpr uint32_t kBvhMaxBig = 16;
constexpr uint32_t kBvhMaxTree = 16382;  // tree spheres addressable by a 14-bit leaf index
constexpr uint32_t kTileMaxSpheres = 1u << 20;
constexpr uint32_t kTileSpheres = 32;    // spheres per tile (rows of the matrix product)
constexpr uint32_t kTileWords = 512;     // 32-bit words of one tile
// Tiles whose candidates a wave keeps before it tests them, in one LDS row
// each (and one row for their first spheres): as many as leave room for five
// workgroups on a CU.  1600x900, 8000 spheres: path kernel 9.13 -> 8.88 ms with
// 13 instead of 8; 1024x1024, 512 spheres 3.00 -> 2.91; 1080p, 257 spheres, one
// visit to four tiles, the same.  In-place launches hold 4 KB more themselves, 6
// with kept hits; a round of eight tiles has to fit.
constexpr uint32_t kTileChunk = 13, kTileChunkInPlace = 9, kTileChunkKeep = 8;
constexpr uint32_t kTileFlat = 16;       // with more tiles, every eight have a box of their own
constexpr uint32_t kBvhGrid = 65535;     // node boxes are 16-bit cells of the tree's box

// Node encoding (4 x u32 = 16 B): cell coordinates of the box corners,
// lo = (x, y, z) and hi = (x, y, z), 16 bits each, then skip (16 bits: node
// index after this node's subtree) and leaf (16 bits: 0 for an inner node,
// else ((first + 1) << 2) | (count - 1)).
struct HostBvh {
    std::vector<uint32_t> nodes; // layouts * n_nodes * 4
    std::vector<float> lsph;     // 4 per sphere, leaf order
    std::vector<int32_t> lidx;
    std::vector<int32_t> big;
    uint32_t n_nodes = 0;
    uint32_t layouts = 0;        // 1 (one depth-first order) or kBvhLayouts (one per direction octant)
    float cx = 0, cy = 0, cz = 0, rb = 0, r_min = 0, r_max = 0;
    float base[3] = {0, 0, 0};   // world position of cell 0
    float scale[3] = {1, 1, 1};  // world size of one cell per axis
    float inv_scale[3] = {1, 1, 1};
    float ext = 0;               // upper bound of kBvhGrid * scale over the axes
    std::vector<uint32_t> tiles; // n_tiles * kTileWords, two halves per word
    std::vector<float> tboxes;   // 8 per box: centre, half size, 0, 0; tiles, then groups of eight
    std::vector<float> tsph;     // 4 per sphere, tile order
    std::vector<int32_t> tidx;
    uint32_t n_tiles = 0;
    float ts = 0;                // tile units per world unit
    float t_lin = 0;             // 2^-18 / smallest radius in tile units (capped)
};

// Row of a tile's matrix that holds its k-th sphere (k < kTileSpheres): the
// product leaves row 8 * (i / 4) + 4 * h + i % 4 in register i of lane half h,
// and the query collects register i of half h at bit 16 * h + 15 - i.
inline uint32_t tile_row(uint32_t k)
{
    const uint32_t i = 15u - (k & 15u), h = k >> 4;
    return 8u * (i / 4u) + 4u * h + i % 4u;
}

// Sorts out the spheres given as (cx, cy, cz, r*r) quadruples that cannot go
// into tiles and builds tiles over the others; with `layouts` 1 or kBvhLayouts
// also the tree, in that many traversal orders (the kernels do not use it:
// 0).  Scenes with fewer than kBvhMinSpheres spheres, or more than kBvhMaxBig
// spheres kept out, or more than kTileMaxSpheres (with a tree kBvhMaxTree)
// others get neither (n_tiles = n_nodes = 0).
void build_bvh(const float* sph4, uint32_t n, uint32_t layouts, HostBvh* out);

// Device bytes of the tiles of an n-sphere scene (upper bound).
size_t bvh_device_bytes(uint64_t n);

}  // namespace atx
