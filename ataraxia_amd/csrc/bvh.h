// bvh.h -- device layout of a scene's tiles, the structure its rays are traced
// with (trace_tiles.h; the host builder is bvh_build.h).
//
// Tiles only decide which spheres a ray tests.  Every sphere that is tested
// goes through the same filtered test as the flat loop (trace_device.h), so
// the closest hit, including the lowest-index rule for equal t
// (Engine/src/Renderer.cu:274), is the one the reference's loop over all
// spheres finds.  Ruling out is conservative with respect to the reference's
// rounded arithmetic, not only to exact geometry.
//
// Layout in HBM (per scene), spheres 32 to a tile, neighbours together:
//   tiles  uint4[n_tiles][128]  matrix operands in half precision
//   tboxes float4[n_nodes][2]   box (centre, half size; tile units) of every
//                           tile, then of every eight consecutive tiles
//   tsph   float4[n]        spheres by slot (cx, cy, cz, r*r): those of the
//                           tiles in tile order, then from slot big0 on the
//                           n_big kept out of the tiles (radius larger than
//                           the region of the others, e.g. a ground sphere, or
//                           non-finite data), which a loop tests first
//   tidx   int32[n]         each slot's sphere in the scene
//   tmat   int32[n]         its material (nullptr: looked up by tidx)
// Boxes are rounded outwards from double precision, so each contains its
// spheres exactly.
#pragma once

#include <stdint.h>
#include <hip/hip_runtime.h>

#include "bvh_build.h"

namespace atx {

struct BvhDev {
    const uint4* tiles;
    const float4* tboxes;
    const float4* tsph;
    const int32_t* tidx;
    const int32_t* tmat;
    uint32_t n_tiles;   // 0 = flat loop over all spheres
    uint32_t n_nodes;   // boxes; 0 = every ray tests every sphere
    uint32_t n_big, big0;
    float cx, cy, cz;   // centre of the tiles' region
    float ts;           // tile units per world unit (a power of two)
    float t_lin;        // 2^-18 / smallest radius in tile units
};

}  // namespace atx
