// device_types.h -- device-side scene layout and the kernels' counters.
//
// HBM layout of one scene (private to libatx; the C ABI takes the reference's
// packed AoS structs and this is built from them on upload):
//   sph      float4[N]   (cx, cy, cz, r*r)      16 B/sphere, the only data the
//                                                closest-hit loop reads
//   sph_mat  int32[N]    material index (clamped to [0, M) on the host)
//   mat      float4[3M]  (albedo, roughness) (F0, metallic)
//                        (emission colour, emission intensity)
//   light    float4[2L]  (position, intensity) (colour * intensity, 0)
// r*r is precomputed once; the reference evaluates radius*radius inside its
// loop (Renderer.cu:264), which rounds to the same value.
#pragma once

#include <stdint.h>
#include <hip/hip_runtime.h>

#include "bvh.h"

namespace atx {

// Counters written by the kernels (device memory, u64 each, on kCounterLines
// lines whose sums are the counts).
enum CounterSlot : uint32_t {
    kCtrRays = 0,          // rays traced (continuation/primary + shadow)
    kCtrExact = 1,         // traces the interval filter left open, settled by exact distances
    kCtrTests = 2,         // ray-sphere tests
    kCtrBoxes = 3,         // tests of tiles' boxes (not of those around eight tiles: counting
                           // them cost the path kernel 0.7 %); again in a round that comes back
    kCtrReused = 4,        // rays answered from the per-pixel first-bounce cache
    kCtrCount = 5,
};
// A wave adds to one line, with one request for all of its sums: every wave
// adding each sum to a single line took 11.6 ns apiece, 4 x 7168 of them at
// the end of a launch (1080p, one frame: path kernel 0.39 -> 0.27 ms;
// 640x360, 4 spheres, 64 frames: 0.57 -> 0.44 ms).
constexpr uint32_t kCounterLines = 16;
constexpr uint32_t kCounterStride = 16;   // 128 bytes
constexpr uint32_t kCounterWords = kCounterLines * kCounterStride;
constexpr size_t kCounterBytes = kCounterWords * sizeof(unsigned long long);

inline unsigned long long counter_sum(const unsigned long long* lines, CounterSlot k)
{
    unsigned long long s = 0;
    for (uint32_t i = 0; i < kCounterLines; ++i)
        s += lines[i * kCounterStride + k];
    return s;
}

}  // namespace atx
