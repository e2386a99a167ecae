// trace_tiles.h -- closest-hit and shadow queries of a whole wave: boxes around
// groups of 32 spheres (tiles) decide which tiles its rays can touch, and the
// matrix cores rule out spheres of a touched tile 32 at a time, with the flat
// loop's exact result (Engine/src/Renderer.cu:251-285 semantics).
//
// Tile filter.  For a ray (o, d), |d| = 1, let f be the point of its line
// closest to the origin of the coordinates (f.d = 0).  A sphere (c, r) has
//   disc = r^2 - dist(c, line)^2 = (c.d)^2 + 2 c.f - (|c|^2 - r^2) - |f|^2
// and the flat loop can only report a hit with disc >= 0.  This is an inner
// product of a vector of the ray (dx dx, dy dy, dz dz, dx dy, dx dz, dy dz, f,
// 1, E - |f|^2) and one of the sphere, so disc + E of 32 rays and 32 spheres is
// one 32x32x32 matrix product (two instructions); E bounds every error below,
// and a negative value rules the pair out.  The few spheres that are kept go
// through filter_sphere like the flat loop's.
//
// Units.  Coordinates are relative to the centre of the tiles' spheres and
// scaled by ts, a power of two, so that every sphere lies within 8 of the
// origin.  A number x enters the product as two half-precision numbers
// hi + lo; hi takes the upper 11 bits of x, so x - hi is exact.
//
// Error bound, with n = |o|, D = n + 8 and u = 2^-24:
//  * the flat loop's own rounding: oc, b, c, disc, sqrt, numerator and quotient
//    are each rounded once.  With F(t) = |o + t d - c|^2 - r^2 and d_c = |o - c|,
//    b is off by at most 4.01 u d_c, c by 6.02 u d_c^2 + u r^2, the rounding of
//    disc moves c by at most 2.02 u (2 d_c^2 + r^2); the root of that quadratic
//    has |F| <= 48.2 u d_c^2 + 16.1 u r^2, and the last three roundings move t by
//    at most u (5.03 d_c + 3.02 r) on a slope of at most 6 d_c + 2 r.  So a hit
//    it reports has |F(t)| <= 93 u d_c^2 + 36 u r^2, and its line disc >= minus
//    that.  o itself is rounded in tile units (3.4 u D^2): within 2^-17 D^2;
//  * hi + lo: ray side within 2^-20 |x| (lo is truncated), sphere side within
//    2^-22 |x|, lo * lo left out (2^-21): 1.75 2^-20 of the terms' absolute sum,
//    which is at most 1.5 (|f| + 8)^2.  E - |f|^2 is truncated towards zero,
//    which keeps more spheres where it is negative;
//  * the single-precision sum of 32 terms, taken as 32 2^-23 of the same sum;
//  * |d|^2 = a instead of 1 in (c.d)^2 and in f: 2 |a - 1| D^2.
// E = 2^-17 D^2 + 1.25 2^-17 (2 |f|^2 + 128) + 2 |a - 1| D^2 covers their sum
// (1.08 for the 1.25).  A ray with |f|^2 > 130 + 2 E passes all spheres.  Rays
// with a far from 1 or E past 4096 (which includes NaN) run the exact flat
// loop.
//
// Boxes.  A tile's box holds its spheres; per ray it is inflated by M, a
// bound of the excess sqrt(r^2 + q) - r, q = 2^-17 (D^2 + r^2), that the first
// error above allows (at most q / (2 r), t_lin = 2^-18 / smallest radius, and
// at most sqrt(q) <= 2^-8.5 (D + 4); r <= 8 <= D), and by 2^-18 (n + 16) for the
// slab test's own rounding (a few u of the coordinates' magnitudes).  Scenes
// of more than kTileFlat tiles also have a box for every eight.  A box is
// skipped when its inflated entry lies beyond an upper bound of the best
// sphere's exact t (best_hi / a, rounded up by 2^-20): everything in it then
// has a strictly larger t, which the reference rejects whatever its index.
// Shadow queries (dist2 >= 0: only the reference's decision t > 0 && t*t < dist2
// on the closest hit matters) also skip boxes beyond sqrt(dist2) and stop at
// the first sphere whose exact t is proven below it; the sphere they return is
// then some occluder, not necessarily the closest.  Without boxes (n_nodes 0:
// ATX_ACCEL_NONE) the product tests every sphere.
//
// What bounds it: VALU issue (0.30 instructions per cycle and SIMD in the path
// kernel; minima, compares and shifts run at half the rate of multiply-adds),
// at 5 waves per SIMD, which spend 39 % of their time issuing, 30 % waiting to
// issue and 31 % waiting for data; loading the next tile's operands early
// changed nothing (19.25 ms per 256 frames of 1080p both ways).  A 32x32x32 product takes about 66 cycles of a SIMD, and
// the 16 shifts that collect its signs run beside it (one conversion of both
// products to 6-bit floats instead of 32 shifts is a third shorter by itself,
// but needs both at once: 18.0 -> 22.1 ms); with the two-product
// form (b and |o - c|^2 - r^2, 2 VALU instructions per pair) it was 125.  All
// control flow is wave-uniform but the candidates' loop (0.3 to 1.4 per ray, 4
// to 5 in the slowest of 64 lanes at 64 to 512 spheres).  Against the per-lane
// walk of the tree's nodes (whose lanes were 37 % active and which re-ran the
// flat loop over all spheres for a ray with an ambiguous pair), whole calls:
// 1920x1080, 257 spheres, 20 frames 4.70 -> 3.40 ms, 256 frames 36.1 -> 25.5;
// 1024x1024, 513 spheres, 64 frames 8.48 -> 6.08; 1600x900, 8001 spheres, 32
// frames 31.1 -> 10.2 (k_first_hit alone 16.1 -> 1.25).  Testing every sphere by
// the product instead of a loop of scalar loads: 853x481, 97 spheres, 8 frames
// 1.33 -> 1.13 ms.
#pragma once

#include "bvh.h"
#include "trace_device.h"

namespace atx {

#if defined(__HIP_DEVICE_COMPILE__)
#define ATX_GLOBAL __attribute__((address_space(1)))
#else
#define ATX_GLOBAL
#endif

struct BvhQuery {
    uint32_t tests = 0;   // sphere tests
    uint32_t boxes = 0;   // box tests
    uint32_t exact = 0;   // orders settled by exact distances, exact loops
    // of the closest hit's sphere (queries but shadow ones that found one)
    float4 sphere = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    int32_t mat = 0;
};

// min(a, b) as one v_min_f32.  fminf on a value carried around a loop costs a
// canonicalising v_max_f32 besides the min; neither operand can be a
// signalling NaN here (both come out of arithmetic), for which that
// canonicalisation exists.
__device__ __forceinline__ float bvh_min_raw(float a, float b)
{
#if defined(__HIP_DEVICE_COMPILE__)
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
#else
    return __builtin_fminf(a, b);
#endif
}

#if defined(__HIP_DEVICE_COMPILE__)
#define TILE_CONST __attribute__((address_space(4)))
typedef _Float16 tile_h8 __attribute__((ext_vector_type(8)));
typedef float tile_f16v __attribute__((ext_vector_type(16)));
typedef uint32_t tile_u4 __attribute__((ext_vector_type(4)));

// (hi, lo) of x as two halves: hi in the low 16 bits.
__device__ __forceinline__ uint32_t tile_split(float x)
{
    const float hi = __uint_as_float(__float_as_uint(x) & 0xffffe000u);
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(hi, x - hi));
}

// The hi halves of two splits.
__device__ __forceinline__ uint32_t tile_his(uint32_t a, uint32_t b)
{
    return __builtin_amdgcn_perm(b, a, 0x05040100u);
}

// Exchanges the upper 32 lanes of a with the lower 32 lanes of b: a becomes
// the first 32 rays' operand (their own value in the lower lanes, b's in the
// upper ones) and b the other 32 rays'.
__device__ __forceinline__ void tile_swap(uint32_t& a, uint32_t& b)
{
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}

__device__ __forceinline__ tile_h8 tile_operand(uint32_t a, uint32_t b, uint32_t c, uint32_t d)
{
    const tile_u4 v = {a, b, c, d};
    return __builtin_bit_cast(tile_h8, v);
}

// Signs of disc + E for 32 rays and the 16 spheres this lane holds of a tile:
// bit 15 - k for the k-th, 1 = ruled out (the bits above hold nothing).
__device__ __forceinline__ uint32_t tile_signs(tile_h8 s0, tile_h8 s1, tile_h8 r0, tile_h8 r1)
{
    tile_f16v v = {};
    v = __builtin_amdgcn_mfma_f32_32x32x16_f16(s0, r0, v, 0, 0, 0);
    v = __builtin_amdgcn_mfma_f32_32x32x16_f16(s1, r1, v, 0, 0, 0);
    uint32_t m = 0u;
    for (int k = 0; k < 16; ++k)
        m = __builtin_amdgcn_alignbit(m, __float_as_uint(v[k]), 31);
    return m;
}
#endif

// The filtered test of filter_sphere, settled on the spot: where the intervals
// of the candidate s (slot or index id) and of the best sphere so far overlap,
// or the candidate's sign is open, both exact t are compared as the flat loop
// does (t > 0, smaller t, lower scene index among equal t).  Returns true when
// s became the new best.
__device__ __forceinline__ bool tile_candidate(const BvhDev& B, float4 s, int32_t slot, f3 o, f3 d, float a, Filter& f,
                                               BvhQuery& q)
{
    const ATX_GLOBAL int32_t* tidx = (const ATX_GLOBAL int32_t*)(uintptr_t)B.tidx;
    const ATX_GLOBAL float4* tsph = (const ATX_GLOBAL float4*)(uintptr_t)B.tsph;
    f.amb = 0u;
    Filter g = f;
    bool better = filter_sphere(s, slot, o, d, a, g);
    if (g.amb != 0u) {
        ++q.exact;
        const float t = exact_t(s, o, d, a);   // NaN where the line misses
        if (f.best < 0) {
            better = t > 0.0f;
        } else {
            const float tb = exact_t(tsph[f.best], o, d, a);
            better = t > 0.0f && t <= tb;
            if (better && t == tb)
                better = tidx[slot] < tidx[f.best];
        }
        if (better) {
            // an interval around the numerator t * a, as filter_sphere's
            const float n = t * a, u = __builtin_fmaxf(__builtin_fabsf(n), 0x1p-30f);
            g.best_lo = __builtin_fmaf(u, -0x1p-16f, n);
            g.best_hi = __builtin_fmaf(u, 0x1p-16f, n);
            g.best = slot;
        }
    }
    if (better) {
        f.best_lo = g.best_lo;
        f.best_hi = g.best_hi;
        f.best = slot;
    }
    return better;
}

// Closest hit (dist2 < 0) or shadow query (dist2 >= 0) of ray (o, d) of the
// lanes with `act`; every lane of the wave must call it (the matrix products
// and lane exchanges take all 64 lanes).  index: the id of a hit is to be the
// sphere's index in the scene (else it is only not negative).  masks: kChunk + 1
// rows of this wave in LDS.  The result of the other lanes is a miss.
template <uint32_t kChunk, class FlatSrc>
__device__ __forceinline__ Hit trace_tiles(const BvhDev& B, const FlatSrc& flat, const int32_t* sph_mat,
                                           uint32_t n_all, f3 o, f3 d, float dist2, bool act, bool index,
                                           uint32_t (*masks)[64], BvhQuery& q)
{
    static_assert(kChunk >= 8u, "a round's eight tiles have to fit");
    Hit h;
    h.id = -1;
    h.t = FLT_MAX;
#if defined(__HIP_DEVICE_COMPILE__)
    const uint32_t lane = threadIdx.x & 63u;
    const float a = dot(d, d);
    const bool shadow = dist2 >= 0.0f, want = act;
    Filter f = filter_init();
    FlatSrc by_slot = flat;   // scalar loads
    by_slot.p = (decltype(by_slot.p))(uintptr_t)B.tsph;
    for (uint32_t j = B.big0; j < B.big0 + B.n_big; ++j)
        tile_candidate(B, by_slot(j), (int32_t)j, o, d, a, f, q);
    q.tests += B.n_nodes ? B.n_big : n_all;   // without boxes every sphere is tested

    // the ray in tile units and its line's closest point to their origin
    const float ox = (o.x - B.cx) * B.ts, oy = (o.y - B.cy) * B.ts, oz = (o.z - B.cz) * B.ts;
    const float n = __builtin_amdgcn_sqrtf((ox * ox + oy * oy) + oz * oz);
    const float D = n + 8.0f, D2 = D * D;
    const float a1 = __builtin_fabsf(a - 1.0f);
    const float t1 = -((ox * d.x + oy * d.y) + oz * d.z);
    float fx = __builtin_fmaf(d.x, t1, ox), fy = __builtin_fmaf(d.y, t1, oy), fz = __builtin_fmaf(d.z, t1, oz);
    const float t2 = -((fx * d.x + fy * d.y) + fz * d.z);
    fx = __builtin_fmaf(d.x, t2, fx);
    fy = __builtin_fmaf(d.y, t2, fy);
    fz = __builtin_fmaf(d.z, t2, fz);
    const float ff = (fx * fx + fy * fy) + fz * fz;
    const float E = __builtin_fmaf(D2, 0x1p-17f + 2.0f * a1, 0x1.4p-17f * (2.0f * ff + 128.0f));
    const bool odd = !(E < 4096.0f) || !(a1 < 0x1p-10f);
    if (odd)
        act = false;
    if (ff > 130.0f + 2.0f * E)
        act = false;
    const float inv_a_up = __builtin_amdgcn_rcpf(a) * (1.0f + 0x1p-20f);
    const float s_up = shadow ? __builtin_amdgcn_sqrtf(dist2) * (1.0f + 0x1p-18f) : __builtin_inff();
    float tlim = __builtin_fminf(f.best_hi * inv_a_up, s_up);
    if (shadow && tlim * tlim < dist2)
        act = false;

    // slab test: t = (c +- h - o) / d per axis, h with the ray's inflation M
    // (2^-64 keeps an axis-parallel ray's reciprocals finite)
    const float ix = __builtin_amdgcn_rcpf(d.x + 0x1p-64f), iy = __builtin_amdgcn_rcpf(d.y + 0x1p-64f),
                iz = __builtin_amdgcn_rcpf(d.z + 0x1p-64f);
    const float jx = __builtin_fabsf(ix), jy = __builtin_fabsf(iy), jz = __builtin_fabsf(iz);
    const float M = __builtin_fminf((D2 + 64.0f) * B.t_lin, (D + 4.0f) * 0x1.6a0ap-9f) + 0x1p-18f * (n + 16.0f);
    const float ux = ox * ix, uy = oy * iy, uz = oz * iz;
    const float px = __builtin_fmaf(-M, jx, -ux), py = __builtin_fmaf(-M, jy, -uy), pz = __builtin_fmaf(-M, jz, -uz);
    const float qx = __builtin_fmaf(M, jx, -ux), qy = __builtin_fmaf(M, jy, -uy), qz = __builtin_fmaf(M, jz, -uz);
    // boxes are read with wave-uniform addresses through the constant address
    // space, as scalar loads
    const TILE_CONST float* boxes = (const TILE_CONST float*)(uintptr_t)B.tboxes;
    const auto touches = [&](uint32_t k, float lim) -> bool {
        const TILE_CONST float* b = boxes + 8u * k;   // centre, half size
        const float ax = __builtin_fmaf(-b[3], jx, __builtin_fmaf(b[0], ix, px)),
                    bx = __builtin_fmaf(b[3], jx, __builtin_fmaf(b[0], ix, qx));
        const float ay = __builtin_fmaf(-b[4], jy, __builtin_fmaf(b[1], iy, py)),
                    by = __builtin_fmaf(b[4], jy, __builtin_fmaf(b[1], iy, qy));
        const float az = __builtin_fmaf(-b[5], jz, __builtin_fmaf(b[2], iz, pz)),
                    bz = __builtin_fmaf(b[5], jz, __builtin_fmaf(b[2], iz, qz));
        const float tn = __builtin_fmaxf(__builtin_fmaxf(__builtin_fmaxf(ax, ay), az), 0.0f);
        const float tf = __builtin_fminf(__builtin_fminf(__builtin_fminf(bx, by), bz), lim);
        return tn <= tf;
    };

    // ray operands: a lane below 32 supplies the first half of a product's 16
    // terms of its ray, the lane 32 above it the second half
    uint32_t r0 = tile_split(d.x * d.x), r1 = tile_split(d.y * d.y), r2 = tile_split(d.z * d.z),
             r3 = tile_split(d.x * d.y), r4 = tile_split(d.x * d.z), r5 = tile_split(d.y * d.z), r6 = tile_split(fx),
             r7 = tile_split(fy), r8 = tile_split(fz), r9 = tile_split(E - ff);
    uint32_t r10 = 0x3c003c00u;   // 1, 1
    uint32_t r11 = tile_his(r0, r1), r12 = tile_his(r2, r3), r13 = tile_his(r4, r5), r14 = tile_his(r6, r7), r15 = r8;
    tile_swap(r0, r4);
    tile_swap(r1, r5);
    tile_swap(r2, r6);
    tile_swap(r3, r7);
    tile_swap(r8, r12);
    tile_swap(r9, r13);
    tile_swap(r10, r14);
    tile_swap(r11, r15);
    const tile_h8 ra0 = tile_operand(r0, r1, r2, r3), ra1 = tile_operand(r8, r9, r10, r11);
    const tile_h8 rb0 = tile_operand(r4, r5, r6, r7), rb1 = tile_operand(r12, r13, r14, r15);

    const ATX_GLOBAL uint4* tiles = (const ATX_GLOBAL uint4*)(uintptr_t)B.tiles + lane;
    const ATX_GLOBAL float4* tsph = (const ATX_GLOBAL float4*)(uintptr_t)B.tsph;
    const uint32_t n_tiles = B.n_tiles;
    const bool boxed = B.n_nodes != 0u, groups = n_tiles > kTileFlat;
    for (uint32_t t = 0; t < n_tiles;) {
        // candidates of up to kChunk touched tiles
        uint32_t nm = 0u, some = 0u;
        const float lim = act ? tlim * B.ts : -1.0f;   // a lane that does not act touches nothing
        for (;;) {
            if (groups && boxed && !__any(touches(n_tiles + t / 8u, lim))) {
                t += 8u;
                if (t >= n_tiles)
                    break;
                continue;
            }
            // which of the next eight tiles this lane's ray touches
            const uint32_t nt = n_tiles - t < 8u ? n_tiles - t : 8u;
            uint32_t touched = 0u, need = 0u;
            if (boxed) {
#pragma unroll
                for (uint32_t k = 0; k < 8u; ++k) {
                    if (k < nt) {
                        const bool touch = touches(t + k, lim);
                        touched |= touch ? 1u << k : 0u;
                        need |= __any(touch) ? 1u << k : 0u;
                    }
                }
                q.boxes += nt;
            } else {
                touched = act ? (1u << nt) - 1u : 0u;
                need = __any(act) ? (1u << nt) - 1u : 0u;
            }
            if (nm + (uint32_t)__popc(need) > kChunk)
                break;   // no room: test the candidates so far, then come back
            while (need != 0u) {
                const uint32_t k = (uint32_t)__builtin_ctz(need);
                need &= need - 1u;
                const bool touch = ((touched >> k) & 1u) != 0u;
                const unsigned long long rays = __ballot(touch);
                const uint4 w0 = tiles[(t + k) * 128u], w1 = tiles[(t + k) * 128u + 64u];
                const tile_h8 s0 = tile_operand(w0.x, w0.y, w0.z, w0.w), s1 = tile_operand(w1.x, w1.y, w1.z, w1.w);
                uint32_t m0 = ~0u, m1 = ~0u;
                if ((uint32_t)rays != 0u)
                    m0 = tile_signs(s0, s1, ra0, ra1);
                if ((uint32_t)(rays >> 32) != 0u)
                    m1 = tile_signs(s0, s1, rb0, rb1);
                tile_swap(m0, m1);   // both halves of this lane's own ray
                const uint32_t keep = touch ? ~((m0 & 0xffffu) | (m1 << 16)) : 0u;
                masks[nm][lane] = keep;
                masks[kChunk][nm] = (t + k) * 32u;
                some |= keep != 0u ? 1u << nm : 0u;
                ++nm;
            }
            t += 8u;
            if (t >= n_tiles)
                break;
        }
        // The next candidate's sphere is on its way while one is tested: whole
        // calls 1080p, 257 spheres, 256 frames 19.41 -> 19.30 ms, 1600x900, 8000
        // spheres 9.81 -> 9.74, 1280x720 in place 0.705 -> 0.697, batch of 12
        // scenes 48.9 -> 48.5.
        uint32_t m = 0u, base = 0u;
        const auto pop = [&]() -> uint32_t {
            if (m == 0u) {
                const uint32_t k = (uint32_t)__builtin_ctz(some);
                some &= some - 1u;
                m = masks[k][lane];
                base = masks[kChunk][k];
            }
            const uint32_t k = base + (uint32_t)__builtin_ctz(m);
            m &= m - 1u;
            return k;
        };
        if (some != 0u) {
            uint32_t k = pop();
            float4 s = tsph[k];
            for (bool more = true; more;) {
                uint32_t kn = k;
                more = (m | some) != 0u;
                if (more)
                    kn = pop();
                const float4 sn = tsph[kn];
                q.tests += boxed ? 1u : 0u;
                if (tile_candidate(B, s, (int32_t)k, o, d, a, f, q))
                    tlim = bvh_min_raw(tlim, f.best_hi * inv_a_up);
                // t of the best sphere <= tlim, and tlim*tlim < dist2 proves it occludes
                if (shadow && tlim * tlim < dist2) {
                    more = false;
                    act = false;
                }
                k = kn;
                s = sn;
            }
        }
    }

    if (want && odd) {
        ++q.exact;
        q.tests += n_all;
        h = trace_exact(flat, n_all, o, d);
        if (h.id >= 0) {
            q.sphere = flat((uint32_t)h.id);
            q.mat = sph_mat[h.id];
        }
    } else if (want && f.best >= 0) {
        // The winner's sphere, index and material are loaded together: a wave
        // spent 40 % of its time in this end of the query and in the shading
        // for a sixth of its instructions, waiting for index, sphere, its
        // material's index, the material and the light one after another.  With
        // one load less to wait for here, two in the shading and one before
        // the next direction, the path kernel went from 20.0 to 19.2 ms (1080p,
        // 257 spheres, 256 frames) and a batch of 12 scenes from 49.2 to 46.7.
        // A shadow query needs nothing but t, and not its exact value where a
        // bound above it already lies before the light.
        const float above = f.best_hi * inv_a_up;
        h.id = f.best;
        h.t = above;
        if (index || (!shadow && !B.tmat))
            h.id = B.tidx[f.best];
        if (!shadow)
            q.mat = B.tmat ? B.tmat[f.best] : sph_mat[h.id];
        if (!(shadow && above * above < dist2)) {
            q.sphere = tsph[f.best];
            h.t = exact_t(q.sphere, o, d, a);
        }
    }
#endif
    return h;
}

}  // namespace atx
