// render_wavefront.hip -- persistent, path-regenerating renderer.
//
// The per-pixel path (Renderer.cu:287-387) runs as a per-lane state machine
// so that all lanes of a wave trace a ray in every iteration:
//   START   begin the path of the lane's (frame, pixel) job
//   CONT    trace the primary/continuation ray; shade the hit; pick a light
//   SHADOW  trace the shadow ray; add the light's Cook-Torrance contribution
//   (then Russian roulette + next direction, or the path ends)
// Every (frame, pixel) path is an independent job.  A lane whose path ends
// stores the sample in the launch's sample buffer and takes the next job at
// once, so the work is shared out one path at a time: no lane waits for
// another pixel's earlier frame and no wave is left with a long tail of
// serial frames when the queue runs dry.  k_accumulate then adds every
// pixel's samples in frame order (Renderer.cu:164-168).  The floating-point
// operations of one path are exactly the plain kernel's (and the oracle's)
// and the additions happen in the same order, so the results are
// bit-identical to rendering each scene alone, one frame per launch, with
// the reference's per-pixel loop.
//
// Work distribution: a wave takes blocks of `chunk_px` consecutive jobs of
// one scene from the launch's counters (kQueueShards) and hands them to its
// lanes as they fall idle.  A scene's jobs come in groups of 8 neighbouring pixels
// times the launch's frames, frame after frame inside a group
// (job_pixel_frame), so a wave traces 8 neighbouring pixels in many frames
// at once: their rays start from the same few hits, which keeps the lanes of
// a wave near the same spheres and makes whole waves miss the same spheres in
// the flat loop.  Samples are stored in job order: a wave's block of jobs
// fills whole 128-byte lines of the sample buffer, which no other wave
// touches, and k_accumulate reads a pixel's frames 8 samples apart.
//
// First-bounce cache: a pixel's primary ray, the shading at its hit and the
// shadow ray towards each light are the same in every frame.  When the
// launch has the cache (k_first_hit, once per camera and scene), bounce 0
// of a path is done where the job is handed out -- the cached term of the
// frame's light if it reaches the hit, roulette, the next direction -- and
// the lane enters the trace loop at its first continuation ray or ends the
// path at once.  With the cache's hit list, jobs cover only the pixels
// whose primary ray hits; k_accumulate adds the others' constant sample.
//
// Rays of scenes with tiles are traced by whole waves (trace_tiles.h): all 64
// lanes go through a query together, those without a ray as well.  In scenes
// without one every ray tests every sphere.  Spheres, boxes and the scene
// table are read with wave-uniform addresses through the constant address
// space, which the compiler lowers to scalar loads.  A wave works on one scene
// at a time and drains its lanes before it switches.
//
// Registers: launches whose scenes all use the flat loop have an instance for
// each of 5 to 8 resident waves per SIMD (amdgpu_waves_per_eu; 7 by default),
// launches with tiles one for 5 (kWfWavesTree).
#include "device_types.h"
#include "trace_device.h"
#include "trace_tiles.h"
#include "wavefront.h"

#include <stdlib.h>

namespace atx {
namespace {

constexpr uint32_t kIdle = 0, kCont = 1, kShadow = 2, kNew = 3, kAgain = 4;

// The scene table and the sphere arrays do not change during a launch; read
// through the constant address space, wave-uniform loads from them become
// scalar loads (s_load) into SGPRs even though the kernel stores to global
// memory elsewhere.  (The host pass only parses the kernel; it gets no
// address space.)
#if defined(__HIP_DEVICE_COMPILE__)
#define ATX_CONST __attribute__((address_space(4)))
#else
#define ATX_CONST
#endif
using CScene = const ATX_CONST WfScene;
using CF4 = const ATX_CONST float4;

template <class T>
__device__ __forceinline__ const ATX_CONST T* as_const(const T* p)
{
    return (const ATX_CONST T*)(uintptr_t)p;
}

// The kernel's argument where it lies: read at its use, it takes no registers
// (in place, 2001 spheres, 8 frames: 2.76 -> 2.73 ms).
__device__ __forceinline__ const ATX_CONST WfPass& kernel_pass()
{
#if defined(__HIP_DEVICE_COMPILE__)
    return *(const ATX_CONST WfPass*)__builtin_amdgcn_kernarg_segment_ptr();
#else
    static const WfPass none{};   // the host pass only parses the kernels
    return none;
#endif
}

struct SphSrc {
    CF4* p;
    __device__ __forceinline__ float4 operator()(uint32_t i) const { return p[i]; }
};

__device__ __forceinline__ f3 xyz(float4 v) { return mk(v.x, v.y, v.z); }

__device__ __forceinline__ unsigned long long wave_sum(unsigned long long v)
{
    for (int off = 32; off > 0; off >>= 1)
        v += __shfl_xor(v, off, 64);
    return v;
}

// Adds the wave's counts to its line of the launch's counters: the lanes'
// test counts, which it clears, and the wave's rays (every lane of the wave
// calls it).  One request to the line carries all four sums.
__device__ __forceinline__ void flush_counters(unsigned long long* ctr, uint32_t lane, uint32_t& tests,
                                               uint32_t& boxes, unsigned long long rays, unsigned long long reused)
{
    const unsigned long long ts = wave_sum(tests);
    const unsigned long long bx = wave_sum(boxes);
    const unsigned long long v = lane == kCtrRays ? rays : lane == kCtrTests ? ts : lane == kCtrBoxes ? bx : reused;
    if (lane < kCtrCount && lane != kCtrExact && v)
        atomicAdd(ctr + lane, v);
    tests = boxes = 0u;
}

// ---- one bounce of the per-pixel path (Renderer.cu:319-381), in pieces
// shared by the path kernel and the first-bounce cache, so that both
// evaluate the same expressions in the same order ----

// Hit point, normal and the origin of the rays that leave the hit
// (Renderer.cu:325-333).
__device__ __forceinline__ void hit_frame(float4 sphere, const Hit& h, f3 ro, f3 rd, f3& pos, f3& nrm, f3& so)
{
    const f3 center = xyz(sphere);
    pos = add(sub(ro, center), scale(rd, h.t));
    nrm = normalize(pos);
    pos = add(pos, center);
    so = add(pos, scale(nrm, 0.0001f));
}

// Direction (normalised) and squared distance from pos to a light
// (Renderer.cu:343-346).
__device__ __forceinline__ void light_ray(float4 light_pos, f3 pos, f3& L, float& dist2)
{
    L = sub(xyz(light_pos), pos);
    dist2 = dot(L, L);
    L = normalize(L);
}

// The shadow decision on the shadow ray's closest hit (Renderer.cu:348-350):
// lit unless that hit lies strictly between the surface and the light.
__device__ __forceinline__ bool lit_by(const Hit& h, float dist2)
{
    const float st = h.id < 0 ? -1.0f : h.t;
    return !(st > 0.0f && st * st < dist2);
}

// The hit material's emission (m2: its last quarter), added to col
// (Renderer.cu:334-337).
__device__ __forceinline__ void add_emission(float4 m2, f3 tp, f3& col)
{
    if (m2.w > 0.0f)
        col = add(col, mul(scale(xyz(m2), m2.w), tp));
}

// Emission of a continuation hit on `sphere` of material mid and the light its
// shadow ray goes to.  Returns true when a shadow ray follows (the scene has
// lights).
__device__ __forceinline__ bool shade_hit(CScene* S, float4 sphere, int32_t mid, const Hit& h, f3 ro, f3 rd, f3 tp,
                                          uint32_t seed, f3& col, f3& nrm, f3& so, uint32_t& lidx, f3& L, float& dist2)
{
    // both loads before the first use of either
    float4 light = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (S->n_light != 0) {
        lidx = umod(pcg_hash(seed), S->div_light);   // pcg_hash(seed) % n_light
        light = S->light[2 * lidx];
    }
    float4 m2 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (S->emits)
        m2 = S->mat[3 * mid + 2];
    f3 pos;
    hit_frame(sphere, h, ro, rd, pos, nrm, so);
    add_emission(m2, tp, col);
    if (S->n_light == 0)
        return false;
    light_ray(light, pos, L, dist2);
    return true;
}

// Cook-Torrance term of a light that reaches the hit, weighted by the path
// throughput (Renderer.cu:351-360).  m0, m1: the material's first two quarters;
// radiance: the light's colour times its intensity.
__device__ __forceinline__ f3 light_term(float4 m0, float4 m1, float4 radiance, f3 nrm, f3 rd, f3 L, f3 tp, bool mild)
{
    const f3 albedo = xyz(m0);
    const float metallic = m1.w;
    const f3 base = add(scale(xyz(m1), 1.0f - metallic), scale(albedo, metallic));
    f3 f;
    bool ok = false;
    if (mild)
        f = cook_torrance_mild(albedo, base, metallic, m0.w, nrm, neg(rd), L, ok);
    if (__builtin_expect(!ok, 0))
        f = cook_torrance(albedo, base, metallic, m0.w, nrm, neg(rd), L);
    return mul(mul(xyz(radiance), f), tp);
}

// Throughput and Russian roulette at the end of a bounce (Renderer.cu:362-379).
// Returns true when the path ends here, by the draw or at its last bounce.
// m0: the material's albedo and roughness.  surface: its roughness and
// metallic, for the next direction.
__device__ __forceinline__ bool roulette(CScene* S, float4 m0, float metallic, f3& tp, int32_t bounce, uint32_t& seed,
                                         f3& surface)
{
    surface.x = m0.w;
    surface.y = metallic;
    tp = mul(tp, xyz(m0));
    float p;
    if (S->mild) {
        // p is 0.1 for every length below that, 1 for every one above it
        float h;
        const float d = __builtin_amdgcn_fmed3f(dot(tp, tp), 0x1p-20f, 4.0f);
        p = gmax(0.1f, gmin(1.0f, sqrt_from(d, __builtin_amdgcn_rsqf(d), h)));
    } else {
        p = gmax(0.1f, gmin(1.0f, length(tp)));
    }
    if (pcg_float(seed) > p)
        return true;
    if (S->mild) {
        const float r = reciprocal_from(p, __builtin_amdgcn_rcpf(p));
        tp = mk(quotient(tp.x, p, r), quotient(tp.y, p, r), quotient(tp.z, p, r));
    } else {
        tp = divs(tp, p);
    }
    return bounce + 1 >= S->max_bounces;
}

// The same at bounce 0, where the throughput is 1: the scene holds p and
// albedo / p per material (mat_rr), which saves a square root and three
// divisions in every path.
__device__ __forceinline__ bool roulette_first(CScene* S, int32_t mid, f3& tp, uint32_t& seed)
{
    const float4 rr = S->mat_rr[mid];
    tp = xyz(rr);
    return pcg_float(seed) > rr.w || S->max_bounces <= 1;
}

// The next direction of a path that goes on (Renderer.cu:381-384).
__device__ __forceinline__ void next_direction(f3 surface, f3 nrm, f3& rd, int32_t& bounce, uint32_t& seed)
{
    rd = sample_next(nrm, surface.y > 0.0f, surface.x, seed);
    ++bounce;
    seed += (uint32_t)bounce;
}

// The pixel of the scene's job `job` (`slots` jobs per frame): the path
// state does not carry it, only the debug captures need it.
__device__ __forceinline__ uint32_t job_pixel(CScene* S, uint32_t slots, uint32_t job)
{
    uint32_t slot, f;
    job_pixel_frame(job, slots, S->div_group, slot, f);
    return S->hit_px ? S->hit_px[slot] : slot;
}

__device__ __forceinline__ f3 primary_direction(CScene* S, uint32_t px)
{
    const uint32_t W = S->width;
    const uint32_t y = px / W, x = px - y * W;
    float ip[16], iv[16];
    for (int k = 0; k < 16; ++k) {
        ip[k] = S->inv_proj[k];
        iv[k] = S->inv_view[k];
    }
    return camera_ray(ip, iv, x, y, W, S->height);
}

// Adds a sample to a channel's running sum (Renderer.cu:165), compensated if
// kahan (c: the compensation).
__device__ __forceinline__ void accumulate(bool kahan, float v, float& acc, float& c)
{
    if (kahan) {
        const float y = v - c, t = acc + y;
        c = (t - acc) - y;
        acc = t;
    } else {
        acc = acc + v;
    }
}

// Display value of a sum over `frame` frames (Renderer.cu:166-168, Renderer.h:70-78).
__device__ __forceinline__ uint32_t display(float4 acc, uint32_t frame)
{
    const float fi = (float)frame;
    return rgba8(gclamp(acc.x / fi, 0.0f, 1.0f), gclamp(acc.y / fi, 0.0f, 1.0f), gclamp(acc.z / fi, 0.0f, 1.0f),
                 gclamp(acc.w / fi, 0.0f, 1.0f));
}

// In-place launches: the sample of pixel px, the same in n frames of the
// launch from f on, goes to the accumulation; the last frame's also to the image.
__device__ __forceinline__ void add_sample(CScene* S, const ATX_CONST WfPass& a, uint32_t px, uint32_t f, uint32_t n,
                                           f3 col)
{
    const uint32_t frame = a.frame0 + f;
    const bool kahan = S->kahan != 0u;
    const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float4 acc = frame == 1u ? zero : S->accum[px];
    float4 c = kahan && frame != 1u ? S->comp[px] : zero;
    for (uint32_t k = 0; k < n; ++k) {
        accumulate(kahan, col.x, acc.x, c.x);
        accumulate(kahan, col.y, acc.y, c.y);
        accumulate(kahan, col.z, acc.z, c.z);
        accumulate(kahan, 1.0f, acc.w, c.w);
    }
    S->accum[px] = acc;
    if (kahan)
        S->comp[px] = c;
    if (f + n == a.frames) {
        S->image[px] = display(acc, frame + n - 1u);
        if (S->dbg_radiance)
            S->dbg_radiance[px] = make_float4(col.x, col.y, col.z, 1.0f);
    }
}

// The sample of the scene's job `job` (`slots` jobs per frame), and the
// last frame's debug capture.
__device__ __forceinline__ void store_sample(CScene* S, uint32_t slots, uint32_t job, f3 col)
{
    S->samples[job] = make_float3(col.x, col.y, col.z);
    if (S->dbg_radiance) {
        uint32_t slot, f;
        job_pixel_frame(job, slots, S->div_group, slot, f);
        if (f == S->frames - 1u)
            S->dbg_radiance[S->hit_px ? S->hit_px[slot] : slot] = make_float4(col.x, col.y, col.z, 1.0f);
    }
}

// kInPlace (scenes with tiles; k_render_flat does the others): a job is a
// pixel, and its lane renders the launch's frames one after another into the
// accumulation; no samples, no first-bounce cache.  A kernel with one lane per
// pixel and frame, 64 pixels to a wave until its longest path ended, took 0.62 ms
// per frame at 1280x720 with 129 spheres; here lanes go on with their next frame
// or another pixel: a call of 4 frames 2.68 -> 0.81 ms, 0.63 with the steps since.
// It is bound like the sampling one, by VALU issue.
// kKeep: a pixel's primary hit is the same in every frame, so its lane keeps it
// and the frames after the first start at its shadow ray, from three frames on
// (1280x720, 129 spheres: 1 frame 266 us without and 281 with it, 2 frames 393 and
// 400, 4 frames 635 and 602, 8 frames 1175 and 965).
template <uint32_t kWaves, bool kTree, bool kInPlace = false, bool kKeep = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kWaves))) void k_render_wavefront(WfPass a)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t P = a.chunk_px;
    // The instances for tiles and for 7 and 8 resident waves per SIMD park the
    // path state that a trace does not read (17 values per lane) in LDS while
    // the trace runs: the state then needs no VGPRs there, and the trace fits
    // its register budget without spilling (17 KB of LDS per 256-lane
    // workgroup, 136 KB per CU at 8 waves per SIMD; a tile query's candidate
    // masks take another 14 KB).
    constexpr bool kPark = kWaves >= 7 || kTree;
    constexpr uint32_t kParked = 17;
    __shared__ uint32_t parked_all[4][kPark ? kParked : 1][64];
    uint32_t(*parked)[64] = parked_all[threadIdx.x >> 6];
    constexpr uint32_t kChunk = kKeep ? kTileChunkKeep : kInPlace ? kTileChunkInPlace : kTileChunk;
    __shared__ uint32_t tile_masks[4][kTree ? kChunk + 1 : 1][64];
    // in place: the pixel's primary direction, the frame its path is in, and the
    // primary ray's hit (sphere, t) if kept
    __shared__ uint32_t own_all[4][kKeep ? 6 : kInPlace ? 4 : 1][64];
    uint32_t(*own)[64] = own_all[threadIdx.x >> 6];

    // ---- wave-uniform scheduling state ----
    CScene* scenes = as_const(a.scenes);
    int32_t sid = -1;
    CScene* S = nullptr;
    int32_t pend = -1;              // a block of another scene, waiting for the lanes to drain
    bool qdone = false;
    bool first_fetch = true;
    uint32_t chunk_end = a.total_chunks;            // no chunk from here on holds a job
    const uint32_t n_waves = gridDim.x * 4u;
    const uint32_t wave_id = (uint32_t)__builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4u + (threadIdx.x >> 6)));
    uint32_t shard = wave_id % kQueueShards;        // the queue's counter this wave asks
    uint32_t dry = 0;                               // counters it has found used up
    uint32_t blk0 = 0, blk_next = 0, blk_end = 0;   // jobs left: [blk0 + next, blk0 + end) of scene S
    uint32_t slots = 0;                             // S's jobs per frame (job_slots)

    // ---- per-lane path state ----
    uint32_t state = kIdle;
    uint32_t job = 0, seed = 0;   // the scene's job index, PCG state
    int32_t bounce = 0;
    // (ro, rd): the lane's next ray -- the primary or continuation ray in
    // kCont, the shadow ray (from the hit towards the light) in kShadow;
    // vd: in kShadow, the direction of the ray that made the hit (the view
    // direction of the light's Cook-Torrance term)
    f3 ro = mk(0.0f, 0.0f, 0.0f), rd = ro, vd = ro, tp = ro, col = ro;
    f3 nrm = ro;                    // normal at the current hit
    float dist2 = 0.0f;             // in kShadow: squared distance to the light
    int32_t mid = 0;                // material of the current hit
    uint32_t lidx = 0;              // light of the current shadow ray
    bool capture = false;           // this path is the last frame's: write the debug capture
    // statistics: rays and cached rays per wave; test counts per lane, added
    // to the launch's 64-bit counters at the end (and earlier if one could
    // overflow); exact retraces (rare) straight to their counter
    unsigned long long rays = 0, reused = 0;
    uint32_t tests = 0, boxes = 0;
    // not kept: computed where it is used
    const auto counters = [&]() { return a.counters + (wave_id % kCounterLines) * kCounterStride; };

    const ATX_CONST WfPass& pass = kernel_pass();
    // in place: starts pixel `job`'s path of the launch's frame f
    const auto start_in_place = [&](uint32_t f, f3 dir) {
        own[3][lane] = f;
        ro = mk(S->cam_pos[0], S->cam_pos[1], S->cam_pos[2]);
        rd = dir;
        tp = mk(1.0f, 1.0f, 1.0f);
        col = mk(0.0f, 0.0f, 0.0f);
        seed = job * (pass.frame0 + f);
        bounce = 0;
        state = kCont;
        capture = (S->dbg_hit || S->dbg_shadow) && f + 1u == pass.frames;
        for (uint32_t i = 0; capture && i < S->dbg_bounces; ++i) {
            if (S->dbg_hit) S->dbg_hit[(size_t)job * S->dbg_bounces + i] = -2;
            if (S->dbg_shadow) S->dbg_shadow[(size_t)job * S->dbg_bounces + i] = -2;
        }
    };

    for (;;) {
        if constexpr (kKeep) {
            // Frames that start at a known primary hit: once a quarter of the
            // lanes that have a path wait for it, so that its shading runs for
            // several at a time but the last few do not wait for each other.
            const uint32_t again = (uint32_t)__popcll(__ballot(state == kAgain));
            if (again != 0u && 4u * again >= (uint32_t)__popcll(__ballot(state != kIdle)) && state == kAgain) {
                start_in_place(own[3][lane], mk(__uint_as_float(own[0][lane]), __uint_as_float(own[1][lane]),
                                                __uint_as_float(own[2][lane])));
                Hit h;
                h.id = (int32_t)own[4][lane];
                h.t = __uint_as_float(own[5][lane]);
                f3 so, L;
                mid = S->sph_mat[h.id];
                shade_hit(S, as_const(S->sph)[h.id], mid, h, ro, rd, tp, seed, col, nrm, so, lidx, L, dist2);
                vd = rd;
                ro = so;
                rd = L;
                state = kShadow;
            }
        }
        // ---------------- hand jobs to idle lanes (uniform control flow) ----------------
        for (;;) {
            const unsigned long long idle = __ballot(state == kIdle);
            if (idle == 0ull)
                break;
            // Jobs are handed out once refill_min lanes wait (or all do):
            // the hand-out and bounce 0 from the cache (about a sixth of the
            // kernel's time) then run for many lanes at once instead of for
            // the one or two whose paths just ended, while the waiting lanes
            // cost the trace loop little (its length is set by its slowest
            // lane).  1080p, A/B: 16 lanes 35.0 -> 34.0 ms per 256-frame
            // launch, 3.72 -> 3.44 ms per 20-frame one.
            if (idle != ~0ull && (uint32_t)__popcll(idle) < a.refill_min && blk_next < blk_end)
                break;
            if (blk_next < blk_end) {
                const uint32_t avail = blk_end - blk_next;
                const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(idle >> 32),
                                                                __builtin_amdgcn_mbcnt_lo((uint32_t)idle, 0u));
                const uint32_t nidle = (uint32_t)__popcll(idle);
                uint32_t cached_rays = 0;   // this lane's rays taken from the first-bounce cache
                if constexpr (kInPlace) {
                    if (state == kIdle && rank < avail) {
                        const uint32_t px = in_place_pixel(blk0 + blk_next + rank, S->width, S->height);
                        if (px != ~0u) {
                            job = px;
                            const f3 dir = primary_direction(S, px);
                            own[0][lane] = __float_as_uint(dir.x);
                            own[1][lane] = __float_as_uint(dir.y);
                            own[2][lane] = __float_as_uint(dir.z);
                            start_in_place(0u, dir);
                        }
                    }
                } else if (state == kIdle && rank < avail) {
                    job = blk0 + blk_next + rank;
                    uint32_t px, frame;
                    job_pixel_frame(job, slots, S->div_group, px, frame);
                    if (S->hit_px)
                        px = S->hit_px[px];
                    frame += S->frame0;
                    ro = mk(S->cam_pos[0], S->cam_pos[1], S->cam_pos[2]);
                    capture = (S->dbg_hit || S->dbg_shadow) && frame == S->frame0 + S->frames - 1u;
                    // bounce 0 from the first-bounce cache needs no primary
                    // direction unless the shadow ray is traced (too many lights)
                    const bool cached = S->first && !capture && S->max_bounces > 0;
                    if (cached && S->n_light <= kFirstMaxLights) {
                        rd = mk(0.0f, 0.0f, 0.0f);
                    } else if (S->dirs) {
                        const float4 dv = S->dirs[px];
                        rd = mk(dv.x, dv.y, dv.z);
                    } else {
                        rd = primary_direction(S, px);
                    }
                    tp = mk(1.0f, 1.0f, 1.0f);
                    col = mk(0.0f, 0.0f, 0.0f);
                    seed = px;   // x + y * W
                    seed *= frame;
                    bounce = 0;
                    if (capture) {
                        for (uint32_t i = 0; i < S->dbg_bounces; ++i) {
                            if (S->dbg_hit) S->dbg_hit[(size_t)px * S->dbg_bounces + i] = -2;
                            if (S->dbg_shadow) S->dbg_shadow[(size_t)px * S->dbg_bounces + i] = -2;
                        }
                    }
                    state = kCont;
                    if (cached) {
                        // bounce 0 from the first-bounce cache; the lane then enters
                        // the trace loop at its first continuation ray, or ends the
                        // path and takes another job
                        // the frame's light is known before the record arrives: issue
                        // the record's four loads and the light term's load together
                        const uint32_t nl = S->n_light;
                        const uint32_t lsel = nl > 0u ? umod(pcg_hash(seed), S->div_light) : 0u;
                        const uint4* fr = S->first + 4 * (size_t)px;
                        const uint4 r0 = fr[0], r1 = fr[1], r2 = fr[2], r3 = fr[3];
                        const float4 lt = S->first_light ? S->first_light[(size_t)lsel * (S->width * S->height) + px]
                                                         : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                        const int32_t hid = (int32_t)r0.x;
                        cached_rays = 1;
                        bool done = false;
                        if (hid < 0) {
                            if (S->sky_light)
                                col = add(col, mul(mk(0.6f, 0.7f, 0.9f), tp));
                            done = true;
                        } else if (S->n_light > kFirstMaxLights) {
                            // too many lights for the mask: shade the cached hit and
                            // trace the shadow ray
                            Hit h;
                            h.id = hid;
                            h.t = __uint_as_float(r0.y);
                            f3 so, L;
                            mid = (int32_t)r0.w;
                            shade_hit(S, as_const(S->sph)[h.id], mid, h, ro, rd, tp, seed, col, nrm, so, lidx, L, dist2);
                            vd = rd;
                            ro = so;
                            rd = L;
                            state = kShadow;
                        } else {
                            nrm = mk(__uint_as_float(r1.x), __uint_as_float(r1.y), __uint_as_float(r1.z));
                            ro = mk(__uint_as_float(r1.w), __uint_as_float(r2.x), __uint_as_float(r2.y));
                            col = mk(__uint_as_float(r2.z), __uint_as_float(r2.w), __uint_as_float(r3.x));
                            mid = (int32_t)r0.w;
                            if (nl > 0u) {
                                // the frame's light, and its term if it reaches the hit
                                lidx = lsel;
                                cached_rays = 2;
                                if ((r0.z >> lidx) & 1u)
                                    col = add(col, xyz(lt));
                            }
                            vd.x = __uint_as_float(r3.y);   // roughness, metallic
                            vd.y = __uint_as_float(r3.z);
                            done = roulette_first(S, mid, tp, seed);
                            state = kNew;
                        }
                        if (done) {
                            store_sample(S, slots, job, col);
                            state = kIdle;
                        }
                    }
                }
                reused += (unsigned long long)(__popcll(__ballot(cached_rays >= 1u)) +
                                               __popcll(__ballot(cached_rays >= 2u)));
                blk_next += nidle < avail ? nidle : avail;
                continue;
            }
            // the block is used up: take the next one
            int32_t c = pend;
            if (c < 0) {
                if (qdone)
                    break;
                // a wave's first chunk is its own index in the grid; the
                // counters hand out the chunks after the grid's first n_waves
                // (kQueueShards)
                uint32_t got = 0;
                if (first_fetch) {
                    got = wave_id;
                    first_fetch = false;
                } else {
                    if (lane == 0)
                        got = queue_chunk(shard, atomicAdd(a.queue + shard * kQueueStride, 1u), n_waves);
                    got = (uint32_t)__builtin_amdgcn_readfirstlane((int)got);
                }
                if (got >= chunk_end) {
                    // this counter is through (for good): go on with the next one
                    // that has chunks left; at most kQueueShards times
                    dry |= 1u << shard;
                    const uint32_t k = (shard + lane) % kQueueShards;
                    const unsigned long long left =
                        __ballot(lane < kQueueShards && !((dry >> k) & 1u) &&
                                 queue_chunk(k, __hip_atomic_load(a.queue + k * kQueueStride, __ATOMIC_RELAXED,
                                                                  __HIP_MEMORY_SCOPE_AGENT), n_waves) < chunk_end);
                    if (left == 0ull) {
                        qdone = true;
                        break;
                    }
                    shard = (shard + (uint32_t)__builtin_ctzll(left)) % kQueueShards;
                    continue;
                }
                c = (int32_t)got;
            }
            // a wave's chunks ascend but where it goes on to another counter
            int32_t s = sid < 0 || (uint32_t)c < scenes[sid].chunk_begin ? 0 : sid;
            while (s + 1 < (int32_t)a.n_scenes && (uint32_t)c >= scenes[s].chunk_begin + scenes[s].n_chunks)
                ++s;
            if (s != sid) {
                // a new scene: only once every lane has finished its path
                if (idle != ~0ull) {
                    pend = c;
                    break;
                }
                sid = s;
                S = &scenes[s];
                slots = (uint32_t)__builtin_amdgcn_readfirstlane((int)job_slots(S->hit_px, S->width * S->height));
            }
            pend = -1;
            const uint32_t jobs = kInPlace ? (uint32_t)in_place_jobs(S->width, S->height) : slots * S->frames;
            blk0 = ((uint32_t)c - S->chunk_begin) * P;
            blk_end = blk0 >= jobs ? 0u : (jobs - blk0 < P ? jobs - blk0 : P);
            blk_next = 0;
            // the host may lay a scene out for more jobs than its hit list
            // holds: past the last scene's jobs every later chunk is empty
            if (blk_end == 0u && s + 1 == (int32_t)a.n_scenes)
                chunk_end = (uint32_t)c;
        }
        if (!__any(state != kIdle) && qdone && pend < 0)
            break;
        // The next direction of every path that goes on: those of the last
        // round and those just handed out together, so that its 200
        // instructions run once per round.  Where each hand-out and each
        // bounce's end computed its own (about 3 per round at 1080p), the path
        // kernel issued 1890 VALU instructions per round instead of 1600
        // (1080p, 256 frames: 22.5 -> 20.0 ms).
        if (state == kNew) {
            next_direction(vd, nrm, rd, bounce, seed);
            state = kCont;
        }

        // ---------------- one closest-hit trace for every tracing lane ----------------
        const bool tracing = state == kCont || state == kShadow;
        bool end_path = state == kCont && S->max_bounces <= 0;   // zero bounces: black sample
        bool end_bounce = false;   // run light term + RR
        const bool traces = tracing && !end_path;
        rays += (unsigned long long)__popcll(__ballot(traces));
        const bool shadow = state == kShadow;
        Hit h;
        float4 hit_sphere;
        int32_t hit_mat;
        const bool tree = kTree && S && S->bvh.n_tiles != 0u;
        const auto query = [&]() {
            if constexpr (kPark) {
                const uint32_t v[kParked] = {__float_as_uint(col.x), __float_as_uint(col.y), __float_as_uint(col.z),
                                             __float_as_uint(tp.x),  __float_as_uint(tp.y),  __float_as_uint(tp.z),
                                             __float_as_uint(nrm.x), __float_as_uint(nrm.y), __float_as_uint(nrm.z),
                                             __float_as_uint(vd.x),  __float_as_uint(vd.y),  __float_as_uint(vd.z),
                                             seed, (uint32_t)bounce, job, (uint32_t)mid, lidx};
                for (uint32_t k = 0; k < kParked; ++k)
                    parked[k][lane] = v[k];
                // keep the compiler from forwarding the stored values past the trace
                __asm__ volatile("" ::: "memory");
            }
            const SphSrc flat{as_const(S->sph)};
            // the debug capture records the closest occluder; otherwise any proven one will do
            const float qd2 = (shadow && !(capture && S->dbg_shadow)) ? dist2 : -1.0f;
            BvhQuery q;
            if (tree) {
                const BvhDev B = S->bvh;
                h = trace_tiles<kChunk>(B, flat, S->sph_mat, S->n_sph, ro, rd, qd2, traces,
                                        capture || (kKeep && bounce == 0),
                                        tile_masks[threadIdx.x >> 6], q);
            } else {
                h = trace_filtered(flat, S->n_sph, ro, rd, q.exact);
                q.tests = S->n_sph;
                if (h.id >= 0 && !shadow) {
                    q.sphere = flat((uint32_t)h.id);
                    q.mat = S->sph_mat[h.id];
                }
            }
            hit_sphere = q.sphere;
            hit_mat = q.mat;
            if constexpr (kPark) {
                __asm__ volatile("" ::: "memory");
                col = mk(__uint_as_float(parked[0][lane]), __uint_as_float(parked[1][lane]),
                         __uint_as_float(parked[2][lane]));
                tp = mk(__uint_as_float(parked[3][lane]), __uint_as_float(parked[4][lane]),
                        __uint_as_float(parked[5][lane]));
                nrm = mk(__uint_as_float(parked[6][lane]), __uint_as_float(parked[7][lane]),
                         __uint_as_float(parked[8][lane]));
                if (shadow)
                    vd = mk(__uint_as_float(parked[9][lane]), __uint_as_float(parked[10][lane]),
                            __uint_as_float(parked[11][lane]));
                seed = parked[12][lane];
                bounce = (int32_t)parked[13][lane];
                job = parked[14][lane];
                mid = (int32_t)parked[15][lane];
                lidx = parked[16][lane];
            }
            if (traces) {
                if (q.exact)   // a trace counts once, however many orders were open
                    atomicAdd(counters() + kCtrExact, 1ull);
                tests += q.tests;
                boxes += q.boxes;
            }
        };

        const auto pixel = [&]() { return kInPlace ? job : job_pixel(S, slots, job); };
        const auto shade = [&]() {
            // ---------------- shading (divergent) ----------------
            if (!shadow) {
                if (capture && S->dbg_hit && (uint32_t)bounce < S->dbg_bounces)
                    S->dbg_hit[(size_t)pixel() * S->dbg_bounces + bounce] = h.id;
                if (kKeep && bounce == 0) {
                    own[4][lane] = (uint32_t)h.id;
                    own[5][lane] = __float_as_uint(h.t);
                }
                if (h.id < 0) {
                    if (S->sky_light)
                        col = add(col, mul(mk(0.6f, 0.7f, 0.9f), tp));
                    end_path = true;
                } else {
                    f3 so, L;
                    mid = hit_mat;
                    if (shade_hit(S, hit_sphere, mid, h, ro, rd, tp, seed, col, nrm, so, lidx, L, dist2)) {
                        vd = rd;
                        rd = L;
                        state = kShadow;
                        ro = so;
                    } else {
                        ro = so;
                        end_bounce = true;
                    }
                }
            } else {
                if (capture && S->dbg_shadow && (uint32_t)bounce < S->dbg_bounces)
                    S->dbg_shadow[(size_t)pixel() * S->dbg_bounces + bounce] = h.id;
                end_bounce = true;
            }
        };
        if constexpr (kTree) {
            if (tree || traces)   // every lane takes part in a tile query's matrix products
                query();
            if (traces)
                shade();
        } else if (traces) {
            query();
            shade();
        }
        if (end_bounce) {
            // The material once, for the light's term and the roulette; a light's
            // radiance as one product; the first-bounce record names roughness and
            // metallic; emission, hit ids and a shadow hit's sphere are loaded only
            // where they are used: 2.5e8 instead of 3.0e8 vector loads in 256
            // frames of 1080p with 257 spheres (the return path of loads was busy
            // 92 % of the time).  Whole calls 21.41 -> 21.29 ms, 20 frames 2.81 ->
            // 2.78, 640x360 with 4 spheres, 64 frames 0.710 -> 0.691.
            const float4 m0 = S->mat[3 * mid], m1 = S->mat[3 * mid + 1];
            if (shadow && lit_by(h, dist2))
                col = add(col, light_term(m0, m1, S->light[2 * lidx + 1], nrm, vd, rd, tp, S->mild != 0u));
            // the next ray leaves from the hit's offset origin, which ro holds
            if (roulette(S, m0, m1.w, tp, bounce, seed, vd))
                end_path = true;
            else
                state = kNew;
        }
        if (__any(tests >= 0x80000000u || boxes >= 0x80000000u))
            flush_counters(counters(), lane, tests, boxes, 0ull, 0ull);
        if (end_path) {
            state = kIdle;
            if constexpr (kInPlace) {
                const uint32_t f = own[3][lane];
                // the debug captures trace every ray; without lights the hit's
                // bounce ends where it is shaded
                const bool known = kKeep && S->n_light != 0 && S->max_bounces > 0 && !S->dbg_hit && !S->dbg_shadow;
                const bool miss = known && (int32_t)own[4][lane] < 0;
                const uint32_t n = miss ? pass.frames - f : 1u;
                add_sample(S, pass, job, f, n, col);
                if (f + n < pass.frames) {
                    own[3][lane] = f + n;
                    if (known)
                        state = kAgain;
                    else
                        start_in_place(f + n, mk(__uint_as_float(own[0][lane]), __uint_as_float(own[1][lane]),
                                                 __uint_as_float(own[2][lane])));
                }
            } else {
                store_sample(S, slots, job, col);
            }
        }
    }

    flush_counters(counters(), lane, tests, boxes, rays, reused);
}

// In-place launches of scenes without tiles: a lane per pixel, a wave per 8 x 8
// pixels, both rays of a bounce in one round, so that a path's chain of dependent
// instructions, which bounds it (the loads and square roots of one ray after the
// other), stays short.  The persistent kernel's in-place mode, whose round is one ray
// and which hands out pixels, took longer at every size (one frame, 13 spheres:
// 64x64 51 us, here 32; 640x360 97 and 50; 1920x1080 223 and 98).
// kFrames: a lane goes on to its next frame without waiting for the others and
// keeps its primary hit (1280x720, 13 spheres, 32 frames: 1.54 ms with a loop over
// frames around one over bounces, 1.33 with this one, 1.88 persistent).  A launch of
// one frame has an instance of its own, 8 % shorter.
template <bool kFrames>
__global__ __launch_bounds__(64) void k_render_flat(WfPass a)
{
    CScene* const S = as_const(a.scenes);
    const ATX_CONST WfPass& pass = kernel_pass();
    const uint32_t lane = threadIdx.x;
    const uint32_t px = in_place_pixel(blockIdx.x * 64u + lane, S->width, S->height);
    const SphSrc flat{as_const(S->sph)};
    uint32_t rays = 0, exact = 0;   // this lane's
    if (px != ~0u) {
        const f3 eye = mk(S->cam_pos[0], S->cam_pos[1], S->cam_pos[2]), dir = primary_direction(S, px);
        const bool debug = S->dbg_hit || S->dbg_shadow;
        const auto trace = [&](f3 o, f3 d) {
            ++rays;
            return S->exact ? trace_exact(flat, S->n_sph, o, d) : trace_filtered(flat, S->n_sph, o, d, exact);
        };
        uint32_t f = 0, seed = 0;
        int32_t bounce = 0;
        f3 ro, rd, tp, col;
        bool capture = false;
        const auto start = [&]() {   // the path of frame f
            ro = eye;
            rd = dir;
            tp = mk(1.0f, 1.0f, 1.0f);
            col = mk(0.0f, 0.0f, 0.0f);
            seed = px * (pass.frame0 + f);
            bounce = 0;
            capture = debug && f + 1u == pass.frames;
            for (uint32_t i = 0; capture && i < S->dbg_bounces; ++i) {
                if (S->dbg_hit) S->dbg_hit[(size_t)px * S->dbg_bounces + i] = -2;
                if (S->dbg_shadow) S->dbg_shadow[(size_t)px * S->dbg_bounces + i] = -2;
            }
        };
        // one bounce; true when the path ends
        Hit first;   // the primary ray's
        first.id = -1;
        first.t = FLT_MAX;
        const auto step = [&]() -> bool {
            if (S->max_bounces <= 0)
                return true;
            Hit h = first;
            if (!kFrames || bounce != 0 || f == 0u)
                h = trace(ro, rd);
            if (kFrames && bounce == 0)
                first = h;
            const size_t at = (size_t)px * S->dbg_bounces + (uint32_t)bounce;
            const bool record = capture && (uint32_t)bounce < S->dbg_bounces;
            if (record && S->dbg_hit)
                S->dbg_hit[at] = h.id;
            if (h.id < 0) {
                if (S->sky_light)
                    col = add(col, mul(mk(0.6f, 0.7f, 0.9f), tp));
                return true;
            }
            const int32_t mid = S->sph_mat[h.id];
            const float4 m0 = S->mat[3 * mid], m1 = S->mat[3 * mid + 1];
            f3 nrm, so, L, surface;
            uint32_t lidx = 0;
            float dist2 = 0.0f;
            if (shade_hit(S, flat((uint32_t)h.id), mid, h, ro, rd, tp, seed, col, nrm, so, lidx, L, dist2)) {
                const Hit sh = trace(so, L);
                if (record && S->dbg_shadow)
                    S->dbg_shadow[at] = sh.id;
                if (lit_by(sh, dist2))
                    col = add(col, light_term(m0, m1, S->light[2 * lidx + 1], nrm, rd, L, tp, S->mild != 0u));
            }
            if (roulette(S, m0, m1.w, tp, bounce, seed, surface))
                return true;
            ro = so;
            next_direction(surface, nrm, rd, bounce, seed);
            return false;
        };
        start();
        if constexpr (!kFrames) {
            while (!step()) {
            }
            add_sample(S, pass, px, 0u, 1u, col);
        } else {
            while (f < pass.frames) {
                if (step()) {
                    // a primary ray that misses does so in every frame
                    const bool miss = bounce == 0 && first.id < 0 && !debug;
                    const uint32_t n = miss ? pass.frames - f : 1u;
                    add_sample(S, pass, px, f, n, col);
                    f += n;
                    if (f < pass.frames)
                        start();
                }
            }
        }
    }
    const unsigned long long r = wave_sum(rays), e = wave_sum(exact);
    const unsigned long long v = lane == kCtrRays ? r : lane == kCtrTests ? r * S->n_sph : lane == kCtrExact ? e : 0ull;
    if (v)
        atomicAdd(a.counters + (blockIdx.x % kCounterLines) * kCounterStride + lane, v);
}

// Adds every pixel's samples of the launch to its accumulation in frame order
// (Renderer.cu:164-165; frame 1 starts from zero, which is what the
// reference's memset provides) and writes the RGBA8 value (Renderer.cu:166-168,
// Renderer.h:70-78).  One lane per pixel of the launch's pixel range; a
// pixel's samples lie at job_of(slot, f), m samples apart from one frame to
// the next (m = 8 but in a scene's last group of slots).
__global__ __launch_bounds__(256) void k_accumulate(WfPass a)
{
    const uint32_t g = blockIdx.x * 256u + threadIdx.x;
    if (a.totals && blockIdx.x == 0u && threadIdx.x <= kCtrCount) {
        unsigned long long s = 0;
        if (threadIdx.x == kCtrCount)
            s = a.n_hits ? *a.n_hits : 0u;
        else
            for (uint32_t k = 0; k < kCounterLines; ++k)
                s += a.counters[k * kCounterStride + threadIdx.x];
        a.totals[threadIdx.x] = s;
    }
    if (g >= a.total_px)
        return;
    uint32_t lo = 0, hi = a.n_scenes;          // last scene with px_begin <= g
    while (hi - lo > 1u) {
        const uint32_t mid = (lo + hi) / 2u;
        if (a.scenes[mid].px_begin <= g) lo = mid;
        else hi = mid;
    }
    const WfScene& S = a.scenes[lo];
    const uint32_t npx = S.width * S.height;
    const uint32_t px = g - S.px_begin;
    if (px >= npx)
        return;
    const bool first = S.frame0 == 1u;
    // a pixel left out of the jobs (its primary ray misses): every frame's
    // sample is the one such a path returns, the sky colour or black
    uint32_t slot = S.hit_px ? __float_as_uint(S.dirs[px].w) : px;
    const bool sky = slot == kNoSlot;
    slot = sky ? 0u : slot;
    const float4 sky_c = S.sky_light ? make_float4(0.6f, 0.7f, 0.9f, 1.0f) : make_float4(0.0f, 0.0f, 0.0f, 1.0f);
    float4 acc = first ? make_float4(0.0f, 0.0f, 0.0f, 0.0f) : S.accum[px];
    // this pixel's samples: frame f at sp[f * step] (slots are hit-list
    // indices with a hit list, else pixels; a sky pixel has none)
    const uint32_t slots = job_slots(S.hit_px, npx);
    const uint32_t left = slots - (slot & ~(kJobGroupPx - 1u));
    const uint32_t step = left < kJobGroupPx ? left : kJobGroupPx;
    const ATX_GLOBAL float3* sp = (const ATX_GLOBAL float3*)(uintptr_t)S.samples + job_of(slot, 0u, slots, S.frames);
    if (S.kahan) {
        float4 cp = first ? make_float4(0.0f, 0.0f, 0.0f, 0.0f) : S.comp[px];
        const auto add = [&](const float4 c) {
            float yv, t;
            yv = c.x - cp.x; t = acc.x + yv; cp.x = (t - acc.x) - yv; acc.x = t;
            yv = c.y - cp.y; t = acc.y + yv; cp.y = (t - acc.y) - yv; acc.y = t;
            yv = c.z - cp.z; t = acc.z + yv; cp.z = (t - acc.z) - yv; acc.z = t;
            yv = c.w - cp.w; t = acc.w + yv; cp.w = (t - acc.w) - yv; acc.w = t;
        };
        // two loops: a select between sky_c and a loaded sample becomes a
        // select of addresses, and sky_c then lives in scratch memory
        if (sky) {
            for (uint32_t f = 0; f < S.frames; ++f)
                add(sky_c);
        } else {
            for (uint32_t f = 0; f < S.frames; ++f) {
                const float3 c = sp[(size_t)f * step];
                add(make_float4(c.x, c.y, c.z, 1.0f));
            }
        }
        S.comp[px] = cp;
    } else if (sky) {
        for (uint32_t f = 0; f < S.frames; ++f) {
            acc.x = acc.x + sky_c.x;
            acc.y = acc.y + sky_c.y;
            acc.z = acc.z + sky_c.z;
            acc.w = acc.w + sky_c.w;
        }
    } else {
        // four frames' loads in flight ahead of their additions (in frame
        // order); every sample's alpha is 1
        uint32_t f = 0;
        for (; f + 4u <= S.frames; f += 4u) {
            float3 c[4];
            for (int k = 0; k < 4; ++k)
                c[k] = sp[(size_t)(f + k) * step];
            for (int k = 0; k < 4; ++k) {
                acc.x = acc.x + c[k].x;
                acc.y = acc.y + c[k].y;
                acc.z = acc.z + c[k].z;
                acc.w = acc.w + 1.0f;
            }
        }
        for (; f < S.frames; ++f) {
            const float3 c = sp[(size_t)f * step];
            acc.x = acc.x + c.x;
            acc.y = acc.y + c.y;
            acc.z = acc.z + c.z;
            acc.w = acc.w + 1.0f;
        }
    }
    S.accum[px] = acc;
    S.image[px] = display(acc, S.frame0 + S.frames - 1u);
}

struct CamDirArgs {
    float inv_proj[16];
    float inv_view[16];
    uint32_t width, height;
    float4* dirs;
};

__global__ __launch_bounds__(256) void k_camera_dirs(CamDirArgs c)
{
    const uint32_t px = blockIdx.x * 256u + threadIdx.x;
    if (px >= c.width * c.height)
        return;
    const uint32_t y = px / c.width, x = px - y * c.width;
    const f3 d = camera_ray(c.inv_proj, c.inv_view, x, y, c.width, c.height);
    c.dirs[px] = make_float4(d.x, d.y, d.z, 0.0f);
}

struct FirstArgs {
    WfScene s;
    uint4* rec;        // 4 per pixel
    float4* light;     // [light][pixel], or nullptr
    uint32_t* hits;    // pixels whose primary ray hits, appended
    float4* dirs;      // s.dirs, whose w takes each pixel's index among them
    uint32_t* n_hits;  // their count (zero before the launch)
};

// One lane per pixel: the primary ray's closest hit, the shading at it, and
// for scenes of at most kFirstMaxLights lights each light's shadow decision
// and Cook-Torrance term, with the path kernel's expressions (hit_frame,
// add_emission, light_ray, lit_by, light_term; tp = 1 at bounce 0) and
// queries, so the cached values are the ones every frame's path computes.
// A wave takes an 8 x 8 tile of pixels: its rays stay closer together than
// along a 64-pixel row (1080p: 0.586 -> 0.556 ms), and the hit list then
// runs tile by tile.
// A workgroup appends its hits to the list with one atomic (one per 11.6 ns on
// the device, whoever asks): one per wave bounded the kernel, 1080p with 257
// spheres 0.376 -> 0.295 ms, 640x360 with 4 0.042 -> 0.016 ms.  With tiles 4 waves,
// which wait less for each other (8: 0.311 ms; 1600x900, 8000 spheres 1.12 and
// 1.19), else 8 (4: 0.020 ms, 16: 0.015).
template <bool kTree>
constexpr uint32_t kFirstWaves = kTree ? 4 : 8;
template <bool kTree>
__global__ __launch_bounds__(kFirstWaves<kTree> * 64) void k_first_hit(FirstArgs a)
{
    const WfScene& s = a.s;
    const uint32_t npx = s.width * s.height;
    // one 8 x 8 tile of pixels per wave
    const uint32_t tiles_x = (s.width + 7u) / 8u;
    const uint32_t wave = blockIdx.x * kFirstWaves<kTree> + (threadIdx.x >> 6);
    const uint32_t ty = wave / tiles_x, tx = wave - ty * tiles_x;
    const uint32_t x = tx * 8u + (threadIdx.x & 7u), y = ty * 8u + ((threadIdx.x >> 3) & 7u);
    // lanes past the image's edge stay for the wave's tile queries
    const bool in = x < s.width && y < s.height;
    const uint32_t px = in ? y * s.width + x : 0u;
    const f3 ro = mk(s.cam_pos[0], s.cam_pos[1], s.cam_pos[2]);
    const float4 dv = s.dirs[px];
    const f3 rd = mk(dv.x, dv.y, dv.z);
    const SphSrc flat{as_const(s.sph)};
    __shared__ uint32_t tile_masks[kFirstWaves<kTree>][kTree ? kTileChunk + 1 : 1][64];
    __shared__ uint32_t wave_hits[kFirstWaves<kTree>], list_base;
    const BvhDev B = s.bvh;
    const f3 one = mk(1.0f, 1.0f, 1.0f);
    const f3 zero = mk(0.0f, 0.0f, 0.0f);
    f3 pos = zero, nrm = zero, so = zero, col = zero;
    Hit first;   // the primary hit
    first.id = -1;
    first.t = FLT_MAX;
    int32_t mid = 0;
    float4 hit_sphere = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    uint32_t mask = 0u;
    uint32_t slot = kNoSlot;   // index in the hit list
    // the primary ray, then a shadow ray towards each light (one query in the
    // code: a second copy of it would take the registers of both)
    const uint32_t n_rays = 1u + (a.light ? s.n_light : 0u);
    for (uint32_t k = 0; k < n_rays; ++k) {
        const bool hit = first.id >= 0, act = k == 0u ? in : hit;
        f3 o = ro, d = rd;
        float dist2 = -1.0f;
        if (k > 0u) {
            o = so;
            d = one;
            if (hit)
                light_ray(s.light[2 * (k - 1u)], pos, d, dist2);
        }
        Hit h;
        h.id = -1;
        h.t = FLT_MAX;
        if constexpr (kTree) {
            BvhQuery q;
            if (__any(act))   // a wave of missing pixels has no shadow rays
                h = trace_tiles<kTileChunk>(B, flat, s.sph_mat, s.n_sph, o, d, dist2, act, k == 0u,
                                            tile_masks[threadIdx.x >> 6], q);
            if (k == 0u) {
                hit_sphere = q.sphere;
                mid = q.mat;
            }
        } else if (act) {
            uint32_t ex = 0;
            h = trace_filtered(flat, s.n_sph, o, d, ex);
            if (k == 0u && h.id >= 0) {
                hit_sphere = flat((uint32_t)h.id);
                mid = s.sph_mat[h.id];
            }
        }
        if (k == 0u) {
            first = h;
            if (!in)
                first.id = -1;
            // append the workgroup's hit pixels to the list (every wave comes
            // here once)
            const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
            const unsigned long long hm = __ballot(first.id >= 0);
            if (lane == 0)
                wave_hits[w] = (uint32_t)__popcll(hm);
            __syncthreads();
            uint32_t base = 0, all = 0;
            for (uint32_t i = 0; i < kFirstWaves<kTree>; ++i) {
                const uint32_t n = wave_hits[i];
                base += i < w ? n : 0u;
                all += n;
            }
            if (threadIdx.x == 0)
                list_base = all ? atomicAdd(a.n_hits, all) : 0u;
            __syncthreads();
            base += list_base;
            if (first.id >= 0) {
                const unsigned long long below = lane == 0 ? 0ull : (~0ull >> (64u - lane));
                slot = base + (uint32_t)__popcll(hm & below);
                a.hits[slot] = px;
                hit_frame(hit_sphere, first, ro, rd, pos, nrm, so);
                add_emission(s.mat[3 * mid + 2], one, col);
            }
        } else if (in) {
            const uint32_t l = k - 1u;
            f3 term = zero;
            if (hit && lit_by(h, dist2)) {
                mask |= 1u << l;
                term = light_term(s.mat[3 * mid], s.mat[3 * mid + 1], s.light[2 * l + 1], nrm, rd, d, one, s.mild != 0u);
            }
            a.light[(size_t)l * npx + px] = make_float4(term.x, term.y, term.z, 0.0f);
        }
    }
    if (!in)
        return;
    a.dirs[px].w = __uint_as_float(slot);
    uint4* r = a.rec + 4 * (size_t)px;
    r[0] = make_uint4((uint32_t)first.id, __float_as_uint(first.t), mask, (uint32_t)mid);
    r[1] = make_uint4(__float_as_uint(nrm.x), __float_as_uint(nrm.y), __float_as_uint(nrm.z), __float_as_uint(so.x));
    r[2] = make_uint4(__float_as_uint(so.y), __float_as_uint(so.z), __float_as_uint(col.x), __float_as_uint(col.y));
    float rough = 0.0f, metallic = 0.0f;
    if (first.id >= 0) {
        rough = s.mat[3 * mid].w;
        metallic = s.mat[3 * mid + 1].w;
    }
    r[3] = make_uint4(__float_as_uint(col.z), __float_as_uint(rough), __float_as_uint(metallic), 0u);
}

__global__ void k_zero_u32(unsigned int* p, uint32_t n)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

// The path kernel's instance for a launch (wf_waves).
using PathKernel = void (*)(WfPass);
PathKernel path_kernel(bool flat_only, uint32_t waves)
{
    if (!flat_only)
        return k_render_wavefront<kWfWavesTree, true>;
    switch (wf_waves(waves, flat_only)) {
    case 5: return k_render_wavefront<5, false>;
    case 6: return k_render_wavefront<6, false>;
    case 7: return k_render_wavefront<7, false>;
    default: return k_render_wavefront<8, false>;
    }
}

}  // namespace

hipError_t launch_wavefront(const WfPass& pass, const WfLaunch& l, hipStream_t stream, hipEvent_t paths_done)
{
    if (pass.total_px == 0)
        return hipSuccess;
    WfPass p = pass;
    static const uint32_t refill = [] {
        const char* env = getenv("ATX_WF_REFILL");
        const long v = env ? strtol(env, nullptr, 10) : (long)kRefillMin;
        return (uint32_t)(v < 1 ? 1 : v > 64 ? 64 : v);
    }();
    p.refill_min = refill;
    if (p.chunk_px == 0 || p.chunk_px % 64 != 0 || p.chunk_px > kMaxChunkPx)
        return hipErrorInvalidValue;
    // no jobs (every pixel's primary ray misses): k_accumulate alone
    if (p.total_chunks > 0) {
        // no workgroup without a first chunk for a wave
        const uint32_t most = (p.total_chunks + 3u) / 4u;
        hipLaunchKernelGGL(path_kernel(l.flat_only, l.waves), dim3(l.workgroups < most ? l.workgroups : most),
                           dim3(256), 0, stream, p);
    }
    hipError_t e = hipGetLastError();
    if (e == hipSuccess && paths_done)
        e = hipEventRecord(paths_done, stream);
    if (e != hipSuccess)
        return e;
    hipLaunchKernelGGL(k_accumulate, dim3((p.total_px + 255u) / 256u), dim3(256), 0, stream, p);
    return hipGetLastError();
}

hipError_t launch_in_place(const WfScene& s, const WfPass& pass, hipStream_t stream)
{
    WfPass p = pass;
    p.refill_min = kRefillMin;
    if (p.total_chunks == 0 || p.n_scenes != 1 || p.frames == 0)
        return hipErrorInvalidValue;
    if (s.bvh.n_tiles == 0u) {
        hipLaunchKernelGGL(p.frames > 1u ? k_render_flat<true> : k_render_flat<false>, dim3(p.total_chunks), dim3(64),
                           0, stream, p);
        return hipGetLastError();
    }
    const PathKernel kernel = p.frames >= kKeepFrames ? k_render_wavefront<kWfWavesTree, true, true, true>
                                                      : k_render_wavefront<kWfWavesTree, true, true>;
    int dev = 0, cus = 0, blocks = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, kernel, 256, 0);
    if (e != hipSuccess)
        return e;
    const uint32_t full = (uint32_t)(cus > 0 ? cus : 1) * (uint32_t)(blocks > 0 ? blocks : 1);
    const uint32_t most = (p.total_chunks + 3u) / 4u;   // a first chunk for each wave
    hipLaunchKernelGGL(kernel, dim3(full < most ? full : most), dim3(256), 0, stream, p);
    return hipGetLastError();
}

hipError_t launch_camera_dirs(const WfScene& s, float4* dirs, hipStream_t stream)
{
    const uint32_t n = s.width * s.height;
    if (n == 0)
        return hipSuccess;
    CamDirArgs c;
    for (int k = 0; k < 16; ++k) {
        c.inv_proj[k] = s.inv_proj[k];
        c.inv_view[k] = s.inv_view[k];
    }
    c.width = s.width;
    c.height = s.height;
    c.dirs = dirs;
    hipLaunchKernelGGL(k_camera_dirs, dim3((n + 255u) / 256u), dim3(256), 0, stream, c);
    return hipGetLastError();
}

hipError_t launch_first_hits(const WfScene& s, hipStream_t stream)
{
    const uint32_t n = s.width * s.height;
    if (n == 0)
        return hipSuccess;
    const bool lights = s.n_light >= 1 && s.n_light <= kFirstMaxLights;
    if (!s.dirs || !s.first || lights != (s.first_light != nullptr))
        return hipErrorInvalidValue;
    const FirstCacheView v = first_cache_view(const_cast<uint4*>(s.first), n, s.n_light);
    FirstArgs a;
    a.s = s;
    a.rec = v.rec;
    a.light = v.light;
    a.hits = v.hits;
    a.dirs = const_cast<float4*>(s.dirs);
    a.n_hits = v.n_hits;
    hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(64), 0, stream, v.n_hits, 1u);
    const uint32_t tiles = ((s.width + 7u) / 8u) * ((s.height + 7u) / 8u);
    const auto kernel = s.bvh.n_tiles ? k_first_hit<true> : k_first_hit<false>;
    const uint32_t waves = s.bvh.n_tiles ? kFirstWaves<true> : kFirstWaves<false>;
    hipLaunchKernelGGL(kernel, dim3((tiles + waves - 1u) / waves), dim3(waves * 64u), 0, stream, a);
    return hipGetLastError();
}

hipError_t launch_zero_u32(unsigned int* p, uint32_t n, hipStream_t stream)
{
    if (n == 0)
        return hipSuccess;
    hipLaunchKernelGGL(k_zero_u32, dim3((n + 255) / 256), dim3(256), 0, stream, p, n);
    return hipGetLastError();
}

int wavefront_max_blocks_per_cu(bool flat_only, uint32_t waves)
{
    int blocks = 0;
    const hipError_t e =
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, path_kernel(flat_only, waves), 256, 0);
    if (e != hipSuccess)
        return 1;
    return blocks > 0 ? blocks : 1;
}

}  // namespace atx
