// render_noalloc.hip -- the allocation-free render entry point.
//
// atx_render_frames_noalloc renders frames of one scene in place
// (launch_in_place: every pixel's frames one after another in one lane, up to
// kInPlaceFrames frames of the call in a launch), with the results of
// atx_renderer_render_frames, but allocates no device memory: the caller
// passes the accumulation, compensation and image buffers, and everything else
// the kernel reads (the scene in its device layout, its tiles, the table entry,
// the queue and the statistics counters) lives in one file-scope device array,
// `scratch`, of kScratchBytes.  It is for callers that cannot call hipMalloc
// (serving loops, harnesses that forbid allocation).
//
// Each device holds its own copy of `scratch` for the life of the process,
// at its own address; that address is looked up once per device with
// hipGetSymbolAddress and only the looked-up pointer is handed to kernels and
// copies (the symbol's host-side name is not a device address).  Every call
// on a device shares its array: calls that overlap on one device (two host
// threads, or two streams) race on it.  A call returns after its frames are
// rendered, so consecutive calls on one thread do not overlap.
#include <algorithm>
#include <mutex>
#include <string.h>
#include <vector>

#include "camera_host.h"
#include "device_types.h"
#include "host_common.h"
#include "wavefront_host.h"

namespace atx {
namespace {

constexpr size_t kScratchBytes = 8u << 20;   // per device: 8 MiB for the scene
constexpr size_t kControlBytes = 8192;       // and two pages for counters, queue and table entry, before it
constexpr int kMaxDevices = 64;

static __device__ __align__(256) unsigned char scratch[kScratchBytes + kControlBytes];

std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// Device address of this device's `scratch`, looked up on the first call
// made with the device current.
int scratch_address(int dev, unsigned char** out)
{
    ATX_CHECK_ARG(dev >= 0 && dev < kMaxDevices, "device %d out of range", dev);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        ATX_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        ATX_CHECK_ARG(p != nullptr, "scratch has no device address");
        g_scratch_ptr[dev] = p;
    }
    *out = static_cast<unsigned char*>(g_scratch_ptr[dev]);
    return ATX_OK;
}

}  // namespace
}  // namespace atx

using namespace atx;

extern "C" int atx_render_frames_noalloc(const atx_sphere* spheres, uint64_t num_spheres,
                                         const atx_material* materials, uint64_t num_materials,
                                         const atx_light* lights, uint64_t num_lights, const atx_settings* settings,
                                         const atx_camera* cam, uint32_t first_frame, uint32_t frames, int accel,
                                         int accumulator, float* accum, float* comp, uint32_t* image,
                                         void* stream_handle)
{
    ATX_CHECK_ARG(settings && cam, "settings or camera is NULL");
    ATX_CHECK_ARG(cam->width > 0 && cam->height > 0, "Width or height cannot be zero");
    ATX_CHECK_ARG(settings->max_bounces >= 0, "max_bounces must be >= 0");
    ATX_CHECK_ARG(first_frame >= 1, "first_frame must be >= 1 (the reference's frame index starts at 1)");
    ATX_CHECK_ARG(accel == ATX_ACCEL_BVH || accel == ATX_ACCEL_NONE, "unknown accel %d", accel);
    ATX_CHECK_ARG(accumulator == ATX_ACCUM_NAIVE || accumulator == ATX_ACCUM_KAHAN, "unknown accumulator %d",
                  accumulator);
    ATX_CHECK_ARG(accum && image, "accum and image must be device buffers of width*height entries");
    ATX_CHECK_ARG(accumulator == ATX_ACCUM_NAIVE || comp, "Kahan accumulation needs the comp buffer");
    if (frames == 0) return ATX_OK;
    ATX_CHECK_ARG(!settings->accumulation || first_frame + (frames - 1u) >= first_frame, "frame index overflows");

    HostSceneLayout L;
    int rc = build_scene_layout(spheres, num_spheres, materials, num_materials, lights, num_lights, &L);
    if (rc != ATX_OK) return rc;
    HostBvh tiles;
    const HostBvh none;
    build_bvh(L.sph.data(), (uint32_t)num_spheres, 0, &tiles);
    // scratch layout: counters | queue | table entry, then from kControlBytes on
    // spheres | material ids | materials | lights | tiles
    const size_t off_queue = kCounterBytes;
    const size_t off_table = off_queue + kQueueWords * sizeof(unsigned int);
    static_assert(kCounterBytes % 256 == 0 && kQueueWords % 64 == 0, "aligned parts");
    static_assert(kCounterBytes + kQueueWords * sizeof(unsigned int) + sizeof(WfScene) <= kControlBytes,
                  "control pages");
    // a scene that fits only without its tiles has none; without lookups, so that
    // as many spheres as possible fit
    const ScenePack with_tiles(L, tiles, false, 256), bare(L, none, false, 256);
    const bool tiled = with_tiles.bytes <= kScratchBytes;
    const HostBvh& T = tiled ? tiles : none;
    const ScenePack& pack = tiled ? with_tiles : bare;
    const size_t total = pack.bytes;
    if (total > kScratchBytes) {
        set_error("scene needs %zu bytes of device scratch; atx_render_frames_noalloc holds at most %zu "
                  "(use atx_renderer_* for larger scenes)",
                  total, kScratchBytes);
        return ATX_ERR_INVALID;
    }

    int dev = 0;
    ATX_HIP(hipGetDevice(&dev));
    unsigned char* base = nullptr;
    rc = scratch_address(dev, &base);
    if (rc != ATX_OK) return rc;
    hipStream_t stream = static_cast<hipStream_t>(stream_handle);

    unsigned char* const scene = base + kControlBytes;
    WfScene w{};
    w.sph = pack.at<float4>(scene, ScenePack::kSph);
    w.sph_mat = pack.at<int32_t>(scene, ScenePack::kSphMat);
    w.mat = pack.at<float4>(scene, ScenePack::kMat);
    w.light = pack.at<float4>(scene, ScenePack::kLight);
    w.n_sph = (uint32_t)num_spheres;
    w.n_mat = (uint32_t)num_materials;
    w.n_light = (uint32_t)num_lights;
    w.mild = mild_materials(L.least_albedo, L.unit_materials, settings->max_bounces) ? 1u : 0u;
    w.emits = L.emits ? 1u : 0u;
    w.bvh = pack.bvh(T, scene);
    if (accel != ATX_ACCEL_BVH) w.bvh.n_nodes = 0;
    const bool kahan = accumulator == ATX_ACCUM_KAHAN;
    fill_wf_view(*settings, *cam, reinterpret_cast<float4*>(accum), kahan ? reinterpret_cast<float4*>(comp) : nullptr,
                 image, kahan, first_frame, settings->accumulation ? std::min(frames, kInPlaceFrames) : 1u, &w);
    WfPass p{};
    ATX_CHECK_ARG(layout_in_place(w, &p), "viewport too large");
    p.scenes = reinterpret_cast<const WfScene*>(base + off_table);
    p.queue = reinterpret_cast<unsigned int*>(base + off_queue);
    p.counters = reinterpret_cast<unsigned long long*>(base);
    // One launch for up to kInPlaceFrames frames; with accumulation off a launch
    // per frame, the index back at 1 after the first (Renderer.cu:245-248).  The
    // table entry, the queue and the counters (both zero) go up with the scene, in
    // one copy (two copies and two fill kernels less: 1280x720, 129 spheres, 4 frames
    // 635 -> 629 us).
    std::vector<unsigned char> block(kControlBytes, 0);
    memcpy(block.data() + off_table, &w, sizeof(w));
    const std::vector<unsigned char> packed = pack.block();
    block.insert(block.end(), packed.begin(), packed.end());
    hipError_t e = hipMemcpyAsync(base, block.data(), block.size(), hipMemcpyHostToDevice, stream);
    for (uint32_t left = frames; left > 0 && e == hipSuccess;) {
        e = launch_in_place(w, p, stream);
        left -= p.frames;
        p.frame0 = settings->accumulation ? p.frame0 + p.frames : 1u;
        p.frames = std::min(left, p.frames);
        if (e == hipSuccess && left > 0) e = launch_zero_u32(p.queue, kQueueWords, stream);
    }
    // the copy reads `block`, which ends with this call
    const hipError_t done = hipStreamSynchronize(stream);
    ATX_HIP(e != hipSuccess ? e : done);
    return ATX_OK;
}
