// host_common.cpp -- error state, scene layout, device queries, camera C ABI.
#include "host_common.h"

#include <stdlib.h>
#include <string.h>

#include "camera_host.h"

namespace atx {

static thread_local std::string g_last_error;

void set_error(const char* fmt, ...)
{
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_last_error = buf;
}

int build_scene_layout(const atx_sphere* spheres, uint64_t n, const atx_material* materials,
                       uint64_t m, const atx_light* lights, uint64_t l, HostSceneLayout* out)
{
    ATX_CHECK_ARG(n == 0 || spheres, "spheres is NULL with num_spheres=%llu", (unsigned long long)n);
    ATX_CHECK_ARG(m == 0 || materials, "materials is NULL with num_materials=%llu", (unsigned long long)m);
    ATX_CHECK_ARG(l == 0 || lights, "lights is NULL with num_lights=%llu", (unsigned long long)l);
    ATX_CHECK_ARG(n < (1ull << 31) && m < (1ull << 28) && l < (1ull << 28), "scene too large");
    if (n > 0 && m == 0) {
        set_error("scene has %llu spheres but no material", (unsigned long long)n);
        return ATX_ERR_INVALID;
    }
    out->sph.resize(4 * n);
    out->sph_mat.resize(n);
    for (uint64_t i = 0; i < n; ++i) {
        const atx_sphere& s = spheres[i];
        out->sph[4 * i + 0] = s.center[0];
        out->sph[4 * i + 1] = s.center[1];
        out->sph[4 * i + 2] = s.center[2];
        out->sph[4 * i + 3] = s.radius * s.radius;
        int32_t id = s.material;
        if ((uint32_t)id >= m) {
            fprintf(stderr, "Sphere ID out of bounds: %d\n", id);
            id = 0;
        }
        out->sph_mat[i] = id;
    }
    out->mat.resize(12 * m);
    out->mat_rr.resize(4 * m);
    for (uint64_t i = 0; i < m; ++i) {
        const atx_material& a = materials[i];
        float* o = &out->mat[12 * i];
        o[0] = a.albedo[0]; o[1] = a.albedo[1]; o[2] = a.albedo[2]; o[3] = a.roughness;
        o[4] = a.F0[0]; o[5] = a.F0[1]; o[6] = a.F0[2]; o[7] = a.metallic;
        o[8] = a.emission_color[0]; o[9] = a.emission_color[1]; o[10] = a.emission_color[2];
        o[11] = a.emission_intensity;
        const f3 albedo = mk(a.albedo[0], a.albedo[1], a.albedo[2]);
        const float p = gmax(0.1f, gmin(1.0f, length(albedo)));
        const f3 tp = divs(albedo, p);
        float* r = &out->mat_rr[4 * i];
        r[0] = tp.x; r[1] = tp.y; r[2] = tp.z; r[3] = p;
        const float in_unit[] = {a.albedo[0], a.albedo[1], a.albedo[2], a.F0[0], a.F0[1], a.F0[2], a.metallic, a.roughness};
        for (float v : in_unit)
            if (!(v >= 0.0f && v <= 1.0f)) out->unit_materials = false;
        if (a.roughness > 0.0f && a.roughness < 0x1p-10f) out->unit_materials = false;
        if (a.emission_intensity > 0.0f) out->emits = true;
        for (int k = 0; k < 3; ++k)
            if (a.albedo[k] > 0.0f && a.albedo[k] < out->least_albedo) out->least_albedo = a.albedo[k];
    }
    out->light.resize(8 * l);
    for (uint64_t i = 0; i < l; ++i) {
        const atx_light& a = lights[i];
        float* o = &out->light[8 * i];
        o[0] = a.position[0]; o[1] = a.position[1]; o[2] = a.position[2]; o[3] = a.intensity;
        for (int k = 0; k < 3; ++k)
            o[4 + k] = a.color[k] * a.intensity;
        o[7] = 0.0f;
    }
    return ATX_OK;
}

size_t scene_device_bytes(uint64_t n, uint64_t m, uint64_t l)
{
    return 16 * n + 4 * n + 4 * n + 48 * m + 16 * m + 32 * l + bvh_device_bytes(n) + (ScenePack::kArrays + 1) * 16;
}

ScenePack::ScenePack(const HostSceneLayout& L, const HostBvh& T, bool lookups, size_t align)
    : tile_sph(T.tsph), tile_idx(T.tidx)
{
    if (T.n_tiles > 0) {
        for (int32_t id : T.big) {
            tile_sph.insert(tile_sph.end(), &L.sph[4 * (size_t)id], &L.sph[4 * (size_t)id] + 4);
            tile_idx.push_back(id);
        }
        for (int32_t id : tile_idx)
            if (lookups) tile_mat.push_back(L.sph_mat[id]);
    }
    const auto put = [this, align](Array a, const auto& v) {
        off[a] = bytes;
        src[a] = v.data();
        src_bytes[a] = v.size() * 4;
        bytes += (src_bytes[a] + align - 1) / align * align;
    };
    bytes = 0;
    put(kSph, L.sph);
    put(kSphMat, L.sph_mat);
    put(kMat, L.mat);
    put(kLight, L.light);
    put(kTiles, T.tiles);
    put(kTileBoxes, T.tboxes);
    put(kTileSph, tile_sph);
    put(kTileIdx, tile_idx);
    put(kTileMat, tile_mat);
    const std::vector<float> none;
    if (lookups) put(kMatRr, L.mat_rr);
    else put(kMatRr, none);
}

std::vector<unsigned char> ScenePack::block() const
{
    std::vector<unsigned char> b(bytes);
    for (int a = 0; a < kArrays; ++a)
        if (src_bytes[a]) memcpy(b.data() + off[a], src[a], src_bytes[a]);
    return b;
}

BvhDev ScenePack::bvh(const HostBvh& T, const void* base) const
{
    BvhDev b{};
    if (T.n_tiles == 0) return b;
    b.tiles = at<uint4>(base, kTiles);
    b.tboxes = at<float4>(base, kTileBoxes);
    b.tsph = at<float4>(base, kTileSph);
    b.tidx = at<int32_t>(base, kTileIdx);
    b.tmat = tile_mat.empty() ? nullptr : at<int32_t>(base, kTileMat);
    b.n_tiles = T.n_tiles;
    b.n_nodes = (uint32_t)(T.tboxes.size() / 8);
    b.n_big = (uint32_t)T.big.size();
    b.big0 = (uint32_t)T.tidx.size();
    b.cx = T.cx;
    b.cy = T.cy;
    b.cz = T.cz;
    b.ts = T.ts;
    b.t_lin = T.t_lin;
    return b;
}

int upload_scene(const atx_sphere* spheres, uint64_t n, const atx_material* materials, uint64_t m,
                 const atx_light* lights, uint64_t l, DevScene* out)
{
    HostSceneLayout L;
    int rc = build_scene_layout(spheres, n, materials, m, lights, l, &L);
    if (rc != ATX_OK) return rc;
    HostBvh T;
    build_bvh(L.sph.data(), (uint32_t)n, 0, &T);
    const ScenePack pack(L, T);
    // the block's growth frees the former scene: until this one is there, there is none
    out->forget();
    // never an empty block: the kernels' pointers stay valid without spheres
    ATX_HIP(out->block.reserve(pack.bytes + 16));
    if (pack.bytes) ATX_HIP(hipMemcpy(out->block.get(), pack.block().data(), pack.bytes, hipMemcpyHostToDevice));
    const void* base = out->block.get();
    out->sph = pack.at<float4>(base, ScenePack::kSph);
    out->sph_mat = pack.at<int32_t>(base, ScenePack::kSphMat);
    out->mat = pack.at<float4>(base, ScenePack::kMat);
    out->mat_rr = pack.at<float4>(base, ScenePack::kMatRr);
    out->light = pack.at<float4>(base, ScenePack::kLight);
    out->n_sph = (uint32_t)n;
    out->n_mat = (uint32_t)m;
    out->n_light = (uint32_t)l;
    out->least_albedo = L.least_albedo;
    out->unit_materials = L.unit_materials;
    out->emits = L.emits;
    out->bvh = pack.bvh(T, base);
    return ATX_OK;
}

}  // namespace atx

using namespace atx;

extern "C" {

const char* atx_last_error(void) { return g_last_error.c_str(); }

const char* atx_version(void) { return "ataraxia-amd 0.1 (gfx950)"; }

int atx_device_count(int* count)
{
    ATX_CHECK_ARG(count, "count is NULL");
    int c = 0;
    hipError_t e = hipGetDeviceCount(&c);
    if (e != hipSuccess) {
        *count = 0;
        set_error("hipGetDeviceCount: %s", hipGetErrorString(e));
        return ATX_ERR_NODEVICE;
    }
    *count = c;
    return ATX_OK;
}

int atx_device_synchronize(void)
{
    ATX_HIP(hipDeviceSynchronize());
    return ATX_OK;
}

int atx_camera_matrices(const atx_camera* cam, float* inv_proj, float* inv_view)
{
    ATX_CHECK_ARG(cam && inv_proj && inv_view, "NULL argument");
    ATX_CHECK_ARG(cam->width > 0 && cam->height > 0, "Width or height cannot be zero");
    camera_inverse_matrices(cam->position, cam->direction, cam->fov_deg, cam->near_clip, cam->far_clip,
                            cam->width, cam->height, inv_proj, inv_view);
    return ATX_OK;
}

int atx_camera_ray_directions(const atx_camera* cam, float* dirs, uint64_t num_floats)
{
    ATX_CHECK_ARG(cam && dirs, "NULL argument");
    ATX_CHECK_ARG(cam->width > 0 && cam->height > 0, "Width or height cannot be zero");
    ATX_CHECK_ARG(num_floats >= 3ull * cam->width * cam->height, "dirs holds %llu floats, need %llu",
                  (unsigned long long)num_floats, 3ull * cam->width * cam->height);
    float ip[16], iv[16];
    camera_inverse_matrices(cam->position, cam->direction, cam->fov_deg, cam->near_clip, cam->far_clip,
                            cam->width, cam->height, ip, iv);
    for (uint32_t y = 0; y < cam->height; ++y)
        for (uint32_t x = 0; x < cam->width; ++x) {
            const f3 d = camera_ray(ip, iv, x, y, cam->width, cam->height);
            float* o = dirs + 3 * ((size_t)x + (size_t)y * cam->width);
            o[0] = d.x; o[1] = d.y; o[2] = d.z;
        }
    return ATX_OK;
}

int atx_write_ppm(const char* path, const uint32_t* rgba, uint32_t width, uint32_t height, int flip_vertical)
{
    ATX_CHECK_ARG(path && rgba, "NULL argument");
    ATX_CHECK_ARG(width > 0 && height > 0, "Width or height cannot be zero");
    FILE* f = fopen(path, "wb");
    if (!f) {
        set_error("cannot open %s for writing", path);
        return ATX_ERR_IO;
    }
    fprintf(f, "P6\n%u %u\n255\n", width, height);
    std::vector<unsigned char> row((size_t)width * 3);
    bool ok = true;
    for (uint32_t r = 0; r < height && ok; ++r) {
        const uint32_t y = flip_vertical ? height - 1 - r : r;
        const uint32_t* src = rgba + (size_t)y * width;
        for (uint32_t x = 0; x < width; ++x) {
            row[3 * x + 0] = (unsigned char)(src[x] & 0xFF);
            row[3 * x + 1] = (unsigned char)((src[x] >> 8) & 0xFF);
            row[3 * x + 2] = (unsigned char)((src[x] >> 16) & 0xFF);
        }
        ok = fwrite(row.data(), 1, row.size(), f) == row.size();
    }
    if (fclose(f) != 0 || !ok) {
        set_error("write to %s failed", path);
        return ATX_ERR_IO;
    }
    return ATX_OK;
}

}  // extern "C"
