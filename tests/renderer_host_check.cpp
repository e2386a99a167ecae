// Host checks of the renderer's C ABI (ataraxia_amd/csrc/renderer.cpp) over
// tests/fake_hip.h.  Built by tests/test_renderer_host.py; the argument names the check.
#include "fake_hip.h"

#include <string>
#include <thread>
#include <vector>

static int bad = 0;
#define CHECK(c)                                                                     \
    do {                                                                             \
        if (!(c)) {                                                                  \
            std::fprintf(stderr, "line %d: %s (%s)\n", __LINE__, #c, atx_last_error()); \
            ++bad;                                                                   \
        }                                                                            \
    } while (0)

static int set_scene(atx_renderer* r, uint64_t spheres, uint64_t materials)
{
    std::vector<atx_sphere> s(spheres + 1);
    std::vector<atx_material> m(materials + 1);
    for (uint64_t i = 0; i < spheres; ++i) {
        s[i] = atx_sphere{};
        s[i].center[0] = (float)i;
        s[i].radius = 0.4f;
    }
    return atx_renderer_set_scene(r, s.data(), spheres, m.data(), materials, nullptr, 0);
}

// A scene that cannot be uploaded: one refused for its arguments leaves the
// former scene in place; one whose device memory cannot be had leaves none, and no
// kernel is given the former one's memory, which is freed.
static void upload(atx_renderer* r, const atx_camera& cam)
{
    CHECK(atx_renderer_render(r, &cam) == ATX_ERR_STATE);
    CHECK(set_scene(r, 20, 1) == ATX_OK);
    CHECK(atx_renderer_render(r, &cam) == ATX_OK);
    CHECK(set_scene(r, 4, 0) == ATX_ERR_INVALID);
    CHECK(atx_renderer_render(r, &cam) == ATX_OK);
    fake::fail_mallocs = 1;
    CHECK(set_scene(r, 4000, 1) == ATX_ERR_NOMEM);
    const int before = fake::kernel_launches;
    CHECK(atx_renderer_render(r, &cam) == ATX_ERR_STATE);
    CHECK(atx_renderer_reserve(r, 4) == ATX_OK);
    CHECK(fake::kernel_launches == before);
    CHECK(set_scene(r, 4000, 1) == ATX_OK);
    CHECK(atx_renderer_render(r, &cam) == ATX_OK);
}

// Results read by a thread whose current device is another one than the
// renderer's: the first results and later ones.
static void devices(atx_renderer* r, const atx_camera& cam)
{
    CHECK(set_scene(r, 3, 1) == ATX_OK);
    CHECK(atx_renderer_render(r, &cam) == ATX_OK);
    std::vector<uint32_t> image(16 * 8);
    std::vector<float> sums(4 * 16 * 8);
    std::thread([&] {
        (void)hipSetDevice(1);
        CHECK(atx_renderer_get_image(r, image.data(), image.size()) == ATX_OK);
        CHECK(atx_renderer_get_accumulation(r, sums.data(), sums.size()) == ATX_OK);
        int now = 0;
        CHECK(hipGetDevice(&now) == hipSuccess && now == 1);
    }).join();
    CHECK(atx_renderer_get_image(r, image.data(), image.size()) == ATX_OK);
}

int main(int argc, char** argv)
{
    const std::string name = argc > 1 ? argv[1] : "";
    atx_renderer* r = nullptr;
    CHECK(atx_renderer_create(&r) == ATX_OK);
    CHECK(atx_renderer_on_resize(r, 16, 8) == ATX_OK);
    atx_camera cam{};
    cam.direction[2] = -1.0f;
    cam.fov_deg = 45.0f;
    cam.near_clip = 0.1f;
    cam.far_clip = 100.0f;
    cam.width = 16;
    cam.height = 8;
    if (name == "upload") upload(r, cam);
    else if (name == "devices") devices(r, cam);
    else ++bad;
    CHECK(atx_renderer_destroy(r) == ATX_OK);
    std::printf(bad ? "%d checks failed\n" : "all checks passed\n", bad);
    return bad != 0;
}
