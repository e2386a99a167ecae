// Host-side check of the in-place launches' layout (layout_in_place in
// ataraxia_amd/csrc/wavefront_host.h).  Built host-only (hipcc
// --offload-host-only) by tests/test_in_place_host.py.
#include <cstdio>
#include <vector>

#include "wavefront_host.h"

using namespace atx;

int main()
{
    int bad = 0;
    // any number of frames: 8 * frames, which is 0 in 32 bits for a multiple of 2^29,
    // divides nothing in place
    for (uint32_t frames : {1u, 4097u, 1u << 29, 3u << 29, 0xffffffffu}) {
        WfScene s{};
        s.width = 65;
        s.height = 33;
        s.frames = frames;
        WfPass p{};
        bad += !layout_in_place(s, &p) || s.div_group.d != 0 || s.div_group.m != 0 ||
               p.total_chunks != 9 * 5 || p.n_scenes != 1 || s.frames != frames;
    }
    // every pixel is one job, whatever the image's shape
    const uint32_t sizes[][2] = {{1, 1}, {1, 70}, {70, 1}, {7, 9}, {9, 7}, {8, 8}, {9, 17}, {64, 8}, {133, 61}};
    for (const auto& z : sizes) {
        std::vector<int> seen(z[0] * z[1], 0);
        const uint64_t jobs = in_place_jobs(z[0], z[1]);
        bad += jobs % kInPlaceChunk != 0;
        for (uint32_t j = 0; j < jobs; ++j) {
            const uint32_t px = in_place_pixel(j, z[0], z[1]);
            if (px != ~0u) seen.at(px)++;
        }
        for (int n : seen) bad += n != 1;
    }
    // long thin images are accepted as long as their pixels fit 32 bits: tiles of
    // the first two hold 8 and 1.8 times as many jobs as pixels
    const struct { uint32_t w, h; bool fits; } limit[] = {
        {1, 600000000, true}, {9, 400000000, true}, {600000000, 7, true}, {65535, 65536, true}, {65536, 65536, false},
        {0xffffff00u, 1, true}, {3, 0x60000000u, false}};
    for (const auto& l : limit) {
        WfScene s{};
        s.width = l.w;
        s.height = l.h;
        s.frames = 1;
        WfPass p{};
        bad += layout_in_place(s, &p) != l.fits;
        const uint32_t last = l.w * l.h - 1u;
        if (l.fits && in_place_rows(l.w, l.h))
            bad += in_place_pixel(last, l.w, l.h) != last || (uint64_t)p.total_chunks * 64u <= last;
    }
    std::printf(bad ? "%d checks failed\n" : "all checks passed\n", bad);
    return bad != 0;
}
