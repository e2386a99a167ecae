// Host-side check of the in-place launches' layout (layout_in_place in
// ataraxia_amd/csrc/wavefront_host.h).  Built host-only (hipcc
// --offload-host-only) by tests/test_in_place_host.py.
#include <cstdio>

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
    std::printf(bad ? "%d checks failed\n" : "all checks passed\n", bad);
    return bad != 0;
}
