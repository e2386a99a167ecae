// tests/tile_check.cpp, its main included, over the tiles that the library builds:
// without the tree whose leaf order the check's own builds start from; and before
// that a scene of more spheres than a tree can hold.  Built by
// tests/test_tiles_production_host.py.
#include "../ataraxia_amd/csrc/bvh_build.h"

namespace atx {
constexpr uint32_t kNoTree = 0;
}
#define kBvhLayouts kNoTree
#include "tile_check.cpp"

static const bool checked = [] {
    Rng g{17000};
    Scene sc{"past a tree's limit", {}};
    for (int i = 0; i < 17000; ++i) push(sc, g.uni(-160, 160), g.uni(0, 6), g.uni(-160, 160), g.uni(0.3f, 1.5f));
    push(sc, 0, -1000, 0, 1000);
    if (check_scene(sc, 500)) std::exit(1);
    return true;
}();
