// tile_check.cpp -- host-side check of the tile queries (trace_tiles.h and
// build_tiles in bvh_build.cpp) against the oracle's flat closest-hit loop
// (ora_trace_ray: the reference's Renderer.cu:251-285).
//
// A float restatement of the query forms the ray's half-precision operands as
// the kernel does (truncated splits), reads tiles and boxes as built, sums the
// products in single precision in several orders, one of them with the sum
// pushed towards ruling a sphere out by half of what the kernel's bound
// allows, and tests the spheres that are kept, settling those whose order the
// filter leaves open as the kernel does.  Closest hits (index and t bit
// for bit) and shadow decisions must be the oracle's for the scenes of
// bvh_check.cpp and for trees around the sizes where a tile, a round of eight
// tiles or the groups' boxes end: rays as in bvh_check.cpp, rays that are not
// quite unit vectors and origins up to 1e5 away.  Also checks that tiles hold
// every sphere once, in the row its bit stands for and inside the boxes, and
// that the rows past the last sphere are never kept.
//
// Build: g++ -std=c++17 -O2 -ffp-contract=off tile_check.cpp bvh_build.cpp atx_oracle.c
#include <algorithm>

#define main bvh_check_main
#include "bvh_check.cpp"
#undef main

namespace {

double half_to(uint16_t h)
{
    const int e = (h >> 10) & 31, m = h & 1023;
    const double v = e ? std::ldexp(1024.0 + m, e - 25) : std::ldexp((double)m, -24);
    return h & 0x8000u ? -v : v;
}

// x truncated to half precision (the packed conversion rounds towards zero).
float half_trunc(float x)
{
    const double m = std::fabs((double)x);
    int e = 0;
    std::frexp(m, &e);
    const double ulp = std::ldexp(1.0, std::max(e - 11, -24));
    return (float)std::copysign(std::floor(m / ulp) * ulp, (double)x);
}

struct Halves {
    float hi, lo;
};

Halves split(float x)
{
    uint32_t u;
    std::memcpy(&u, &x, 4);
    u &= 0xffffe000u;
    float hi;
    std::memcpy(&hi, &u, 4);
    return {half_trunc(hi), half_trunc(x - hi)};
}

// Sum of 32 products in single precision, in one of three orders.
float sum32(const double* p, int order)
{
    float s = 0.0f, abs_sum = 0.0f;
    for (int k = 0; k < 32; ++k) {
        const int j = order == 0 ? k : order == 1 ? 31 - k : (k * 5) % 32;
        s = (float)((double)s + p[j]);
        abs_sum += (float)std::fabs(p[j]);
    }
    return order == 2 ? s - 0x1p-19f * abs_sum : s;   // half of 32 * 2^-23 of the terms
}

struct TileQuery {
    uint64_t kept = 0, rays = 0, exact = 0, padding = 0, tiles = 0, odd = 0;
};

double tile_half(const HostBvh& B, uint32_t k, uint32_t j)   // half j of the k-th sphere
{
    const uint32_t* tile = &B.tiles[(size_t)(k / atx::kTileSpheres) * atx::kTileWords];
    const uint32_t w = tile[((j / 8) * 32u + atx::tile_row(k % atx::kTileSpheres)) * 4u + (j % 8) / 2];
    return half_to((uint16_t)(j & 1 ? w >> 16 : w & 0xffffu));
}

// tile_candidate: the filtered test, settled by the exact t where it is open.
bool candidate(const std::vector<float>& sph, int32_t id, V o, V d, float a, Filter& f, TileQuery& q)
{
    Filter g = f;
    g.amb = false;
    bool better = filter_sphere(&sph[4 * id], id, o, d, a, g);
    if (g.amb) {
        ++q.exact;
        const float t = exact_t(&sph[4 * id], o, d, a);   // NaN where disc < 0
        if (f.best < 0) {
            better = t > 0.0f;
        } else {
            const float tb = exact_t(&sph[4 * f.best], o, d, a);
            better = t > 0.0f && (t < tb || (t == tb && id < f.best));
        }
        const float n = t * a, u = std::fmax(std::fabs(n), 0x1p-30f);
        g.lo = std::fma(u, -0x1p-16f, n);
        g.hi = std::fma(u, 0x1p-16f, n);
        g.best = id;
    }
    if (better) {
        f.lo = g.lo;
        f.hi = g.hi;
        f.best = id;
    }
    return better;
}

int32_t trace_tiles(const HostBvh& B, const std::vector<float>& sph, V o, V d, float dist2, int order, float* t,
                    TileQuery& q)
{
    const float a = vdot(d, d);
    const bool shadow = dist2 >= 0.0f;
    bool act = true;
    Filter f;
    for (int32_t id : B.big) candidate(sph, id, o, d, a, f, q);
    const float ox = (o.x - B.cx) * B.ts, oy = (o.y - B.cy) * B.ts, oz = (o.z - B.cz) * B.ts;
    const float n = std::sqrt((ox * ox + oy * oy) + oz * oz);
    const float D = n + 8.0f, D2 = D * D, a1 = std::fabs(a - 1.0f);
    const float t1 = -((ox * d.x + oy * d.y) + oz * d.z);
    float fx = std::fma(d.x, t1, ox), fy = std::fma(d.y, t1, oy), fz = std::fma(d.z, t1, oz);
    const float t2 = -((fx * d.x + fy * d.y) + fz * d.z);
    fx = std::fma(d.x, t2, fx);
    fy = std::fma(d.y, t2, fy);
    fz = std::fma(d.z, t2, fz);
    const float ff = (fx * fx + fy * fy) + fz * fz;
    const float E = std::fma(D2, 0x1p-17f + 2.0f * a1, 0x1.4p-17f * (2.0f * ff + 128.0f));
    const bool odd = !(E < 4096.0f) || !(a1 < 0x1p-10f);
    if (odd) act = false;
    if (ff > 130.0f + 2.0f * E) act = false;
    const float inv_a_up = (1.0f / a) * (1.0f + 0x1p-20f);
    float tlim = std::fmin(f.hi * inv_a_up, shadow ? std::sqrt(dist2) * (1.0f + 0x1p-18f) : INFINITY);
    if (shadow && tlim * tlim < dist2) act = false;
    const float ix = 1.0f / (d.x + 0x1p-64f), iy = 1.0f / (d.y + 0x1p-64f), iz = 1.0f / (d.z + 0x1p-64f);
    const float M = std::fmin((D2 + 64.0f) * B.t_lin, (D + 4.0f) * 0x1.6a0ap-9f) + 0x1p-18f * (n + 16.0f);
    const float jx = std::fabs(ix), jy = std::fabs(iy), jz = std::fabs(iz);
    const float ux = ox * ix, uy = oy * iy, uz = oz * iz;
    const float px = std::fma(-M, jx, -ux), py = std::fma(-M, jy, -uy), pz = std::fma(-M, jz, -uz);
    const float qx = std::fma(M, jx, -ux), qy = std::fma(M, jy, -uy), qz = std::fma(M, jz, -uz);
    auto touches = [&](uint32_t k) {
        const float* b = &B.tboxes[8 * (size_t)k];
        const float ax = std::fma(-b[3], jx, std::fma(b[0], ix, px)), bx = std::fma(b[3], jx, std::fma(b[0], ix, qx));
        const float ay = std::fma(-b[4], jy, std::fma(b[1], iy, py)), by = std::fma(b[4], jy, std::fma(b[1], iy, qy));
        const float az = std::fma(-b[5], jz, std::fma(b[2], iz, pz)), bz = std::fma(b[5], jz, std::fma(b[2], iz, qz));
        return std::fmax(std::fmax(std::fmax(ax, ay), az), 0.0f) <=
               std::fmin(std::fmin(std::fmin(bx, by), bz), tlim * B.ts);
    };
    const Halves r[10] = {split(d.x * d.x), split(d.y * d.y), split(d.z * d.z), split(d.x * d.y), split(d.x * d.z),
                          split(d.y * d.z), split(fx),        split(fy),        split(fz),        split(E - ff)};
    double ray[32];
    for (int j = 0; j < 10; ++j) {
        ray[2 * j] = r[j].hi;
        ray[2 * j + 1] = r[j].lo;
    }
    ray[20] = ray[21] = 1.0;
    for (int j = 0; j < 9; ++j) ray[22 + j] = r[j].hi;
    ray[31] = r[8].lo;
    ++q.rays;
    for (uint32_t tile = 0; act && tile < B.n_tiles; ++tile) {
        if (B.n_tiles > atx::kTileFlat && !touches(B.n_tiles + tile / 8)) continue;
        if (!touches(tile)) continue;
        ++q.tiles;
        for (uint32_t k = tile * 32; act && k < tile * 32 + 32; ++k) {
            double p[32];
            for (uint32_t j = 0; j < 32; ++j) p[j] = tile_half(B, k, j) * ray[j];
            if (std::signbit(sum32(p, order))) continue;
            if (k >= B.tidx.size()) {
                ++q.padding;
                continue;
            }
            ++q.kept;
            if (candidate(sph, B.tidx[k], o, d, a, f, q)) tlim = std::fmin(tlim, f.hi * inv_a_up);
            if (shadow && tlim * tlim < dist2) act = false;
        }
    }
    if (odd) {
        ++q.odd;
        float tm = FLT_MAX;
        int32_t best = -1;
        for (size_t k = 0; k < sph.size() / 4; ++k) {
            const float tt = exact_t(&sph[4 * k], o, d, a);
            if (tt > 0.0f && tt < tm) {   // NaN where disc < 0
                tm = tt;
                best = (int32_t)k;
            }
        }
        *t = tm;
        return best;
    }
    *t = f.best >= 0 ? exact_t(&sph[4 * f.best], o, d, a) : FLT_MAX;
    return f.best;
}

int check_tiles(const HostBvh& B, const char* name)
{
    const uint32_t n = (uint32_t)B.lidx.size(), groups = (B.n_tiles + 7) / 8;
    if (B.n_tiles != (n + 31) / 32 || B.tiles.size() != (size_t)B.n_tiles * atx::kTileWords ||
        B.tidx.size() != n || B.tboxes.size() != 8 * (size_t)(B.n_tiles + groups))
        return fail("tile sizes", name);
    std::vector<int32_t> x = B.tidx, y = B.lidx;
    std::sort(x.begin(), x.end());
    std::sort(y.begin(), y.end());
    if (x != y) return fail("tiles do not hold the tree's spheres", name);
    for (uint32_t k = 0; k < n; ++k) {
        const float* s = &B.tsph[4 * k];
        const double r = std::sqrt((double)s[3]) * B.ts, centre[3] = {B.cx, B.cy, B.cz};
        for (int a = 0; a < 3; ++a) {
            const double c = (s[a] - centre[a]) * B.ts;
            if (std::fabs(tile_half(B, k, 12 + 2 * a) + tile_half(B, k, 28 + a) - 2.0 * c) > 0x1p-20)
                return fail("sphere not in its row", name);
            for (uint32_t b : {k / 32, B.n_tiles + k / 256}) {
                const float* q = &B.tboxes[8 * (size_t)b];
                if (c - r < (double)q[a] - q[3 + a] || c + r > (double)q[a] + q[3 + a])
                    return fail("sphere outside its box", name);
            }
        }
    }
    return 0;
}

int check_scene(const Scene& sc, int rays)
{
    const uint32_t n = (uint32_t)sc.s.size();
    std::vector<float> sph(4 * (size_t)n);
    for (uint32_t i = 0; i < n; ++i) {
        for (int k = 0; k < 3; ++k) sph[4 * i + k] = sc.s[i].center[k];
        sph[4 * i + 3] = sc.s[i].radius * sc.s[i].radius;
    }
    HostBvh B;
    atx::build_bvh(sph.data(), n, atx::kBvhLayouts, &B);
    if (B.n_tiles == 0) return fail("no tiles built", sc.name);
    if (check_tiles(B, sc.name)) return 1;
    Rng g{99 + n};
    TileQuery q;
    const float ext = 8.0f / B.ts;
    for (int r = 0; r < rays; ++r) {
        const uint32_t k = (uint32_t)(g.next() % n), m = (uint32_t)(g.next() % n);
        const float *c = &sph[4 * k], *e = &sph[4 * m];
        const float rad = std::sqrt(c[3]);
        V o;
        switch (r % 5) {
        case 0: {   // leaving a surface
            const V nrm = random_dir(g);
            o = vadd(vadd(V{c[0], c[1], c[2]}, vscale(nrm, rad)), vscale(nrm, 1e-4f));
            break;
        }
        case 1: o = V{c[0] + 0.3f * rad, c[1] - 0.2f * rad, c[2]}; break;   // inside
        case 2: o = vadd(V{B.cx, B.cy, B.cz}, vscale(random_dir(g), ext * g.uni(0, 1.5f))); break;
        case 3: o = vadd(V{B.cx, B.cy, B.cz}, vscale(random_dir(g), ext * g.uni(1.5f, 6.0f))); break;
        default: o = vadd(V{B.cx, B.cy, B.cz}, vscale(random_dir(g), ext * std::exp(g.uni(1.0f, 11.0f)))); break;
        }
        V d;
        switch ((r / 5) % 4) {
        case 0: d = random_dir(g); break;
        case 1: {   // a silhouette
            const V to = vsub(V{e[0], e[1], e[2]}, o);
            V p{to.y, -to.x, 0.0f};
            if (vdot(p, p) < 1e-12f) p = {0.0f, to.z, -to.y};
            d = vsub(vadd(V{e[0], e[1], e[2]}, vscale(vnorm(p), std::sqrt(e[3]) * (1.0f + g.uni(-4e-7f, 4e-7f)))), o);
            d = vdot(d, d) > 0.0f ? vnorm(d) : random_dir(g);
            break;
        }
        case 2: {   // an axis, with signed zeros
            d = V{(r & 8) ? 0.0f : -0.0f, (r & 16) ? 0.0f : -0.0f, (r & 32) ? 0.0f : -0.0f};
            const float v = g.next() & 1 ? 1.0f : -1.0f;
            (g.next() % 3 == 0 ? d.x : g.next() % 2 ? d.y : d.z) = v;
            break;
        }
        default: {
            d = vsub(V{e[0], e[1], e[2]}, o);
            d = vdot(d, d) > 0.0f ? vnorm(d) : random_dir(g);
        }
        }
        if (r % 7 == 3) d = vscale(d, 1.0f + g.uni(-1e-3f, 1e-3f));   // some past the filter's limit
        const float o3[3] = {o.x, o.y, o.z}, d3[3] = {d.x, d.y, d.z};
        float tr = 0.0f, tt = 0.0f;
        const int32_t ir = ora_trace_ray(o3, d3, sc.s.data(), n, &tr);
        const int32_t it = trace_tiles(B, sph, o, d, -1.0f, r % 3, &tt, q);
        if (ir != it || std::memcmp(&tr, &tt, 4) != 0) {
            std::fprintf(stderr, "FAIL [%s] ray %d: o=(%a,%a,%a) d=(%a,%a,%a) oracle=%d t=%a tiles=%d t=%a\n", sc.name,
                         r, o.x, o.y, o.z, d.x, d.y, d.z, ir, tr, it, tt);
            return 1;
        }
        const float along = g.uni(0.0f, 2.0f) * (ir >= 0 ? tr : 10.0f), dist2 = along * along;
        if (!(dist2 > 0.0f)) continue;
        const int32_t is = trace_tiles(B, sph, o, d, dist2, r % 3, &tt, q);
        if ((is >= 0 && tt > 0.0f && tt * tt < dist2) != (ir >= 0 && tr > 0.0f && tr * tr < dist2)) {
            std::fprintf(stderr, "FAIL [%s] shadow ray %d\n", sc.name, r);
            return 1;
        }
    }
    if (q.padding) return fail("a row past the last sphere was kept", sc.name);
    std::printf("%-20s spheres=%4u tiles=%2u rays=%" PRIu64 " tiles/ray=%.2f kept/ray=%.2f settled=%" PRIu64 " flat=%" PRIu64 "\n", sc.name,
                n, B.n_tiles, q.rays, (double)q.tiles / q.rays, (double)q.kept / q.rays, q.exact, q.odd);
    return 0;
}

}  // namespace

int main(int argc, char** argv)
{
    const int rays = argc > 1 ? std::atoi(argv[1]) : 20000;
    std::vector<Scene> scenes = make_scenes();
    // trees around a tile's 32 spheres, a round's 256, and the 16 tiles past
    // which groups have boxes; the largest spreads over three groups
    for (uint32_t n : {16u, 31u, 32u, 33u, 65u, 255u, 257u, 512u, 513u, 700u}) {
        Rng g{n};
        Scene sc{"tree_size", {}};
        const float e = 20.0f * std::sqrt((float)n / 256.0f);
        for (uint32_t i = 0; i < n; ++i) push(sc, g.uni(-e, e), g.uni(0, 6), g.uni(-e, e), g.uni(0.3f, 1.5f));
        push(sc, 0, -1000, 0, 1000);
        scenes.push_back(sc);
    }
    for (const Scene& sc : scenes)
        if (check_scene(sc, rays)) return 1;
    return 0;
}
