// bvh_build.cpp -- host construction of tiles (device layout in bvh.h) and, for
// the host checks, of a sphere BVH.
//
// Tree: binary, surface-area heuristic over sphere boxes, at most kBvhLeafMax
// spheres per leaf.  All geometry is evaluated in double precision; every box
// is rounded outwards to float and then to 16-bit cells of the root box (one
// extra cell on each side), so a node box contains each of its spheres
// (centre c, radius sqrt(r*r)) exactly.  Spheres whose radius exceeds
// the half-diagonal of the region of all other centres (a ground sphere of
// radius 1000 under a cluster of unit spheres) and spheres with non-finite or
// negative data are kept out of the tree: they would make every box, and
// the per-ray inflation that scales with the region, as large as the scene.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "bvh_build.h"

namespace atx {
namespace {

struct Prim {
    double lo[3], hi[3], c[3];
    int32_t idx;
};

struct BNode {
    float lo[3], hi[3];
    int32_t left = -1, right = -1;
    int32_t axis = 0;
    uint32_t first = 0, count = 0;
};

float round_down(double x)
{
    float f = (float)x;
    if ((double)f > x) f = std::nextafter(f, -INFINITY);
    return f;
}

float round_up(double x)
{
    float f = (float)x;
    if ((double)f < x) f = std::nextafter(f, INFINITY);
    return f;
}

double half_area(const double lo[3], const double hi[3])
{
    const double dx = std::max(0.0, hi[0] - lo[0]), dy = std::max(0.0, hi[1] - lo[1]),
                 dz = std::max(0.0, hi[2] - lo[2]);
    return dx * dy + dy * dz + dz * dx;
}

struct Builder {
    std::vector<Prim>& P;
    std::vector<BNode> nodes;
    std::vector<Prim> leaf_order;
    static constexpr double kCostBox = 0.5;   // box test relative to one sphere test

    explicit Builder(std::vector<Prim>& p) : P(p) {}

    void bounds(int b, int e, double lo[3], double hi[3]) const
    {
        for (int k = 0; k < 3; ++k) {
            lo[k] = INFINITY;
            hi[k] = -INFINITY;
        }
        for (int i = b; i < e; ++i)
            for (int k = 0; k < 3; ++k) {
                lo[k] = std::min(lo[k], P[i].lo[k]);
                hi[k] = std::max(hi[k], P[i].hi[k]);
            }
    }

    void sort_axis(int b, int e, int axis)
    {
        std::sort(P.begin() + b, P.begin() + e, [axis](const Prim& x, const Prim& y) {
            return x.c[axis] < y.c[axis] || (x.c[axis] == y.c[axis] && x.idx < y.idx);
        });
    }

    int build(int b, int e)
    {
        const int id = (int)nodes.size();
        nodes.emplace_back();
        double lo[3], hi[3];
        bounds(b, e, lo, hi);
        for (int k = 0; k < 3; ++k) {
            nodes[id].lo[k] = round_down(lo[k]);
            nodes[id].hi[k] = round_up(hi[k]);
        }
        const int n = e - b;
        const double parent = half_area(lo, hi);
        double best_cost = INFINITY;
        int best_axis = -1, best_split = -1;
        std::vector<double> left_area((size_t)n + 1);
        for (int axis = 0; axis < 3 && n > 1; ++axis) {
            sort_axis(b, e, axis);
            double l[3] = {INFINITY, INFINITY, INFINITY}, h[3] = {-INFINITY, -INFINITY, -INFINITY};
            for (int i = 1; i < n; ++i) {
                for (int k = 0; k < 3; ++k) {
                    l[k] = std::min(l[k], P[b + i - 1].lo[k]);
                    h[k] = std::max(h[k], P[b + i - 1].hi[k]);
                }
                left_area[i] = half_area(l, h);
            }
            double rl[3] = {INFINITY, INFINITY, INFINITY}, rh[3] = {-INFINITY, -INFINITY, -INFINITY};
            for (int i = n - 1; i >= 1; --i) {
                for (int k = 0; k < 3; ++k) {
                    rl[k] = std::min(rl[k], P[b + i].lo[k]);
                    rh[k] = std::max(rh[k], P[b + i].hi[k]);
                }
                const double cost = left_area[i] * i + half_area(rl, rh) * (n - i);
                if (cost < best_cost) {
                    best_cost = cost;
                    best_axis = axis;
                    best_split = i;
                }
            }
        }
        const double split_cost =
            parent > 0.0 ? kCostBox + best_cost / parent : kCostBox + (double)n;
        const bool leaf = n == 1 || (n <= (int)kBvhLeafMax && (double)n <= split_cost);
        if (leaf || best_axis < 0) {
            nodes[id].first = (uint32_t)leaf_order.size();
            nodes[id].count = (uint32_t)n;
            for (int i = b; i < e; ++i)
                leaf_order.push_back(P[i]);
            return id;
        }
        sort_axis(b, e, best_axis);
        nodes[id].axis = best_axis;
        const int left = build(b, b + best_split);
        const int right = build(b + best_split, e);
        nodes[id].left = left;
        nodes[id].right = right;
        return id;
    }
};

struct Grid {
    double base[3], scale[3];
};

uint32_t cell_down(double x, const Grid& g, int a)
{
    const double c = std::floor((x - g.base[a]) / g.scale[a]) - 1.0;
    return (uint32_t)std::min(std::max(c, 0.0), (double)kBvhGrid);
}

uint32_t cell_up(double x, const Grid& g, int a)
{
    const double c = std::ceil((x - g.base[a]) / g.scale[a]) + 1.0;
    return (uint32_t)std::min(std::max(c, 0.0), (double)kBvhGrid);
}

void emit(const std::vector<BNode>& T, int id, uint32_t oct, const Grid& g, std::vector<uint32_t>& out,
          uint32_t& cur)
{
    const uint32_t me = cur++;
    uint32_t* d = out.data() + (size_t)me * 4;
    const BNode& nd = T[id];
    uint32_t skip, leaf;
    if (nd.left < 0) {
        skip = me + 1;
        leaf = ((nd.first + 1u) << 2) | (nd.count - 1u);
    } else {
        const bool neg = (oct >> nd.axis) & 1u;
        emit(T, neg ? nd.right : nd.left, oct, g, out, cur);
        emit(T, neg ? nd.left : nd.right, oct, g, out, cur);
        skip = cur;
        leaf = 0;
    }
    const uint32_t lx = cell_down(nd.lo[0], g, 0), ly = cell_down(nd.lo[1], g, 1), lz = cell_down(nd.lo[2], g, 2);
    const uint32_t hx = cell_up(nd.hi[0], g, 0), hy = cell_up(nd.hi[1], g, 1), hz = cell_up(nd.hi[2], g, 2);
    d[0] = lx | (ly << 16);
    d[1] = lz | (hx << 16);
    d[2] = hy | (hz << 16);
    d[3] = skip | (leaf << 16);
}

bool finite_sphere(const float* s)
{
    for (int k = 0; k < 4; ++k)
        if (!std::isfinite(s[k])) return false;
    return s[3] >= 0.0f && std::fabs(s[0]) < 1e15f && std::fabs(s[1]) < 1e15f && std::fabs(s[2]) < 1e15f &&
           s[3] < 1e30f;
}

// Nearest half-precision number (ties to even); |x| < 65504.
uint16_t half_bits(double x)
{
    const uint16_t sign = std::signbit(x) ? 0x8000u : 0u;
    const double m = std::fabs(x);
    if (m < 0x1p-14) return (uint16_t)(sign | (uint16_t)std::nearbyint(m * 0x1p24));   // subnormal: multiples of 2^-24
    int e = 0;
    const double f = std::frexp(m, &e);                       // m = f * 2^e, f in [0.5, 1)
    const long q = (long)std::nearbyint(f * 2048.0);          // 11 significant bits
    return (uint16_t)(sign | (uint16_t)(((e + 13) << 10) + q));   // a carry out of q moves the exponent up
}

double half_value(uint16_t h)
{
    const int e = (h >> 10) & 31, m = h & 1023;
    const double v = e ? std::ldexp(1024.0 + m, e - 25) : std::ldexp((double)m, -24);
    return h & 0x8000u ? -v : v;
}

// x as two halves: hi in the low 16 bits, the rest's nearest half above it.
void half_split(double x, uint16_t& hi, uint16_t& lo)
{
    hi = half_bits(x);
    lo = half_bits(x - half_value(hi));
}

// Orders spheres idx[b, e) so that every kTileSpheres of them lie close
// together, and every eight such tiles too: halves along the longest side of
// the centres' box, cut at a multiple of a tile (of eight tiles where there
// are more than eight).
void tile_order(const std::vector<float>& s, std::vector<uint32_t>& idx, size_t b, size_t e)
{
    const size_t tiles = (e - b + kTileSpheres - 1) / kTileSpheres;
    if (tiles <= 1) return;
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (size_t i = b; i < e; ++i)
        for (int a = 0; a < 3; ++a) {
            lo[a] = std::min(lo[a], s[4 * idx[i] + a]);
            hi[a] = std::max(hi[a], s[4 * idx[i] + a]);
        }
    int axis = 0;
    for (int a = 1; a < 3; ++a)
        if (hi[a] - lo[a] > hi[axis] - lo[axis]) axis = a;
    const size_t unit = tiles > 8 ? 8 : 1;
    const size_t left = ((tiles + 1) / 2 + unit - 1) / unit * unit;
    const size_t m = std::min(e, b + left * kTileSpheres);
    std::nth_element(idx.begin() + b, idx.begin() + m, idx.begin() + e, [&](uint32_t x, uint32_t y) {
        return s[4 * x + axis] < s[4 * y + axis] || (s[4 * x + axis] == s[4 * y + axis] && x < y);
    });
    tile_order(s, idx, b, m);
    tile_order(s, idx, m, e);
}

// Tiles of the tree's spheres (layout and error bound in trace_tiles.h).  Per
// sphere 32 halves, of its centre c in tile units and w = |c|^2 - radius^2
// (v = hi part, v' = lo part):
//   twice each  xx yy zz 2xy 2xz 2yz 2x 2y 2z,  1 1 -w -w',
//   xx' yy' zz' 2xy' 2xz' 2yz' 2x' 2y' 2z' 0
// Lane l of a tile's k-th product (k = 0, 1) holds halves 16 k + 8 (l / 32) .. + 7
// of the sphere in row l % 32.  Rows past the last sphere hold a sphere no ray
// meets (-w far below zero, centre 0).
void build_tiles(HostBvh* B)
{
    const uint32_t n = (uint32_t)B->lidx.size();
    const double reach = ((double)B->rb + (double)B->r_max) * (1.0 + 0x1p-20);
    int e = 0;
    std::frexp(reach, &e);                                     // reach <= 2^e
    const double ts = std::ldexp(1.0, 3 - e);                  // reach * ts <= 8
    B->ts = (float)ts;
    B->t_lin = round_up(std::min(0x1p-18 / std::max((double)B->r_min * ts, 1e-30), 1e6));
    B->n_tiles = (n + kTileSpheres - 1) / kTileSpheres;
    std::vector<uint32_t> order(n);
    for (uint32_t k = 0; k < n; ++k) order[k] = k;
    tile_order(B->lsph, order, 0, n);
    B->tiles.assign((size_t)B->n_tiles * kTileWords, 0u);
    const float centre[3] = {B->cx, B->cy, B->cz};
    const uint32_t groups = (B->n_tiles + 7u) / 8u;
    std::vector<double> lo(3 * (B->n_tiles + groups), INFINITY), hi(3 * (B->n_tiles + groups), -INFINITY);
    for (uint32_t k = 0; k < B->n_tiles * kTileSpheres; ++k) {
        const uint32_t t = k / kTileSpheres, g = B->n_tiles + t / 8u;
        uint16_t v[32] = {};
        v[18] = v[19] = half_bits(1.0);
        if (k < n) {
            const float* s = &B->lsph[4 * (size_t)order[k]];
            B->tsph.insert(B->tsph.end(), s, s + 4);
            B->tidx.push_back(B->lidx[order[k]]);
            const double r = std::sqrt((double)s[3]) * ts * (1.0 + 0x1p-40);
            double c[3], w = -(double)s[3] * ts * ts;
            for (int a = 0; a < 3; ++a) {
                c[a] = ((double)s[a] - (double)centre[a]) * ts;
                w += c[a] * c[a];
                for (uint32_t b : {t, g}) {
                    lo[3 * b + a] = std::min(lo[3 * b + a], c[a] - r);
                    hi[3 * b + a] = std::max(hi[3 * b + a], c[a] + r);
                }
            }
            const double p[9] = {c[0] * c[0],       c[1] * c[1],       c[2] * c[2],
                                 2.0 * c[0] * c[1], 2.0 * c[0] * c[2], 2.0 * c[1] * c[2],
                                 2.0 * c[0],        2.0 * c[1],        2.0 * c[2]};
            for (int j = 0; j < 9; ++j) {
                half_split(p[j], v[2 * j], v[22 + j]);
                v[2 * j + 1] = v[2 * j];
            }
            half_split(-w, v[20], v[21]);
        } else {
            v[20] = half_bits(-60000.0);
        }
        uint32_t* tile = &B->tiles[(size_t)t * kTileWords];
        const uint32_t row = tile_row(k % kTileSpheres);
        for (uint32_t j = 0; j < 32; j += 2)
            tile[((j / 8) * 32u + row) * 4u + (j % 8) / 2] = v[j] | ((uint32_t)v[j + 1] << 16);
    }
    for (uint32_t b = 0; b < B->n_tiles + groups; ++b) {
        float c[3], half[3];
        for (int a = 0; a < 3; ++a) {
            c[a] = (float)(0.5 * (lo[3 * b + a] + hi[3 * b + a]));
            half[a] = round_up(std::max(hi[3 * b + a] - (double)c[a], (double)c[a] - lo[3 * b + a]));
        }
        B->tboxes.insert(B->tboxes.end(), {c[0], c[1], c[2], half[0], half[1], half[2], 0.0f, 0.0f});
    }
}

// The tree's nodes in `layouts` orders; leaves P in leaf order.
void build_nodes(std::vector<Prim>& P, uint32_t layouts, HostBvh* out)
{
    Builder B(P);
    B.build(0, (int)P.size());
    const uint32_t nn = (uint32_t)B.nodes.size();

    // Cell grid over the root box: world = base + cell * scale, with scale a
    // float so that the device's grid coordinates mean exactly the same boxes.
    // Boxes round outwards and get one extra cell on each side.
    Grid g;
    for (int a = 0; a < 3; ++a) {
        const double lo_a = B.nodes[0].lo[a], hi_a = B.nodes[0].hi[a];
        const double span = hi_a - lo_a;
        float sc = round_up(span > 0.0 ? span / (double)(kBvhGrid - 4) : 1.0);
        if (!(sc > 0.0f)) sc = 1.0f;
        g.base[a] = lo_a;
        g.scale[a] = sc;
        out->base[a] = B.nodes[0].lo[a];
        out->scale[a] = sc;
        out->inv_scale[a] = (float)(1.0 / (double)sc);
    }
    out->ext = round_up((double)kBvhGrid * std::max(std::max(g.scale[0], g.scale[1]), g.scale[2]) * (1.0 + 0x1p-30));
    out->n_nodes = nn;
    out->layouts = layouts;
    out->nodes.assign((size_t)layouts * nn * 4, 0u);
    for (uint32_t oct = 0; oct < layouts; ++oct) {
        std::vector<uint32_t> lay((size_t)nn * 4);
        uint32_t cur = 0;
        emit(B.nodes, 0, oct, g, lay, cur);
        std::copy(lay.begin(), lay.end(), out->nodes.begin() + (size_t)oct * nn * 4);
    }
    std::vector<Prim> ordered = std::move(B.leaf_order);
    P.swap(ordered);
}

}  // namespace

void build_bvh(const float* sph4, uint32_t n, uint32_t layouts, HostBvh* out)
{
    *out = HostBvh();
    layouts = layouts >= kBvhLayouts ? kBvhLayouts : layouts;
    if (n < kBvhMinSpheres) return;

    std::vector<int32_t> big;
    std::vector<char> is_big(n, 0);
    std::vector<uint32_t> valid;
    for (uint32_t i = 0; i < n; ++i) {
        if (finite_sphere(sph4 + 4 * i)) {
            valid.push_back(i);
        } else {
            big.push_back((int32_t)i);
            is_big[i] = 1;
        }
    }
    // Largest spheres first: a sphere goes out of the tree while its radius
    // exceeds the half-diagonal of the box around all remaining centres.
    std::vector<uint32_t> by_r = valid;
    std::sort(by_r.begin(), by_r.end(), [&](uint32_t a, uint32_t b) {
        return sph4[4 * a + 3] > sph4[4 * b + 3] || (sph4[4 * a + 3] == sph4[4 * b + 3] && a < b);
    });
    for (size_t k = 0; k < by_r.size() && big.size() < kBvhMaxBig + 1; ++k) {
        const uint32_t cand = by_r[k];
        double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
        for (uint32_t i : valid) {
            if (is_big[i] || i == cand) continue;
            for (int a = 0; a < 3; ++a) {
                lo[a] = std::min(lo[a], (double)sph4[4 * i + a]);
                hi[a] = std::max(hi[a], (double)sph4[4 * i + a]);
            }
        }
        if (!(lo[0] <= hi[0])) break;
        const double dx = hi[0] - lo[0], dy = hi[1] - lo[1], dz = hi[2] - lo[2];
        const double half_diag = 0.5 * std::sqrt(dx * dx + dy * dy + dz * dz);
        if (std::sqrt((double)sph4[4 * cand + 3]) > half_diag) {
            big.push_back((int32_t)cand);
            is_big[cand] = 1;
        } else {
            break;
        }
    }
    std::vector<Prim> P;
    for (uint32_t i : valid) {
        if (is_big[i]) continue;
        Prim p;
        const double r = std::sqrt((double)sph4[4 * i + 3]) * (1.0 + 0x1p-40);
        for (int a = 0; a < 3; ++a) {
            p.c[a] = sph4[4 * i + a];
            p.lo[a] = p.c[a] - r;
            p.hi[a] = p.c[a] + r;
        }
        p.idx = (int32_t)i;
        P.push_back(p);
    }
    if (big.size() > kBvhMaxBig || P.size() < kBvhMinSpheres || P.size() > (layouts ? kBvhMaxTree : kTileMaxSpheres))
        return;
    std::sort(big.begin(), big.end());

    // Region of the tree: centre of the centres' box, bounds of distance and radius.
    double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    double r2_min = INFINITY, r2_max = 0.0;
    for (const Prim& p : P) {
        for (int a = 0; a < 3; ++a) {
            lo[a] = std::min(lo[a], p.c[a]);
            hi[a] = std::max(hi[a], p.c[a]);
        }
        const double r2 = sph4[4 * p.idx + 3];
        r2_min = std::min(r2_min, r2);
        r2_max = std::max(r2_max, r2);
    }
    const double C[3] = {0.5 * (lo[0] + hi[0]), 0.5 * (lo[1] + hi[1]), 0.5 * (lo[2] + hi[2])};
    const float Cf[3] = {(float)C[0], (float)C[1], (float)C[2]};
    double rb = 0.0;
    for (const Prim& p : P) {
        const double dx = p.c[0] - Cf[0], dy = p.c[1] - Cf[1], dz = p.c[2] - Cf[2];
        rb = std::max(rb, std::sqrt(dx * dx + dy * dy + dz * dz));
    }

    if (layouts) build_nodes(P, layouts, out);
    for (const Prim& p : P) {
        for (int a = 0; a < 4; ++a)
            out->lsph.push_back(sph4[4 * p.idx + a]);
        out->lidx.push_back(p.idx);
    }
    out->big = big;
    out->cx = Cf[0];
    out->cy = Cf[1];
    out->cz = Cf[2];
    out->rb = round_up(rb * (1.0 + 0x1p-30));
    out->r_min = round_down(std::sqrt(r2_min) * (1.0 - 0x1p-30));
    out->r_max = round_up(std::sqrt(r2_max) * (1.0 + 0x1p-30));
    build_tiles(out);
}

size_t bvh_device_bytes(uint64_t n)
{
    const uint64_t tiles = (n + kTileSpheres - 1) / kTileSpheres, boxes = tiles + (tiles + 7) / 8;
    if (n < kBvhMinSpheres || n > kTileMaxSpheres + kBvhMaxBig) return 0;   // no tiles
    return (size_t)(tiles * kTileWords * 4 + boxes * 32 + 32) + (size_t)(16 * n + 16) + (size_t)(4 * n + 16);
}

}  // namespace atx
