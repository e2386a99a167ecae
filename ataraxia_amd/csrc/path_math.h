// path_math.h -- scalar arithmetic of the per-pixel path, shared by the HIP
// kernels and by the host-side camera code of libatx.
//
// Every function rounds exactly as the reference's GLM expressions do under
// IEEE-754 binary32 with no contraction (this file must be compiled with
// -ffp-contract=off and without fast-math; fused multiply-adds appear only
// where written as fmaf, in the sin/cos kernels).  GLM semantics restated
// (GLM is an unvendored dependency of the reference, see .gitmodules:1-4):
//   dot(a,b)     = (a.x*b.x + a.y*b.y) + a.z*b.z
//   normalize(v) = v * (1 / sqrt(dot(v,v)))
//   max(a,b)     = a < b ? b : a,  min(a,b) = b < a ? b : a
//   mix(x,y,a)   = x*(1-a) + y*a
//   mat4*vec4    = (m0*x + m1*y) + (m2*z + m3*w)
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define ATX_HD __host__ __device__ __forceinline__
#else
#include <math.h>
#define ATX_HD inline
#endif

#if defined(__FAST_MATH__)
#error "path arithmetic must not be compiled with fast-math"
#endif

namespace atx {

constexpr float kPi = 3.14159274101257324219f;  // glm::pi<float>()

struct f3 {
    float x, y, z;
};

ATX_HD f3 mk(float x, float y, float z) { f3 r; r.x = x; r.y = y; r.z = z; return r; }
ATX_HD f3 add(f3 a, f3 b) { return mk(a.x + b.x, a.y + b.y, a.z + b.z); }
ATX_HD f3 sub(f3 a, f3 b) { return mk(a.x - b.x, a.y - b.y, a.z - b.z); }
ATX_HD f3 mul(f3 a, f3 b) { return mk(a.x * b.x, a.y * b.y, a.z * b.z); }
ATX_HD f3 scale(f3 a, float s) { return mk(a.x * s, a.y * s, a.z * s); }
ATX_HD f3 divs(f3 a, float s) { return mk(a.x / s, a.y / s, a.z / s); }
ATX_HD f3 neg(f3 a) { return mk(-a.x, -a.y, -a.z); }
ATX_HD float dot(f3 a, f3 b) { return (a.x * b.x + a.y * b.y) + a.z * b.z; }

#if defined(__HIP_DEVICE_COMPILE__)
ATX_HD float sqrt_cr(float x) { return __builtin_sqrtf(x); }   // correctly rounded (HIP default)
ATX_HD float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
ATX_HD float rint_(float x) { return __builtin_rintf(x); }
ATX_HD float fabs_(float x) { return __builtin_fabsf(x); }
#else
ATX_HD float sqrt_cr(float x) { return sqrtf(x); }
ATX_HD float fma_(float a, float b, float c) { return fmaf(a, b, c); }
ATX_HD float rint_(float x) { return rintf(x); }
ATX_HD float fabs_(float x) { return fabsf(x); }
#endif

// ---- square roots and quotients without the compiler's range handling -------
// The compiler's correctly rounded square root takes 14 instructions and its
// division 11, 7 and 5 of them on the slower of the two VALU pipes: scaling
// into and out of range and special cases.  Where the operands are known (or
// tested, one test for several) to lie far from both ends of the exponent
// range, the steps below give the same bits for 8 and 8, and for 5 per further
// quotient by the same divisor (Markstein, "Computation of elementary
// functions on the IBM RISC System/6000 processor", 1990).  Path kernel: 640x360,
// 4 spheres, 64 frames 0.409 -> 0.383 ms (14.5 % fewer vector instructions),
// 1080p, 257 spheres, 256 frames 20.6 -> 20.1 ms (5 % fewer).

// sqrt(d) from y, 1 / sqrt(d) to one ulp; h: half its inverse, closer than y.
ATX_HD float sqrt_from(float d, float y, float& h)
{
    float g = d * y;
    h = 0.5f * y;
    const float e = fma_(-h, g, 0.5f);
    g = fma_(g, e, g);
    h = fma_(h, e, h);
    return fma_(fma_(-g, g, d), h, g);
}
ATX_HD uint32_t bits_of(float x) { return __builtin_bit_cast(uint32_t, x); }
// 1 / s from that h.  The start is moved up one ulp: two steps then round
// correctly for every s, also those just below a power of two.
ATX_HD float inverse_from(float s, float h)
{
    float r = __builtin_bit_cast(float, bits_of(h + h) + 1u);
    r = fma_(fma_(-s, r, 1.0f), r, r);
    return fma_(fma_(-s, r, 1.0f), r, r);
}
// 1 / y from the device's approximation r0, one ulp off at most.  One step rounds
// correctly from any such start but for 33 pairs of divisor and start out of
// 2^23 * 3 (1 - 2^-24 from 1 is one), in which the second steps of `quotient` can
// tie; gfx950's v_rcp_f32, checked over every mantissa, gives none of them.
ATX_HD float reciprocal_from(float y, float r0) { return fma_(fma_(-y, r0, 1.0f), r0, r0); }
// x / y from r, the reciprocal of y.
ATX_HD float quotient(float x, float y, float r)
{
    const float q0 = x * r;
    const float q1 = fma_(fma_(-y, q0, x), r, q0);
    return fma_(fma_(-y, q1, x), r, q1);
}
// x / kPi for |x| in {0} and [2^-90, 2^90] (but for the sign of a zero).
ATX_HD float over_pi(float x)
{
    constexpr float kInv = 0x1.45f306p-2f;   // 1 / kPi
    const float q = x * kInv;
    return fma_(fma_(-kPi, q, x), kInv, q);
}
// 2^-96 <= x <= 2^96: square roots and quotients of such numbers stay normal.
ATX_HD bool mid_range(float x) { return bits_of(x) - 0x0f800000u <= 0x6f800000u - 0x0f800000u; }

ATX_HD float length(f3 a) { return sqrt_cr(dot(a, a)); }
ATX_HD f3 normalize(f3 a)
{
    const float d = dot(a, a);
#if defined(__HIP_DEVICE_COMPILE__)
    float h;
    const float len = sqrt_from(d, __builtin_amdgcn_rsqf(d), h);
    float inv = inverse_from(len, h);
    if (__builtin_expect(!mid_range(d), 0))
        inv = 1.0f / sqrt_cr(d);
    return scale(a, inv);
#else
    return scale(a, 1.0f / sqrt_cr(d));
#endif
}
ATX_HD f3 cross(f3 a, f3 b)
{
    return mk(a.y * b.z - b.y * a.z, a.z * b.x - b.z * a.x, a.x * b.y - b.x * a.y);
}
ATX_HD float gmax(float a, float b) { return a < b ? b : a; }
ATX_HD float gmin(float a, float b) { return b < a ? b : a; }
ATX_HD float gclamp(float x, float lo, float hi) { return gmin(gmax(x, lo), hi); }


// ---- PCG hash (Core/include/Random.h:59-70) --------------------------------
ATX_HD uint32_t pcg_hash(uint32_t seed)
{
    uint32_t state = seed * 747796405u + 2891336453u;
    uint32_t word = ((state >> ((state >> 28u) + 4u)) ^ state) * 277803737u;
    return (word >> 22u) ^ word;
}
// float(seed) / float(UINT32_MAX): float(UINT32_MAX) rounds to 2^32, so the
// quotient is float(seed) * 2^-32 exactly.
ATX_HD float pcg_float(uint32_t& seed)
{
    seed = pcg_hash(seed);
    return (float)seed * 0x1p-32f;
}

// ---- sin / cos: Cody-Waite reduction + Taylor polynomials ------------------
// x = k*pi/2 + r, pi/2 = C1 + C2 + C3 subtracted with one fma per part; sin
// to degree 9 and cos to degree 10 on [-pi/4, pi/4].  Accurate to about one
// ulp for |x| < 100; the path only evaluates x in [0, 2*pi].
ATX_HD void sincos_(float x, float& s, float& c)
{
    const float k = rint_(x * 0x1.45f306p-1f);
    float r = fma_(-k, 0x1.921fb6p+0f, x);
    r = fma_(-k, -0x1.777a5cp-25f, r);
    r = fma_(-k, -0x1.ee59dap-50f, r);
    const float r2 = r * r;
    float p = 0x1.71de3ap-19f;
    p = fma_(p, r2, -0x1.a01a02p-13f);
    p = fma_(p, r2, 0x1.111112p-7f);
    p = fma_(p, r2, -0x1.555556p-3f);
    const float r3 = r2 * r;
    const float ps = fma_(r3, p, r);
    float q = -0x1.27e4fcp-22f;
    q = fma_(q, r2, 0x1.a01a02p-16f);
    q = fma_(q, r2, -0x1.6c16c2p-10f);
    q = fma_(q, r2, 0x1.555556p-5f);
    q = fma_(q, r2, -0.5f);
    const float pc = fma_(q, r2, 1.0f);
    const int quad = ((int)k) & 3;
    const float a = (quad & 1) ? pc : ps;     // sin magnitude source
    const float b = (quad & 1) ? ps : pc;     // cos magnitude source
    s = (quad & 2) ? -a : a;
    c = ((quad + 1) & 2) ? -b : b;
}

ATX_HD float pow5(float x)
{
    const float x2 = x * x;
    const float x4 = x2 * x2;
    return x4 * x;
}

// ---- camera (Engine/src/Camera.cpp:134-195) ---------------------------------
// Column-major 4x4, m[col*4+row].
ATX_HD void mat_vec4(const float* m, float x, float y, float z, float w, float out[4])
{
    for (int r = 0; r < 4; ++r) {
        const float mul0 = m[0 * 4 + r] * x;
        const float mul1 = m[1 * 4 + r] * y;
        const float mul2 = m[2 * 4 + r] * z;
        const float mul3 = m[3 * 4 + r] * w;
        out[r] = (mul0 + mul1) + (mul2 + mul3);
    }
}

// Primary ray direction of pixel (x, y): coord = (x/W, y/H)*2 - 1 (no pixel
// centre offset, no jitter), unprojected and rotated into world space.
ATX_HD f3 camera_ray(const float* inv_proj, const float* inv_view, uint32_t x, uint32_t y,
                     uint32_t width, uint32_t height)
{
    float cx = (float)x / (float)width;
    float cy = (float)y / (float)height;
    cx = cx * 2.0f - 1.0f;
    cy = cy * 2.0f - 1.0f;
    float t[4];
    mat_vec4(inv_proj, cx, cy, 1.0f, 1.0f, t);
    const f3 t3 = mk(t[0] / t[3], t[1] / t[3], t[2] / t[3]);
    const f3 n = normalize(t3);
    float w[4];
    mat_vec4(inv_view, n.x, n.y, n.z, 0.0f, w);
    return normalize(mk(w[0], w[1], w[2]));
}

// ---- BRDF (Engine/src/BRDF.cu:9-70) ----------------------------------------
ATX_HD float distribution_ggx(float n_dot_h, float roughness)
{
    const float a = roughness * roughness;
    const float a2 = a * a;
    const float n_dot_h2 = n_dot_h * n_dot_h;
    float denom = n_dot_h2 * (a2 - 1.0f) + 1.0f;
    denom = kPi * denom * denom;
    return a2 / denom;
}

ATX_HD float geometry_schlick_ggx(float n_dot_v, float roughness)
{
    const float r = roughness + 1.0f;
    const float k = (r * r) / 8.0f;
    return n_dot_v / (n_dot_v * (1.0f - k) + k);
}

ATX_HD f3 cook_torrance(f3 albedo, f3 F0, float metallic, float roughness, f3 N, f3 V, f3 L)
{
    const f3 H = normalize(add(V, L));
    const float n_dot_l = gmax(dot(N, L), 0.0000001f);
    const float n_dot_v = gmax(dot(N, V), 0.0000001f);
    const float n_dot_h = gmax(dot(N, H), 0.0f);
    const float v_dot_h = gmax(dot(V, H), 0.0f);
    const float cos_theta = gclamp(v_dot_h, 0.0f, 1.0f);
    const float p5 = pow5(1.0f - cos_theta);
    const f3 one = mk(1.0f, 1.0f, 1.0f);
    const f3 F = add(F0, scale(sub(one, F0), p5));
    const float D = distribution_ggx(n_dot_h, roughness);
    const float G = geometry_schlick_ggx(n_dot_v, roughness) * geometry_schlick_ggx(n_dot_l, roughness);
    const f3 kD = scale(sub(one, F), 1.0f - metallic);
    const f3 num = scale(F, D * G);
    const float denom = 4.0f * n_dot_l * n_dot_v + 0.001f;
    const f3 specular = divs(num, denom);
    const f3 diffuse = divs(mul(sub(one, F), albedo), kPi);
    return scale(add(mul(kD, diffuse), specular), n_dot_l);
}

#if defined(__HIPCC__)
// cook_torrance for a scene of mild materials (WfScene::mild): the same
// expressions with the quotients above, valid where `ok` comes back true (a
// rounded half-vector term or a specular term near zero leaves it false).
__device__ __forceinline__ f3 cook_torrance_mild(f3 albedo, f3 F0, float metallic, float roughness, f3 N, f3 V, f3 L,
                                                 bool& ok)
{
    const f3 H = normalize(add(V, L));
    const float n_dot_l = gmax(dot(N, L), 0.0000001f);
    const float n_dot_v = gmax(dot(N, V), 0.0000001f);
    const float n_dot_h = gmax(dot(N, H), 0.0f);
    const float v_dot_h = gmax(dot(V, H), 0.0f);
    const float cos_theta = gclamp(v_dot_h, 0.0f, 1.0f);
    const float p5 = pow5(1.0f - cos_theta);
    const f3 one = mk(1.0f, 1.0f, 1.0f);
    const f3 F = add(F0, scale(sub(one, F0), p5));
    const auto over = [](float x, float y) { return quotient(x, y, reciprocal_from(y, __builtin_amdgcn_rcpf(y))); };
    // distribution_ggx: a2 is 0 or at least 2^-40
    const float a = roughness * roughness;
    const float a2 = a * a;
    const float n_dot_h2 = n_dot_h * n_dot_h;
    float d = n_dot_h2 * (a2 - 1.0f) + 1.0f;
    d = kPi * d * d;
    const float D = over(a2, d);
    // geometry_schlick_ggx: 1/8 <= k <= 1/2, so the divisors lie between k and 1
    const float r = roughness + 1.0f;
    const float k = (r * r) / 8.0f;
    const float G = over(n_dot_v, n_dot_v * (1.0f - k) + k) * over(n_dot_l, n_dot_l * (1.0f - k) + k);
    const f3 kD = scale(sub(one, F), 1.0f - metallic);
    const f3 num = scale(F, D * G);
    const float denom = 4.0f * n_dot_l * n_dot_v + 0.001f;
    const float rd = reciprocal_from(denom, __builtin_amdgcn_rcpf(denom));
    const f3 specular = mk(quotient(num.x, denom, rd), quotient(num.y, denom, rd), quotient(num.z, denom, rd));
    // 1 - F is 0 or at least 2^-24 in magnitude, the albedo 0 or at least 2^-40
    const f3 dn = mul(sub(one, F), albedo);
    const f3 diffuse = mk(over_pi(dn.x), over_pi(dn.y), over_pi(dn.z));
    // numerators of the specular term: 0 (wraps to the largest) or at least 2^-80
    const uint32_t least = min(min(bits_of(num.x) - 1u, bits_of(num.y) - 1u), bits_of(num.z) - 1u);
    ok = d >= 0x1p-40f && least >= 0x17800000u - 1u;
    return scale(add(mul(kD, diffuse), specular), n_dot_l);
}
#endif

// ---- samplers (Engine/src/BRDF.cu:72-116) ------------------------------------
ATX_HD f3 to_world(f3 N, float hx, float hy, float hz)
{
    const bool xz = fabs_(N.x) > fabs_(N.y);
    f3 T;
#if defined(__HIP_DEVICE_COMPILE__)
    const float u = xz ? N.x : N.y;
    const float d = u * u + N.z * N.z;   // about 1/2 to 1 for a unit normal
    float h;
    const float s = sqrt_from(d, __builtin_amdgcn_rsqf(d), h);
    const float r = inverse_from(s, h);
    const float tz = quotient(u, s, r), tn = quotient(-N.z, s, r);
    T = xz ? mk(tn, 0.0f, tz) : mk(0.0f, tn, tz);
    // components near zero (or -0) take the compiler's division
    if (__builtin_expect(!(mid_range(d) && fabs_(N.z) >= 0x1p-60f && fabs_(u) >= 0x1p-60f), 0))
#endif
    {
        if (xz)
            T = divs(mk(-N.z, 0.0f, N.x), sqrt_cr(N.x * N.x + N.z * N.z));
        else
            T = divs(mk(0.0f, -N.z, N.y), sqrt_cr(N.y * N.y + N.z * N.z));
    }
    const f3 B = cross(N, T);
    return add(add(scale(T, hx), scale(B, hy)), scale(N, hz));
}

// The next direction of a path (Renderer.cu:381-384): the GGX half-vector
// when the material is metallic (BRDF.cu:95-116: cos theta =
// sqrt((1 - u1) / (1 + (a^2 - 1) u1)), a = roughness^2, sin theta =
// sqrt(1 - cos^2 theta)), else a cosine-weighted direction (BRDF.cu:72-93:
// radius sqrt(u1), height sqrt(1 - u1)).  Both take u1 and u2 from the stream
// in that order and place (radius cos phi, radius sin phi, height) with
// phi = 2 pi u2 in the same frame, so only radius and height depend on the
// branch: written this way a wave whose lanes differ in material runs the
// angle and the frame once.
ATX_HD f3 sample_next(f3 N, bool ggx, float roughness, uint32_t& seed)
{
    const float u1 = pcg_float(seed);
    const float u2 = pcg_float(seed);
    // height = sqrt(A), radius = sqrt(B): the same square roots whichever branch
    float A = 1.0f - u1;
    if (ggx) {
        const float a = roughness * roughness;
        const float den = 1.0f + (a * a - 1.0f) * u1;
#if defined(__HIP_DEVICE_COMPILE__)
        A = quotient(A, den, reciprocal_from(den, __builtin_amdgcn_rcpf(den)));
#else
        A = A / den;
#endif
    }
#if defined(__HIP_DEVICE_COMPILE__)
    float h;
    float height = sqrt_from(A, __builtin_amdgcn_rsqf(A), h);
    float B = ggx ? 1.0f - height * height : u1;
    float radius = sqrt_from(B, __builtin_amdgcn_rsqf(B), h);
    // A is u1's complement (a multiple of 2^-32) or that over a divisor that is
    // a multiple of 2^-24 where it is small: in range unless 0, NaN or far off
    if (__builtin_expect(!(A >= 0x1p-40f && B >= 0x1p-40f), 0)) {
        A = 1.0f - u1;
        if (ggx) {
            const float a = roughness * roughness;
            A = A / (1.0f + (a * a - 1.0f) * u1);
        }
        height = sqrt_cr(A);
        B = ggx ? 1.0f - height * height : u1;
        radius = sqrt_cr(B);
    }
#else
    const float height = sqrt_cr(A);
    const float radius = sqrt_cr(ggx ? 1.0f - height * height : u1);
#endif
    const float phi = 2.0f * kPi * u2;
    float s, c;
    sincos_(phi, s, c);
    return to_world(N, radius * c, radius * s, height);
}

// ---- display (Engine/include/Renderer.h:70-78) -------------------------------
ATX_HD uint32_t to_u8(float v)
{
    const float s = v * 255.0f;
    return (s >= 0.0f) ? ((uint32_t)s & 0xFFu) : 0u;   // NaN -> 0
}
ATX_HD uint32_t rgba8(float r, float g, float b, float a)
{
    return (to_u8(a) << 24) | (to_u8(b) << 16) | (to_u8(g) << 8) | to_u8(r);
}

}  // namespace atx
