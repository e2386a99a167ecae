// Host-side check of the square roots and quotients of
// ataraxia_amd/csrc/path_math.h: over every mantissa, with starting values one
// ulp off to either side, they round as the compiler's do; quotients over many
// random pairs.  Built by tests/test_math_host.py.
#include <cstdio>
#include <cstring>
#include <math.h>
#include <stdint.h>
#include <string.h>

#include "../ataraxia_amd/csrc/path_math.h"

using namespace atx;

static float of(uint32_t u)
{
    float x;
    memcpy(&x, &u, 4);
    return x;
}

int main()
{
    long bad = 0;
    for (uint32_t u = 0x3f800000u; u < 0x40800000u; ++u) {   // [1, 4): both parities of the exponent
        const float d = of(u), s = sqrtf(d), inv = 1.0f / s;
        const uint32_t y = bits_of((float)(1.0 / sqrt((double)d)));
        for (uint32_t k = 0; k < 3; ++k) {
            float h;
            bad += sqrt_from(d, of(y + k - 1u), h) != s;
            bad += inverse_from(s, h) != inv;
        }
    }
    std::printf("square roots: %ld\n", bad);
    for (uint32_t u = 0x3f800000u; u < 0x40000000u; ++u)
        bad += over_pi(of(u)) != of(u) / kPi || reciprocal_from(of(u), 1.0f / of(u)) != 1.0f / of(u);
    std::printf("over pi, reciprocals: %ld\n", bad);
    uint64_t st = 12345;
    for (int i = 0; i < 20000000; ++i) {
        st = st * 6364136223846793005ull + 1442695040888963407ull;
        // exponents from the declared ends of the range
        const uint32_t ex = 47u + (uint32_t)(st >> 8) % 160u, ey = 87u + (uint32_t)(st >> 16) % 80u;
        const float x = of(ex << 23 | (uint32_t)(st >> 41)), y = of(ey << 23 | ((uint32_t)(st >> 18) & 0x7fffffu));
        bad += quotient(x, y, reciprocal_from(y, 1.0f / y)) != x / y;
        bad += quotient(0.0f, y, reciprocal_from(y, 1.0f / y)) != 0.0f;
    }
    std::printf("quotients: %ld\n", bad);
    bad += mid_range(0.0f) || mid_range(-1.0f) || mid_range(of(0x7f800000u)) || mid_range(of(0x7fc00000u)) ||
           mid_range(0x1.fffffep-97f) || !mid_range(0x1p-96f) || !mid_range(0x1p+96f) || mid_range(0x1.000002p+96f);
    std::printf("ranges: %ld\n", bad);
    return bad != 0;
}
