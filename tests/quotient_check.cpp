// Host-side check of the quotients of ataraxia_amd/csrc/path_math.h from
// starting values one ulp off to either side.  Built by tests/test_quotient_host.py.
#include <cstdio>
#include <math.h>
#include <string.h>

#include <vector>

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
    // Every divisor's mantissa.  One step from such a start rounds correctly but for
    // 33 pairs of divisor and start, all of starts that are not the nearest number; what
    // the device starts from is checked there (tests/device_math.hip).
    long wrong = 0, wrong_nearest = 0;
    std::vector<uint32_t> at_risk;
    for (uint32_t u = 0x3f800000u; u < 0x40000000u; ++u) {
        const float y = of(u), r = 1.0f / y;
        for (uint32_t k = 0; k < 3; ++k)
            if (reciprocal_from(y, of(bits_of(r) + k - 1u)) != r) {
                ++wrong;
                wrong_nearest += k == 1;
                at_risk.push_back(u);
            }
    }
    std::printf("reciprocals off: %ld, from the nearest start: %ld\n", wrong, wrong_nearest);
    // quotients from those starts, divisors at risk left out: random pairs of the
    // whole range
    uint64_t st = 777;
    long bad = 0;
    for (int i = 0; i < 20000000; ++i) {
        st = st * 6364136223846793005ull + 1442695040888963407ull;
        const uint32_t ex = 47u + (uint32_t)(st >> 8) % 160u, ey = 87u + (uint32_t)(st >> 16) % 80u;
        const uint32_t my = (uint32_t)(st >> 18) & 0x7fffffu;
        const float x = of(ex << 23 | (uint32_t)(st >> 41)), y = of(ey << 23 | my);
        const float r = of(bits_of(1.0f / y) + (uint32_t)(st >> 5) % 3u - 1u);
        bool risk = false;
        for (uint32_t u : at_risk)
            risk |= (u & 0x7fffffu) == my;
        bad += !risk && quotient(x, y, reciprocal_from(y, r)) != x / y;
    }
    // and all numerators over the divisors at risk, from the nearest start
    for (uint32_t u : at_risk)
        for (uint32_t m = 0x3f800000u; m < 0x40000000u; m += 3u)
            bad += quotient(of(m), of(u), reciprocal_from(of(u), 1.0f / of(u))) != of(m) / of(u);
    std::printf("quotients off: %ld\n", bad);
    return wrong != 33 || wrong_nearest != 0 || bad != 0;
}
