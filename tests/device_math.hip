// Device check of the starting values behind path_math.h's short square roots and
// quotients: over every mantissa the reciprocal, square root and inverse square
// root come out correctly rounded.  Loaded by tests/test_gpu_device_math.py.
#include <math.h>
#include <string.h>

#include <vector>

#include "../ataraxia_amd/csrc/path_math.h"

using namespace atx;

namespace {

constexpr uint32_t kMantissas = 1u << 23, kBlock = 256;

// r[0]: reciprocal, r[1]: square root, r[2]: inverse of that
__global__ void k_math(uint32_t exponent, float* r)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= kMantissas)
        return;
    const float x = __builtin_bit_cast(float, (exponent << 23) + i);
    float h;
    r[i] = reciprocal_from(x, __builtin_amdgcn_rcpf(x));
    const float s = sqrt_from(x, __builtin_amdgcn_rsqf(x), h);
    r[kMantissas + i] = s;
    r[2 * kMantissas + i] = inverse_from(s, h);
}

}  // namespace

// Numbers with this exponent (biased, 1 to 253) whose results differ from the
// host's, or a negative HIP error.
extern "C" long device_math_wrong(uint32_t exponent)
{
    std::vector<float> r(3 * (size_t)kMantissas);
    float* d = nullptr;
    hipError_t e = hipMalloc((void**)&d, r.size() * sizeof(float));
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_math, dim3(kMantissas / kBlock), dim3(kBlock), 0, nullptr, exponent, d);
        e = hipGetLastError();
        if (e == hipSuccess) e = hipMemcpy(r.data(), d, r.size() * sizeof(float), hipMemcpyDeviceToHost);
        (void)hipFree(d);
    }
    if (e != hipSuccess)
        return -(long)e;
    long wrong = 0;
    for (uint32_t i = 0; i < kMantissas; ++i) {
        const float x = __builtin_bit_cast(float, (exponent << 23) + i), s = sqrtf(x);
        wrong += r[i] != 1.0f / x;
        wrong += r[kMantissas + i] != s;
        wrong += r[2 * (size_t)kMantissas + i] != 1.0f / s;
    }
    return wrong;
}
