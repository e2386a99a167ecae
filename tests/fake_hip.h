// The HIP calls of the library's host code over plain host memory, for host
// checks of its error paths: allocations that fail on request, and two devices, of
// which an event and the stream it is recorded on have to share one.  Kernels are
// not launched.
#pragma once

#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "wavefront_host.h"

namespace fake {
inline int fail_mallocs = 0;     // the next so many device allocations fail
inline int kernel_launches = 0;
inline thread_local int device = 0;   // the thread's current one
struct Owned {
    int device;
};
}  // namespace fake

extern "C" {
hipError_t hipGetDeviceCount(int* n) { *n = 2; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = fake::device; return hipSuccess; }
hipError_t hipSetDevice(int d) { fake::device = d; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 4; return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "fake error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n)
{
    *p = nullptr;
    if (fake::fail_mallocs > 0) {
        --fake::fail_mallocs;
        return hipErrorOutOfMemory;
    }
    *p = calloc(1, n);
    return hipSuccess;
}
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = calloc(1, n); return hipSuccess; }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t*, const void*) { return hipErrorInvalidValue; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t) new fake::Owned{fake::device}; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { delete (fake::Owned*)s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t* d) { *d = ((fake::Owned*)s)->device; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t) new fake::Owned{fake::device}; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { delete (fake::Owned*)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    return ((fake::Owned*)e)->device == ((fake::Owned*)s)->device ? hipSuccess : hipErrorInvalidHandle;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0.0f; return hipSuccess; }
}

namespace atx {
hipError_t launch_wavefront(const WfPass&, const WfLaunch&, hipStream_t, hipEvent_t) { ++fake::kernel_launches; return hipSuccess; }
hipError_t launch_in_place(const WfScene&, const WfPass&, hipStream_t) { ++fake::kernel_launches; return hipSuccess; }
hipError_t launch_first_hits(const WfScene&, hipStream_t) { ++fake::kernel_launches; return hipSuccess; }
hipError_t launch_camera_dirs(const WfScene&, float4*, hipStream_t) { ++fake::kernel_launches; return hipSuccess; }
hipError_t launch_zero_u32(unsigned int*, uint32_t, hipStream_t) { ++fake::kernel_launches; return hipSuccess; }
int wavefront_max_blocks_per_cu(bool, uint32_t) { return 5; }
}  // namespace atx
