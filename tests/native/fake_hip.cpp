// fake_hip.cpp -- a stand-in for the HIP runtime on a machine without a GPU:
// loaded before libcbx_sampler.so, its functions take the place of the
// runtime's, keep "device" memory on the host, run no kernel, and keep a log of
// launches (L), asynchronous copies (C) and stream waits (S).  fake_fail makes
// the n-th launch or copy from then on return an error (0: none).
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <string>

namespace {
std::string events;
int fail_launch = 0, fail_copy = 0;
hipError_t last = hipSuccess;
alignas(256) char symbol[1 << 20];

hipError_t one(char what, int& left) {
    events += what;
    return left > 0 && --left == 0 ? hipErrorUnknown : hipSuccess;
}
}  // namespace

extern "C" {
void fake_fail(int launch, int copy) {
    fail_launch = launch;
    fail_copy = copy;
    events.clear();
}
const char* fake_events() { return events.c_str(); }

void** __hipRegisterFatBinary(const void*) {
    static void* handle;
    return &handle;
}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*,
                           void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t* lds, hipStream_t* st) {
    *lds = 0;
    *st = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) {
    return last = one('L', fail_launch);
}
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipMemcpyAsync(void* to, const void* from, size_t n, hipMemcpyKind, hipStream_t) {
    memcpy(to, from, n);
    return one('C', fail_copy);
}
hipError_t hipStreamSynchronize(hipStream_t) {
    events += 'S';
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
    *p = calloc(1, n);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) {
    *d = h;
    return hipSuccess;
}
hipError_t hipMemcpy(void* to, const void* from, size_t n, hipMemcpyKind) {
    memcpy(to, from, n);
    return hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t n) {
    memset(p, v, n);
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {  // the header's versioned name
    memset(p, 0, sizeof(*p));
    p->sharedMemPerBlock = p->sharedMemPerBlockOptin = 163840;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) {
    *p = symbol;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "none" : "an error"; }
hipError_t hipStreamCreateWithFlags(hipStream_t* st, unsigned) {
    *st = nullptr;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
}
