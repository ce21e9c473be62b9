// cbx_debug_t3.hip -- test-only diagnostics of the T3 path
// (libcbx_debug_t3.so, tests/native/cbx_debug_t3.h).
#include <hip/hip_runtime.h>

#include "../../chatterbox.cpp_amd/csrc/cbx_split.h"
#include "../../include/cbx_sampler.h"
#include "cbx_debug_t3.h"

namespace {
__global__ void gelu_kernel(const float* in, float* out, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = cbx::t3_gelu_f(in[i]);
}
}  // namespace

extern "C" {

int cbx_debug_t3_gelu(const float* in, float* out, int64_t n, void* stream) {
    if (!in || !out || n < 1) return CBX_ERR_INVALID;
    hipLaunchKernelGGL(gelu_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                       (hipStream_t)stream, in, out, n);
    return hipGetLastError() == hipSuccess ? CBX_OK : CBX_ERR_HIP;
}

}  // extern "C"
