// cbx_debug_t3.hip -- test-only diagnostics of the T3 path
// (libcbx_debug_t3.so, tests/native/cbx_debug_t3.h).
#include <hip/hip_runtime.h>

#include "../../chatterbox.cpp_amd/csrc/cbx_group.h"
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

int cbx_debug_t3_groups(const int32_t* act, const int32_t* slots, int32_t n_rows, int32_t n_slots,
                        int32_t* rows, void* stream) {
    if (n_rows < 1 || n_slots < 1) return CBX_ERR_INVALID;
    const int G = cbx::group_bound(n_rows, n_slots);
    if (!rows) return G;
    if (!act || !slots) return CBX_ERR_INVALID;
    hipLaunchKernelGGL(cbx::t3_group_rows, dim3(1), dim3(cbx::kGroupThreads), 0,
                       (hipStream_t)stream, act, slots, n_rows, G, rows);
    return hipGetLastError() == hipSuccess ? G : CBX_ERR_HIP;
}

}  // extern "C"
