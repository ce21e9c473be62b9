/* cbx_debug_t3.h -- test-only diagnostics of the T3 path's device building
 * blocks (tests/native/_build/libcbx_debug_t3.so, built from
 * tests/native/cbx_debug_t3.hip; not part of libcbx_sampler.so or its API).
 * Device memory on the current device, asynchronous on `stream`.  Return codes
 * as in cbx_sampler.h. */
#ifndef CBX_DEBUG_T3_H
#define CBX_DEBUG_T3_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* The T3 MLP's gelu (t3_gelu_f, cbx_split.h), elementwise. */
int cbx_debug_t3_gelu(const float* in, float* out, int64_t n, void* stream);

/* The prompt pass's row groups (t3_group_rows, cbx_group.h): returns their
 * bound G; with rows set, 16 G row numbers or -1 are written there. */
int cbx_debug_t3_groups(const int32_t* act, const int32_t* slots, int32_t n_rows, int32_t n_slots,
                        int32_t* rows, void* stream);

#ifdef __cplusplus
}
#endif
#endif
