// cbx_weights.h -- the matrix formats' blocks as the fp16 matrix cores take
// them, shared by the products (cbx_head.hip, cbx_tile.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "cbx_internal.h"
#include "cbx_split.h"
#include "../../include/cbx_sampler.h"

namespace cbx {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
constexpr int32_t kBufWord3 = 0x00020000;  // raw buffer: 32-bit data format

__device__ __forceinline__ float half_bits_to_float(uint32_t hb) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)hb);
}

// Bytes of one block of 32 weights (F16: 32 halves).
template <int WT>
constexpr int block_bytes() {
    return WT == CBX_WTYPE_F16 ? 64 : WT == CBX_WTYPE_Q4_0 ? 18 : WT == CBX_WTYPE_Q5_0 ? 22 : 34;
}

// Bits 0..3 of x to bit 4 of bytes 0..3 (the four products x << 7i land in
// disjoint bit ranges: no carries).
__device__ __forceinline__ uint32_t spread4(uint32_t x) {
    return ((x * 0x00204081u) & 0x01010101u) << 4;
}

// Two bytes b0, b1 of x (bytes sel0, sel1) as fp16 (b - off): the byte under
// the high byte 0x64 is the fp16 1024 + b, exactly, and the packed fp16
// subtraction of 1024 + off leaves b - off (an integer of at most 8 bits:
// exact).
__device__ __forceinline__ uint32_t bytes_f16(uint32_t x, uint32_t sel, _Float16 off) {
    const uint32_t v = __builtin_amdgcn_perm(0x64646464u, x, sel);
    const h2 r = __builtin_bit_cast(h2, v) - h2{off, off};
    return __builtin_bit_cast(uint32_t, r);
}

// The 8 integer weights of lds_w's bytes as fp16: Q4_0 n - 8, Q5_0 q - 16
// (q = n | the element's qh bit << 4), Q8_0 q; and the block's scale d.
template <int WT>
__device__ __forceinline__ u4v int_weights(const uint32_t* q, int g, float& d) {
    d = half_bits_to_float(q[4]);
    uint32_t x0, x1;
    _Float16 off;
    if constexpr (WT == CBX_WTYPE_Q4_0) {
        const int sh = g < 2 ? 0 : 4;
        x0 = (q[0] >> sh) & 0x0f0f0f0fu;
        x1 = (q[1] >> sh) & 0x0f0f0f0fu;
        off = (_Float16)1032.0f;
    } else if constexpr (WT == CBX_WTYPE_Q5_0) {
        // lane group g holds elements 8g .. 8g + 7: qh bits 8g .. 8g + 7
        const int sh = g < 2 ? 0 : 4;
        const uint32_t hb = q[2] >> (8 * g);
        x0 = ((q[0] >> sh) & 0x0f0f0f0fu) | spread4(hb & 15u);
        x1 = ((q[1] >> sh) & 0x0f0f0f0fu) | spread4((hb >> 4) & 15u);
        off = (_Float16)1040.0f;
    } else {
        x0 = q[0] ^ 0x80808080u;
        x1 = q[1] ^ 0x80808080u;
        off = (_Float16)1152.0f;
    }
    // selector bytes: 0-3 the bytes of x, 4 the constant's 0x64
    return u4v{bytes_f16(x0, 0x04010400u, off), bytes_f16(x0, 0x04030402u, off),
               bytes_f16(x1, 0x04010400u, off), bytes_f16(x1, 0x04030402u, off)};
}

__device__ __forceinline__ f4 mfma_f16(const u4v& a, const u4v& b, const f4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, a),
                                                  __builtin_bit_cast(h8, b), c, 0, 0, 0);
}

// Where k or v of row r, column v >= n of a q|k|v product of n columns each
// goes (NULL: nowhere); every 32 columns from a multiple of 32 lie in one head.
__device__ __forceinline__ float* kv_place(const KvOut& kv, int r, int v) {
    if (!kv.act[r]) return nullptr;
    const int n = kv.n_head * 64, c = v - n < n ? v - n : v - 2 * n;
    return (v < 2 * n ? kv.kc : kv.vc) +
           ((((int64_t)kv.slots[r] * kv.n_layer + kv.layer) * kv.n_head + (c >> 6)) * kv.n_ctx +
            kv.positions[r]) * 64 + (c & 63);
}

}  // namespace cbx
