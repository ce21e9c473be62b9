// cbx_t3.hip -- one decode step of the T3 transformer (GPT-2) for n streams,
// each at its own position with its own KV cache: the step graph of
// src/main.cpp:617-633 through build_transformer_core (main.cpp:469-575),
// up to ln_f's output.
//
// Per step, for every stream row:
//   x  = speech_emb[token] + wpe[pos]                       (main.cpp:628-630)
//   per layer l:
//     u   = LN(x) * ln_1_g + ln_1_b                          (:522-523)
//     qkv = c_attn u + b                                     (:524)
//     k, v of this position appended to the stream's cache   (:517-531)
//     a   = softmax(q . K^T / sqrt(64)) V over [0, pos]      (:542-548, N = 1)
//     x  += c_proj a + b                                     (:551)
//     u   = LN(x) * ln_2_g + ln_2_b                          (:554-555)
//     x  += mlp_proj gelu(mlp_fc u + b) + b                  (:556-559)
//   hidden = LN(x) * ln_f_g + ln_f_b                         (:562-563)
// LN(x) = (x - mean) / sqrt(var + eps), var the mean square of x - mean
// (ggml_norm); gelu the tanh form 0.5 x (1 + tanh(sqrt(2/pi) x (1 +
// 0.044715 x^2))) (Hendrycks and Gimpel's approximation, ggml_gelu's).
//
// The four matrix products of a layer have the speech_head's shape (rows of
// n_in weights per output, F16 / Q4_0 / Q5_0 / Q8_0): they run on the head's
// kernels (fp16 matrix cores on split activations from 4 rows, a mat-vec
// below).  From 4 rows the layer norms write the split activations of the
// products they feed themselves, and the two products the residual adds
// take a K split over workgroups when their grid is narrow, their slabs
// added by the norm that follows; gelu is applied as the mlp c_fc product
// stores its outputs.  The kernels here are the row-wise rest: the
// embedding, the residual add fused with the next layer norm, and the
// attention with its cache append (a decode step: a workgroup of 4 waves per
// stream and head, 16 when there are few; the prompt pass: fp32 matrix-core
// tiles of 16 rows).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "cbx_group.h"
#include "cbx_internal.h"
#include "cbx_split.h"
#include "cbx_weights.h"
#include "../../include/cbx_t3.h"

namespace cbx {
namespace {

constexpr int kNormThreads = 256;
constexpr int kHeadDim = 64;
// Products split over K write up to this many slabs.
constexpr int kMaxKSplit = 8;

struct NormArgs {
    int32_t n_embd;
    float eps;
    float* x;              // residual rows [n_rows][n_embd], in/out
    const float* y;        // when set, the ny slabs y + z * ystride (a product
    int32_t ny;            //   split over K, in slab order) are added to x
    int64_t ystride;
    // embedding mode (emb set): x = emb[token] + wpe[pos], or x = inputs[r]
    const float* emb;
    const float* wpe;
    const float* inputs;
    const int32_t* tokens;
    int32_t* positions;
    const int32_t* state;
    const int32_t* slots;  // prefill: the cache slot of each row
    const int32_t* rows;   // prefill: the rows in groups of 16 (t3_group_rows; NULL: in order)
    int32_t n_slots;
    int32_t n_vocab, n_pos, n_ctx;
    int32_t* act;          // per row: 1 when the stream takes this step
    const float* g;
    const float* b;
    float* out;            // LN(x) * g + b
    uint32_t* parts;       // when set, LN(x) * g + b goes there instead, split
    float* inv;            //   for the next product (cbx_split.h), the scales here
    int32_t advance;       // last norm of the step: positions[r] += 1
};

// Whether row r takes this step (embedding mode; stored for the norms after).
__device__ __forceinline__ bool norm_active(const NormArgs& a, int r, int pos, int tok) {
    const int slot = a.slots ? a.slots[r] : r;
    return (!a.state || a.state[r] == CBX_DECODE_RUNNING) && pos >= 0 && pos < a.n_ctx &&
           pos < a.n_pos && (a.inputs || (tok >= 0 && tok < a.n_vocab)) &&
           (!a.slots || (slot >= 0 && slot < a.n_slots));
}

// One row per workgroup: the embedding or the residual add, then the layer
// norm.  Inactive rows (streams that take no step) keep x and write zeros.
template <int EPT>
__global__ __launch_bounds__(kNormThreads) void t3_norm(NormArgs a) {
    __shared__ float red[8];
    int ph = 0;
    const int r = blockIdx.x, tid = threadIdx.x;
    const int n = a.n_embd;
    float* xr = a.x + (int64_t)r * n;
    float* orow = a.out + (int64_t)r * n;
    bool active;
    float xv[EPT];
    if (a.emb || a.inputs) {
        const int pos = a.positions[r];
        const int tok = a.tokens ? a.tokens[r] : 0;
        active = norm_active(a, r, pos, tok);
        if (tid == 0) a.act[r] = active ? 1 : 0;
        if (!active) {
#pragma unroll
            for (int j = 0; j < EPT; ++j) {
                xr[j * kNormThreads + tid] = 0.0f;
                orow[j * kNormThreads + tid] = 0.0f;
            }
            return;
        }
        if (a.inputs) {
            const float* in = a.inputs + (int64_t)r * n;
#pragma unroll
            for (int j = 0; j < EPT; ++j) xv[j] = in[j * kNormThreads + tid];
        } else {
            const float* e = a.emb + (int64_t)tok * n;
            const float* p = a.wpe + (int64_t)pos * n;
#pragma unroll
            for (int j = 0; j < EPT; ++j)
                xv[j] = __fadd_rn(e[j * kNormThreads + tid], p[j * kNormThreads + tid]);
        }
    } else {
        active = a.act[r] != 0;
        if (!active) {
#pragma unroll
            for (int j = 0; j < EPT; ++j) orow[j * kNormThreads + tid] = 0.0f;
            return;
        }
        // the product's slabs (all loads issued first), added in slab order,
        // then the residual (main.cpp:551, :559)
        float ys[kMaxKSplit][EPT];
#pragma unroll
        for (int j = 0; j < EPT; ++j) xv[j] = xr[j * kNormThreads + tid];
        if (a.y) {
            const float* yr = a.y + (int64_t)r * n + tid;
#pragma unroll
            for (int z = 0; z < kMaxKSplit; ++z)
#pragma unroll
                for (int j = 0; j < EPT; ++j)
                    ys[z][j] = z < a.ny ? yr[z * a.ystride + j * kNormThreads] : 0.0f;
#pragma unroll
            for (int j = 0; j < EPT; ++j) {
                float c = ys[0][j];
#pragma unroll
                for (int z = 1; z < kMaxKSplit; ++z)
                    if (z < a.ny) c = __fadd_rn(c, ys[z][j]);
                xv[j] = __fadd_rn(c, xv[j]);
            }
        }
    }
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < EPT; ++j) s = __fadd_rn(s, xv[j]);
    const float mean = __fdiv_rn(block_sum256(s, red, ph), (float)n);
    float q = 0.0f;
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
        const float d = __fsub_rn(xv[j], mean);
        q = __fadd_rn(q, __fmul_rn(d, d));
    }
    const float var = __fdiv_rn(block_sum256(q, red, ph), (float)n);
    const float scale = __fdiv_rn(1.0f, __fsqrt_rn(__fadd_rn(var, a.eps)));
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
        const int i = j * kNormThreads + tid;
        xr[i] = xv[j];
        orow[i] = __fadd_rn(__fmul_rn(__fmul_rn(__fsub_rn(xv[j], mean), scale), a.g[i]), a.b[i]);
    }
    if (a.advance && tid == 0) a.positions[r] += 1;
}

// The same with the norm's rows written split for the matrix cores (a.parts):
// thread j holds values 8j .. 8j + 7 of the row, a group of the split, so the
// loads are 16 bytes a lane and the values go from the sums to the split in
// registers (256 threads of every 256th value each passed them through the
// LDS and left half the threads without a group at 1024).
// us per step or pass at n_embd 1024 (48 of these), 256 threads -> here: 64
// streams 1605 -> 1517, 6 streams Q8_0 1115 -> 1025, one prompt of 251 rows 1815
// -> 1743, 64 prompts of 129-383 rows 31710 -> 31650.
constexpr int kNormSplitMax = 512;  // n_embd 4096
template <int NY>
__global__ __launch_bounds__(kNormSplitMax) void t3_norm_split(NormArgs a) {
    __shared__ float red[2][kNormSplitMax / 64];
    const int r = blockIdx.x, j = threadIdx.x, n = a.n_embd, nw = (int)blockDim.x / 64;
    const bool in = 8 * j < n;  // n_embd 256, 768: the last wave's rest
    const int k = in ? 8 * j : 0;
    float* const xr = a.x + (int64_t)r * n + k;
    const auto load8 = [](const float* p, float (&v)[8]) {
        const f4 u = *reinterpret_cast<const f4*>(p), w = *reinterpret_cast<const f4*>(p + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = u[i];
            v[4 + i] = w[i];
        }
    };
    const auto store8 = [](float* p, const float (&v)[8]) {
        *reinterpret_cast<f4*>(p) = f4{v[0], v[1], v[2], v[3]};
        *reinterpret_cast<f4*>(p + 4) = f4{v[4], v[5], v[6], v[7]};
    };
    float xv[8], gv[8], bv[8];
    bool active;
    if constexpr (NY == 0) {  // the embedding or the input row
        const int pos = a.positions[r];
        const int tok = a.tokens ? a.tokens[r] : 0;
        active = norm_active(a, r, pos, tok);
        if (j == 0) a.act[r] = active ? 1 : 0;
        if (active && a.inputs) {
            const float* const p = a.inputs + (int64_t)r * n + k;  // of any alignment
#pragma unroll
            for (int i = 0; i < 8; ++i) xv[i] = p[i];
        } else if (active) {
            const float* const e = a.emb + (int64_t)tok * n + k;
            const float* const p = a.wpe + (int64_t)pos * n + k;
#pragma unroll
            for (int i = 0; i < 8; ++i) xv[i] = __fadd_rn(e[i], p[i]);
        }
    } else {
        // the product's slabs, added in slab order, then the residual
        // (main.cpp:551, :559); loaded beside the flag
        float ys[NY][8];
        active = a.act[r] != 0;
        load8(xr, xv);
#pragma unroll
        for (int z = 0; z < NY; ++z) load8(a.y + (int64_t)z * a.ystride + (int64_t)r * n + k, ys[z]);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            float c = ys[0][i];
#pragma unroll
            for (int z = 1; z < NY; ++z) c = __fadd_rn(c, ys[z][i]);
            xv[i] = __fadd_rn(c, xv[i]);
        }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        gv[i] = a.g[k + i];
        bv[i] = a.b[k + i];
    }
    if (!active) {
        if (!in) return;
        const float zero[8] = {};
        if (NY == 0) store8(xr, zero);
        split_store(a.parts, r >> 4, r & 15, n / 32, j, zero, 1.0f);
        if ((j & 3) == 0) a.inv[split_inv_index(r >> 4, r & 15, n / 32, j >> 2)] = 1.0f;
        return;
    }
    // a wave's sum as block_sum256's, the waves' in order
    const auto block_sum = [&](float v, float* h) {
        v = sum16_dpp(in ? v : 0.0f);
        const auto lane_v = [&](int l) {
            return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
        };
        const float w = __fadd_rn(__fadd_rn(lane_v(0), lane_v(16)), __fadd_rn(lane_v(32), lane_v(48)));
        if (nw == 1) return w;
        if ((j & 63) == 0) h[j >> 6] = w;
        __syncthreads();
        float s = h[0];
        for (int i = 1; i < nw; ++i) s = __fadd_rn(s, h[i]);
        return s;
    };
    const auto sum8 = [](const float (&v)[8]) {
        return __fadd_rn(__fadd_rn(__fadd_rn(v[0], v[1]), __fadd_rn(v[2], v[3])),
                         __fadd_rn(__fadd_rn(v[4], v[5]), __fadd_rn(v[6], v[7])));
    };
    const float mean = __fdiv_rn(block_sum(sum8(xv), red[0]), (float)n);
    float d[8], q[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        d[i] = __fsub_rn(xv[i], mean);
        q[i] = __fmul_rn(d[i], d[i]);
    }
    const float var = __fdiv_rn(block_sum(sum8(q), red[1]), (float)n);
    const float scale = __fdiv_rn(1.0f, __fsqrt_rn(__fadd_rn(var, a.eps)));
    float mx = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        d[i] = __fadd_rn(__fmul_rn(__fmul_rn(d[i], scale), gv[i]), bv[i]);
        mx = fmaxf(mx, fabsf(d[i]));
    }
    mx = split_block_max4(mx);
    if (!in) return;
    store8(xr, xv);
    float sc, sinv;
    split_scale(mx, sc, sinv);
    split_store(a.parts, r >> 4, r & 15, n / 32, j, d, sc);
    if ((j & 3) == 0) a.inv[split_inv_index(r >> 4, r & 15, n / 32, j >> 2)] = sinv;
}

struct AttnArgs {
    const float* qkv;      // [n_rows][3 n_embd]: q | k | v, head h at h*64
    float* kc;             // this layer's caches: stream r, head h at
    float* vc;             //   ((r * n_layer + layer) * n_head + h) * n_ctx * 64
    int32_t n_layer, layer, n_head, n_ctx;
    const int32_t* positions;
    const int32_t* act;
    const int32_t* slots;  // prefill: the cache slot of each row
    const int32_t* rows;   // prefill: the rows in groups of 16 (t3_group_rows; NULL: in order)
    float* out;            // [n_rows][n_embd]
    uint32_t* parts;       // when set, the rows go there instead, split for the
    float* inv;            //   next product (cbx_split.h), the scales here
    float scale;           // 1 / sqrt(64)
};

// Element `lane` (0..63) of head h of row r's attention output, o, from wave
// 0: to out, or split (the head's 64 values are blocks 2h and 2h + 1 of the
// row: lanes 0-31 and 32-63, each block scaled by its own largest magnitude,
// pairs of lanes joining their fp16 halves into dwords).
__device__ __forceinline__ void attn_store(const AttnArgs& a, int r, int h, int lane, float o) {
    const int n = a.n_head * kHeadDim;
    if (!a.parts) {
        a.out[(int64_t)r * n + h * kHeadDim + lane] = o;
        return;
    }
    float mx = fabsf(o);
#pragma unroll
    for (int q = 1; q < 32; q <<= 1) mx = fmaxf(mx, __shfl_xor(mx, q));
    float sc, sinv;
    split_scale(mx, sc, sinv);
    const float y = __fmul_rn(o, sc);
    const _Float16 hh = (_Float16)y;
    const _Float16 ll = (_Float16)__fsub_rn(y, (float)hh);
    const uint32_t hv = __builtin_bit_cast(uint16_t, hh), lv = __builtin_bit_cast(uint16_t, ll);
    const uint32_t ho = (uint32_t)__shfl_xor((int)hv, 1), lo = (uint32_t)__shfl_xor((int)lv, 1);
    const int nball = n / 32, kb = 2 * h + (lane >> 5), k = lane & 31;
    const int T = r >> 4, m = r & 15;
    if ((lane & 1) == 0) {
        // dword (k % 8) / 2 of lane 16 (k / 8) + m's hi (lo) 16 bytes
        uint32_t* const base =
            a.parts + ((int64_t)T * nball + kb) * 512 + 4 * (16 * (k >> 3) + m) + (k & 7) / 2;
        base[0] = hv | (ho << 16);
        base[256] = lv | (lo << 16);
    }
    if (k == 0) a.inv[split_inv_index(T, m, nball, kb)] = sinv;
}


__device__ __forceinline__ f4 mfma_f32(float x, float y, const f4& acc) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, acc, 0, 0, 0);
}

// Dimensions 4c .. 4c + 3 of head h of row r's attention output from lane c
// of a 16-lane row (every lane of the wave takes part; nothing stored past
// n_rows): to out, or split as attn_store does (block 2h + c / 8, its largest
// magnitude over 8 lanes).
__device__ __forceinline__ void attn_store4(const AttnArgs& a, int n_rows, int r, int h, int c,
                                            const f4& o) {
    if (!a.parts) {
        if (r < n_rows)
            *reinterpret_cast<f4*>(a.out + (int64_t)r * a.n_head * kHeadDim + h * kHeadDim + 4 * c) = o;
        return;
    }
    float mx = fmaxf(fmaxf(fabsf(o[0]), fabsf(o[1])), fmaxf(fabsf(o[2]), fabsf(o[3])));
#pragma unroll
    for (int x = 1; x < 8; x <<= 1) mx = fmaxf(mx, __shfl_xor(mx, x));
    if (r >= n_rows) return;
    float sc, sinv;
    split_scale(mx, sc, sinv);
    uint32_t hi[2], lo[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const float y0 = __fmul_rn(o[2 * i], sc), y1 = __fmul_rn(o[2 * i + 1], sc);
        const _Float16 h0 = (_Float16)y0, h1 = (_Float16)y1;
        hi[i] = __builtin_bit_cast(uint32_t, split_h2{h0, h1});
        lo[i] = __builtin_bit_cast(uint32_t, split_h2{(_Float16)__fsub_rn(y0, (float)h0),
                                                      (_Float16)__fsub_rn(y1, (float)h1)});
    }
    const int nball = a.n_head * kHeadDim / 32, kb = 2 * h + (c >> 3), T = r >> 4, m = r & 15;
    // values 4 (c % 8) .. of the block: half (c & 1) of group (c % 8) / 2
    uint32_t* const d =
        a.parts + ((int64_t)T * nball + kb) * 512 + 4 * (16 * ((c & 7) >> 1) + m) + 2 * (c & 1);
    *reinterpret_cast<uint2*>(d) = make_uint2(hi[0], hi[1]);
    *reinterpret_cast<uint2*>(d + 256) = make_uint2(lo[0], lo[1]);
    if ((c & 7) == 0) a.inv[split_inv_index(T, m, nball, kb)] = sinv;
}

// Prefill: every row's k and v stored at its slot and position before any
// row attends, so rows of one stream in one call see each other causally.
// Here after the mat-vecs (a call of up to 3 rows); the matrix-core products
// store k and v there themselves (a pass over 180 MB and a launch less per
// layer: 83 us at 14975 rows, 4.2 at 251).
__global__ __launch_bounds__(kHeadDim) void t3_kv_append(AttnArgs a) {
    const int r = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
    if (!a.act[r]) return;
    const int n = a.n_head * kHeadDim;
    const int slot = a.slots[r], pos = a.positions[r];
    const float* qr = a.qkv + (int64_t)r * 3 * n + h * kHeadDim;
    const int64_t base =
        (((int64_t)slot * a.n_layer + a.layer) * a.n_head + h) * a.n_ctx * kHeadDim + (int64_t)pos * kHeadDim;
    a.kc[base + lane] = qr[n + lane];
    a.vc[base + lane] = qr[2 * n + lane];
}

// One workgroup of kAttnWaves waves per (stream, head).  Wave 0 stores the
// new k and v at the stream's position (and keeps them in LDS: that position
// is never read back from memory).  The positions are cut into
// kAttnWaves runs, one per wave; a wave's lanes take 16 per cache row, 4 rows
// per load instruction, kAttnBatch rows per lane in flight, and go over the
// run once with a running softmax (max, sum, weighted v sums, rescaled as the
// max grows); the runs of the 4 row groups of a wave and of the waves are
// merged by the same rescaling in a fixed order.  4 waves x 6 rows (every
// workgroup resident at once; 16 waves when rows x heads are under 256, see
// t3_attn_wide); measured at 64 streams 1.89 -> 1.85 ms per step against 4 x 8.
template <int kAttnBatch, int kAttnWaves>
__global__ __launch_bounds__(kAttnWaves * kHeadDim) void t3_attn(AttnArgs a) {
    __shared__ __align__(16) float kn_s[kHeadDim];
    __shared__ __align__(16) float vn_s[kHeadDim];
    __shared__ float red[2 * kAttnWaves];
    __shared__ __align__(16) float part[kAttnWaves][kHeadDim];
    const int r = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
    const int lane = tid & 63, w = tid >> 6;
    const int n = a.n_head * kHeadDim;
    if (!a.act[r]) {
        if (tid < kHeadDim) attn_store(a, r, h, tid, 0.0f);
        return;
    }
    const int pos = a.positions[r];
    const float* qr = a.qkv + (int64_t)r * 3 * n + h * kHeadDim;
    const int64_t base = (((int64_t)r * a.n_layer + a.layer) * a.n_head + h) * a.n_ctx * kHeadDim;
    float* kc = a.kc + base;
    float* vc = a.vc + base;
    if (w == 0) {
        const float kn = qr[n + lane], vn = qr[2 * n + lane];
        kc[(int64_t)pos * kHeadDim + lane] = kn;
        vc[(int64_t)pos * kHeadDim + lane] = vn;
        kn_s[lane] = kn;
        vn_s[lane] = vn;
    }
    // lane = 16 sub + e holds q[4e .. 4e + 3] and takes position c0 + sub + 4i,
    // dimensions 4e .. 4e + 3: a wave reads 4 rows of k per instruction
    const int sub = lane >> 4, e4 = 4 * (lane & 15);
    const float4 q4 = *reinterpret_cast<const float4*>(qr + e4);
    // positions [0, L) in kAttnWaves runs
    const int L = pos + 1;
    const int run = (L + kAttnWaves - 1) / kAttnWaves;
    const int c0 = min(w * run, L), c1 = min(c0 + run, L);
    __syncthreads();
    // Each lane keeps, over the positions of its 16-lane group (position order),
    // the running max m of the scores, the sum s of expf(score - m) and the
    // sums acc of expf(score - m) v[4e .. 4e + 3], rescaled whenever m grows
    // (one pass: k and v rows of a batch are loaded together, kAttnBatch per
    // lane, a row past the run reading the run's last row, unused; the new
    // position's k and v are taken from LDS, their stores above need not be
    // visible).
    const float4 kn4 = *reinterpret_cast<const float4*>(kn_s + e4);
    const float4 vn4 = *reinterpret_cast<const float4*>(vn_s + e4);
    float m = -INFINITY, s = 0.0f;
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int j0 = c0; j0 < c1; j0 += 4 * kAttnBatch) {
        float4 kk[kAttnBatch], vv[kAttnBatch];
#pragma unroll
        for (int u = 0; u < kAttnBatch; ++u) {
            const int64_t jc = min(j0 + 4 * u + sub, c1 - 1);
            kk[u] = *reinterpret_cast<const float4*>(kc + jc * kHeadDim + e4);
            vv[u] = *reinterpret_cast<const float4*>(vc + jc * kHeadDim + e4);
        }
        float sc[kAttnBatch];
        float bm = -INFINITY;
#pragma unroll
        for (int u = 0; u < kAttnBatch; ++u) {
            const int j = j0 + 4 * u + sub;
            const float4 k4 = j == pos ? kn4 : kk[u];
            float dot = __fadd_rn(__fadd_rn(__fmul_rn(q4.x, k4.x), __fmul_rn(q4.y, k4.y)),
                                  __fadd_rn(__fmul_rn(q4.z, k4.z), __fmul_rn(q4.w, k4.w)));
            // the 16 lanes of a row: butterfly over e (the same sum in each)
            dot = sum16_dpp(dot);
            sc[u] = __fmul_rn(dot, a.scale);
            if (j < c1) bm = fmaxf(bm, sc[u]);
        }
        if (bm > m) {
            const float f = m == -INFINITY ? 0.0f : expf(__fsub_rn(m, bm));
            s = __fmul_rn(s, f);
            acc.x = __fmul_rn(acc.x, f);
            acc.y = __fmul_rn(acc.y, f);
            acc.z = __fmul_rn(acc.z, f);
            acc.w = __fmul_rn(acc.w, f);
            m = bm;
        }
#pragma unroll
        for (int u = 0; u < kAttnBatch; ++u) {
            const int j = j0 + 4 * u + sub;
            if (j < c1) {
                const float e = expf(__fsub_rn(sc[u], m));
                const float4 v4 = j == pos ? vn4 : vv[u];
                s = __fadd_rn(s, e);
                acc.x = __fadd_rn(acc.x, __fmul_rn(e, v4.x));
                acc.y = __fadd_rn(acc.y, __fmul_rn(e, v4.y));
                acc.z = __fadd_rn(acc.z, __fmul_rn(e, v4.z));
                acc.w = __fadd_rn(acc.w, __fmul_rn(e, v4.w));
            }
        }
    }
    // the 4 groups of a wave, then the 4 waves, merged by the same rescaling:
    // each pair's two products added in either lane give the same sum
#pragma unroll
    for (int o = 16; o <= 32; o <<= 1) {
        const float mo = __shfl_xor(m, o), so = __shfl_xor(s, o);
        const float4 ao = make_float4(__shfl_xor(acc.x, o), __shfl_xor(acc.y, o),
                                      __shfl_xor(acc.z, o), __shfl_xor(acc.w, o));
        const float M = fmaxf(m, mo);
        const float f = m == -INFINITY ? 0.0f : expf(__fsub_rn(m, M));
        const float fo = mo == -INFINITY ? 0.0f : expf(__fsub_rn(mo, M));
        s = __fadd_rn(__fmul_rn(s, f), __fmul_rn(so, fo));
        acc.x = __fadd_rn(__fmul_rn(acc.x, f), __fmul_rn(ao.x, fo));
        acc.y = __fadd_rn(__fmul_rn(acc.y, f), __fmul_rn(ao.y, fo));
        acc.z = __fadd_rn(__fmul_rn(acc.z, f), __fmul_rn(ao.z, fo));
        acc.w = __fadd_rn(__fmul_rn(acc.w, f), __fmul_rn(ao.w, fo));
        m = M;
    }
    if (lane == 0) {
        red[w] = m;
        red[kAttnWaves + w] = s;
    }
    if (sub == 0) *reinterpret_cast<float4*>(&part[w][e4]) = acc;
    __syncthreads();
    if (w == 0) {
        float M = red[0];
#pragma unroll
        for (int q = 1; q < kAttnWaves; ++q) M = fmaxf(M, red[q]);
        float st = 0.0f, at = 0.0f;
#pragma unroll
        for (int q = 0; q < kAttnWaves; ++q) {
            const float f = red[q] == -INFINITY ? 0.0f : expf(__fsub_rn(red[q], M));
            st = __fadd_rn(st, __fmul_rn(red[kAttnWaves + q], f));
            at = __fadd_rn(at, __fmul_rn(part[q][lane], f));
        }
        attn_store(a, r, h, lane, __fdiv_rn(at, st));
    }
}

// The prompt pass's attention on the fp32 matrix cores: a wave takes 16
// consecutive rows of one head and walks their stream's positions in tiles
// of 16, so a tile of K and V is read once for all its rows (a workgroup per
// row read both again for every row, which bound it).
// v_mfma_f32_16x16x4_f32 throughout: products and sums in binary32.
//  * Scores transposed, S^T = K Q^T: lane (g = l/16, c = l%16) feeds K row c
//    and Q row c at dimensions 16 cc + 4 g + e (step (cc, e); the four lane
//    groups of a step supply its four dimensions, any order), and holds the
//    scores of row c at keys 4 g + v: its own row's mask, maximum and sum,
//    joined over g by two exchanges.
//  * P V: those scores' exponentials are the A operand as they stand (row c,
//    step v: key 4 g + v), V[4 g + v][4 c ..] the B operand, one 16-byte load
//    for four output tiles (tile dt, column c: dimension 4 c + dt), so lane
//    (g, c) ends with rows 4 g + v at dimensions 4 c .. 4 c + 3.
// Each row has its running max, sum and outputs (rescaled as its max grows;
// a tile in which a row sees no key leaves that row's as they are), so a
// row's result does not depend on the rows beside it.  The 16 rows may belong
// to any slots: one pass per distinct slot, the other rows' keys masked; the
// caller's rows are grouped by slot first (t3_group_rows).
// A masked key's weight is 0, and 0 times a V that is not finite would reach
// rows that do not see that key: tiles that some row does not see whole look
// for such values and, where one is found, add row by row with the unseen
// keys' V at 0, each row in the same order of adds.
// KS = 4: the workgroup's four waves take the same rows and every fourth
// pair of tiles, merged through LDS by the same rescaling in wave order
// (small calls); KS = 1: each wave its own rows.
// Measured per layer at 64 prompts of 129 to 383 rows (14975 in all), 16
// heads: 1051 -> 175 us (matrix cores busy 35% of its cycles, VALU 34%; ready
// waves that another is issued before, 47% of the waves' time); one prompt of 251
// rows 24.5 -> 9.4 us.  32 rows per wave (half the loads of K and V) measured 235,
// where this took 200: registers for two waves per SIMD, not three.
template <int KS>
__global__ __launch_bounds__(4 * kHeadDim) void t3_attn_tile(AttnArgs a, int n_rows,
                                                            int n_groups) {
    constexpr int kWaves = 4, KT = 2;  // KT tiles of 16 keys per iteration
    static_assert(KS == 1 || KS == kWaves, "every wave its own rows, or all the same");
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int g = lane >> 4, c = lane & 15;
    // grouped rows: a group's heads first, so that the empty groups come last
    const int h = a.rows ? blockIdx.x : blockIdx.y;
    const int wg = a.rows ? blockIdx.y : blockIdx.x;
    const int n = a.n_head * kHeadDim;
    const int group = KS == 1 ? wg * kWaves + w : wg;
    // this lane's row (n_rows: none)
    int row = 16 * group + c;
    if (a.rows) {
        const int at = group < n_groups ? a.rows[row] : -1;
        row = at < 0 ? n_rows : at;
    }
    // an empty group: whole workgroups, or whole waves where no barrier
    // follows (KS = 1)
    if (!__ballot(row < n_rows)) return;
    const int rc = min(row, n_rows - 1);
    const bool real = row < n_rows && a.act[rc] != 0;
    const int pos = a.positions[rc], slot = a.slots[rc];
    f4 q[4], o[4];
    {
        const float* const qr = a.qkv + (int64_t)rc * 3 * n + h * kHeadDim + 4 * g;
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) {
            q[cc] = *reinterpret_cast<const f4*>(qr + 16 * cc);
            o[cc] = f4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    float m = -INFINITY, s = 0.0f;
    bool todo = real;
    for (;;) {
        // the first row still to do names the pass's slot
        const uint64_t left = __ballot(todo);
        if (!left) break;
        const int cur = __builtin_amdgcn_readlane(slot, (int)__builtin_ctzll(left));
        // lim: the last position the row sees in this pass (-1: none); last
        // over the rows, least over the group's active rows
        const bool now = todo && slot == cur;
        todo = todo && !now;
        const int lim = now ? pos : -1;
        int last = lim, least = real ? lim : INT32_MAX;
#pragma unroll
        for (int x = 1; x < 16; x <<= 1) {
            last = max(last, __shfl_xor(last, x));
            least = min(least, __shfl_xor(least, x));
        }
        last = __builtin_amdgcn_readfirstlane(last);
        least = __builtin_amdgcn_readfirstlane(least);
        const int64_t base =
            (((int64_t)cur * a.n_layer + a.layer) * a.n_head + h) * a.n_ctx * kHeadDim;
        const float* const kc = a.kc + base;
        const float* const vc = a.vc + base;
        for (int j0 = KS == 1 ? 0 : 16 * KT * w; j0 <= last; j0 += 16 * KT * KS) {
            // keys past the last read the last one's row, at weight 0
            f4 kk[KT][4], vv[KT][4], p[KT];
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) {
                const float* const kr =
                    kc + (int64_t)min(j0 + 16 * kt + c, last) * kHeadDim + 4 * g;
#pragma unroll
                for (int cc = 0; cc < 4; ++cc)
                    kk[kt][cc] = *reinterpret_cast<const f4*>(kr + 16 * cc);
            }
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    vv[kt][v] = *reinterpret_cast<const f4*>(
                        vc + (int64_t)min(j0 + 16 * kt + 4 * g + v, last) * kHeadDim + 4 * c);
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) p[kt] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int cc = 0; cc < 4; ++cc)
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int kt = 0; kt < KT; ++kt)
                        p[kt] = mfma_f32(kk[kt][cc][e], q[cc][e], p[kt]);
            float bm = -INFINITY;
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    p[kt][v] = __fmul_rn(p[kt][v], a.scale);
                    if (j0 + 16 * kt + 4 * g + v <= lim) bm = fmaxf(bm, p[kt][v]);
                }
            bm = fmaxf(bm, __shfl_xor(bm, 16));
            bm = fmaxf(bm, __shfl_xor(bm, 32));
            if (__ballot(bm > m)) {
                const float nm = fmaxf(m, bm);
                const float f = m == -INFINITY ? 0.0f : expf(__fsub_rn(m, nm));
                s = __fmul_rn(s, f);
                m = nm;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const float fv = __shfl(f, 4 * g + v);  // row 4 g + v's
#pragma unroll
                    for (int dt = 0; dt < 4; ++dt) o[dt][v] = __fmul_rn(o[dt][v], fv);
                }
            }
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const bool seen = j0 + 16 * kt + 4 * g + v <= lim;
                    p[kt][v] = seen ? expf(__fsub_rn(p[kt][v], m)) : 0.0f;
                    s = __fadd_rn(s, p[kt][v]);
                }
            bool plain = true;
            if (j0 + 16 * KT - 1 > least) {
                float z = 0.0f;  // NaN once a value is not finite
#pragma unroll
                for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
#pragma unroll
                        for (int dt = 0; dt < 4; ++dt) z = __fmaf_rn(vv[kt][v][dt], 0.0f, z);
                plain = __ballot(z != z) == 0;
            }
            if (plain) {
#pragma unroll
                for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
#pragma unroll
                        for (int dt = 0; dt < 4; ++dt)
                            o[dt] = mfma_f32(p[kt][v], vv[kt][v][dt], o[dt]);
            } else {
#pragma unroll 1
                for (int i = 0; i < 16; ++i) {
                    const int li = __builtin_amdgcn_readlane(lim, i);
#pragma unroll
                    for (int dt = 0; dt < 4; ++dt) {
                        f4 add = o[dt];
#pragma unroll
                        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                            for (int v = 0; v < 4; ++v) {
                                const bool seen = j0 + 16 * kt + 4 * g + v <= li;
                                add = mfma_f32(p[kt][v], seen ? vv[kt][v][dt] : 0.0f, add);
                            }
#pragma unroll
                        for (int v = 0; v < 4; ++v)
                            if (4 * g + v == i) o[dt][v] = add[v];
                    }
                }
            }
        }
    }
    s = __fadd_rn(s, __shfl_xor(s, 16));  // the row's sum over its four lanes
    s = __fadd_rn(s, __shfl_xor(s, 32));
    if constexpr (KS == 1) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float sv = __shfl(s, 4 * g + v);
            const bool on = __shfl((int)real, 4 * g + v) != 0;
            f4 x;
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) x[dt] = on ? __fdiv_rn(o[dt][v], sv) : 0.0f;
            attn_store4(a, n_rows, __shfl(row, 4 * g + v), h, c, x);
        }
    } else {
        // wave w joins the four waves' rows 4 g + w
        __shared__ f4 os[KS][4][64];
        __shared__ float ms[KS][16], ss[KS][16];
#pragma unroll
        for (int v = 0; v < 4; ++v) os[w][v][lane] = f4{o[0][v], o[1][v], o[2][v], o[3][v]};
        if (g == 0) {
            ms[w][c] = m;
            ss[w][c] = s;
        }
        __syncthreads();
        const int i = 4 * g + w;
        float M = ms[0][i];
#pragma unroll
        for (int x = 1; x < KS; ++x) M = fmaxf(M, ms[x][i]);
        float st = 0.0f;
        f4 at = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int x = 0; x < KS; ++x) {
            const float f = ms[x][i] == -INFINITY ? 0.0f : expf(__fsub_rn(ms[x][i], M));
            st = __fadd_rn(st, __fmul_rn(ss[x][i], f));
            const f4 ov = os[x][w][lane];
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) at[dt] = __fadd_rn(at[dt], __fmul_rn(ov[dt], f));
        }
        const bool on = __shfl((int)real, i) != 0;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) at[dt] = on ? __fdiv_rn(at[dt], st) : 0.0f;
        attn_store4(a, n_rows, __shfl(row, i), h, c, at);
    }
}

template <int EPT>
hipError_t launch_norm_ept(const NormArgs& a, int n_rows, hipStream_t st) {
    hipLaunchKernelGGL(t3_norm<EPT>, dim3((unsigned)n_rows), dim3(kNormThreads), 0, st, a);
    return hipGetLastError();
}

// One 16-row group per wave, or four waves per group (KS = 4) while the
// groups would not give every SIMD (1024) a wave.  ms per prompt pass, KS = 4 /
// KS = 1: 1 x 251 rows 1.91 / 2.23, 1 x 700 3.77 / 4.29, 4 x 251 (1008 groups)
// 4.49 / 4.53, 64 x 24 (1536) 6.10 / 5.90, 16 x 251 14.48 / 14.43, 48 x 290
// 50.6 / 50.0.
// n_groups: those of a.rows, or all rows in order.
hipError_t launch_attn_tile(const AttnArgs& a, int n_rows, int n_groups, hipStream_t st) {
    const bool split = (int64_t)((n_rows + 15) / 16) * a.n_head < 1024;
    const unsigned wgs = (unsigned)(split ? n_groups : (n_groups + 3) / 4), heads = (unsigned)a.n_head;
    hipLaunchKernelGGL((split ? t3_attn_tile<4> : t3_attn_tile<1>),
                       a.rows ? dim3(heads, wgs) : dim3(wgs, heads), dim3(4 * kHeadDim), 0, st, a,
                       n_rows, n_groups);
    return hipGetLastError();
}

template <int NY>
hipError_t launch_norm_split(const NormArgs& a, int n_rows, hipStream_t st) {
    hipLaunchKernelGGL(t3_norm_split<NY>, dim3((unsigned)n_rows),
                       dim3((unsigned)((a.n_embd / 8 + 63) / 64 * 64)), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_norm(const NormArgs& a, int n_rows, hipStream_t st) {
    if (a.parts) {  // slabs: none (the embedding) or a power of two
        switch (a.y ? a.ny : 0) {
            case 0: return launch_norm_split<0>(a, n_rows, st);
            case 1: return launch_norm_split<1>(a, n_rows, st);
            case 2: return launch_norm_split<2>(a, n_rows, st);
            case 4: return launch_norm_split<4>(a, n_rows, st);
            case 8: return launch_norm_split<8>(a, n_rows, st);
            default: return hipErrorInvalidValue;
        }
    }
    switch (a.n_embd / kNormThreads) {
        case 1: return launch_norm_ept<1>(a, n_rows, st);
        case 2: return launch_norm_ept<2>(a, n_rows, st);
        case 3: return launch_norm_ept<3>(a, n_rows, st);
        case 4: return launch_norm_ept<4>(a, n_rows, st);
        case 6: return launch_norm_ept<6>(a, n_rows, st);
        case 8: return launch_norm_ept<8>(a, n_rows, st);
        case 12: return launch_norm_ept<12>(a, n_rows, st);
        case 16: return launch_norm_ept<16>(a, n_rows, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

bool t3_shape_ok(int32_t n_embd, int32_t n_head) {
    const int e = n_embd / kNormThreads;
    return n_head >= 1 && n_embd == n_head * kHeadDim && n_embd % kNormThreads == 0 &&
           (e == 1 || e == 2 || e == 3 || e == 4 || e == 6 || e == 8 || e == 12 || e == 16);
}

size_t t3_attn_lds(int32_t) { return 0; }  // one pass: no per-position LDS

// Decode steps whose grid of rows x heads is small run 16 waves per (row,
// head) instead of 4, so the few workgroups still spread each stream's
// positions over many waves (measured at one stream, 16 heads: 0.91 ->
// 0.86 ms per step against 4 waves with the positions split over 16
// workgroups and merged by a second kernel).
bool t3_attn_wide(int32_t n_rows, int32_t n_head) { return (int64_t)n_rows * n_head < 256; }

// Streams on the matrix cores, every product's input written split by its
// producer; fewer run the mat-vecs on plain rows.  us per step of the Turbo
// shape at position 256, mat-vecs / matrix cores: Q4_0 4 streams 1146 / 1012, 6
// 1381 / 1052, 8 1497 / 1050, 15 2128 / 1115; Q8_0 6 1406 / 1107.  3 streams,
// 1153 / 982, stay on the mat-vecs all the same: their activations stay fp32
// operands, and a stream's rows are bit for bit what they are beside one other
// or alone (the folded norms are checked against the separate ones there).
static bool t3_matrix(int32_t n_rows, int32_t n_embd) {
    return n_rows >= 4 || !head_uses_gemv(n_rows, false, n_embd);
}

// Bytes of one split buffer of the widest input (also where the mat-vecs'
// LDS cannot hold rows of 4 n_embd).
static size_t t3_split_bytes(int32_t n_rows, int32_t n_embd) {
    if (!t3_matrix(n_rows, n_embd) && head_uses_gemv(n_rows, false, 4 * n_embd)) return 0;
    return (split_bytes((n_rows + 15) / 16 * 16, 4 * n_embd) + 255) / 256 * 256;
}

// Bytes of the prompt pass's row groups (group_bound: at most n_rows of them).
static size_t t3_group_bytes(int32_t n_rows) { return ((size_t)n_rows * 64 + 255) / 256 * 256; }

// Workspace of a step: x, u, a [n_rows][n_embd], y [kMaxKSplit][n_rows][n_embd],
// qkv [n_rows][3 n_embd], f [n_rows][4 n_embd], act [n_rows], then two
// buffers of split activations for the matrix products (each for the widest
// input, 4 n_embd): the norms and the attention write the first, the mlp's
// c_fc the second (c_fc reads the first as it writes), then the prompt pass's
// row groups and, where the rows are many (head_uses_tiles), the largest matrix
// unpacked for its product.
size_t t3_workspace_bytes(int32_t n_rows, int32_t n_embd) {
    const size_t row = (size_t)n_rows * n_embd * 4;
    const size_t body = (3 + kMaxKSplit) * row + 3 * row + 4 * row +
                        ((size_t)n_rows * 4 + 255) / 256 * 256;
    return body + 2 * t3_split_bytes(n_rows, n_embd) + t3_group_bytes(n_rows) +
           max(tile_scratch_bytes(n_rows, 4 * n_embd, n_embd),
               tile_scratch_bytes(n_rows, n_embd, 4 * n_embd));
}

hipError_t launch_t3_step(const cbx_t3_model& m, int32_t n_rows, const int32_t* tokens,
                          const float* inputs, int32_t* positions, const int32_t* state,
                          const int32_t* slots, int32_t n_slots, const cbx_t3_cache& c,
                          float* hidden, void* ws, hipStream_t st) {
    // slots set: a prefill (rows of one stream may share a call: their k and v
    // are stored before the attention, and positions do not advance)
    const bool prefill = slots != nullptr;
    const int n = m.n_embd;
    const size_t row = (size_t)n_rows * n;
    float* x = static_cast<float*>(ws);
    float* u = x + row;
    float* att = u + row;
    float* y = att + row;
    float* qkv = y + kMaxKSplit * row;
    float* f = qkv + 3 * row;
    int32_t* act = reinterpret_cast<int32_t*>(f + 4 * row);
    const bool wide = !prefill && t3_attn_wide(n_rows, m.n_head);
    void* split = reinterpret_cast<char*>(act) + ((size_t)n_rows * 4 + 255) / 256 * 256;
    void* split2 = static_cast<char*>(split) + t3_split_bytes(n_rows, n);
    int32_t* const groups =
        reinterpret_cast<int32_t*>(static_cast<char*>(split2) + t3_split_bytes(n_rows, n));
    void* unpacked = reinterpret_cast<char*>(groups) + t3_group_bytes(n_rows);

    NormArgs na{};
    na.n_embd = n;
    na.eps = m.eps;
    na.x = x;
    na.emb = inputs ? nullptr : m.speech_emb;
    na.wpe = m.wpe;
    na.inputs = inputs;
    na.tokens = inputs ? nullptr : tokens;
    na.positions = positions;
    na.state = state;
    na.slots = slots;
    na.n_slots = n_slots;
    na.n_vocab = m.n_speech_vocab;
    na.n_pos = m.n_pos;
    na.n_ctx = c.n_ctx;
    na.act = act;
    na.g = m.layers[0].ln_1_g;
    na.b = m.layers[0].ln_1_b;
    na.out = u;
    // on the matrix cores every product's input is written split by its
    // producer (the norms, the attention, c_fc); else plain rows
    const bool mc = t3_matrix(n_rows, n);
    uint32_t* const sparts = static_cast<uint32_t*>(split);
    float* const sinv = reinterpret_cast<float*>(static_cast<char*>(split) +
                                                 split_inv_offset(16 * ((n_rows + 15) / 16), n));
    na.parts = mc ? sparts : nullptr;
    na.inv = sinv;
    hipError_t e = launch_norm(na, n_rows, st);
    if (e != hipSuccess) return e;

    AttnArgs aa{};
    aa.qkv = qkv;
    aa.kc = c.k;
    aa.vc = c.v;
    aa.n_layer = m.n_layer;
    aa.n_head = m.n_head;
    aa.n_ctx = c.n_ctx;
    aa.positions = positions;
    aa.act = act;
    aa.slots = slots;
    aa.out = att;
    aa.parts = mc ? sparts : nullptr;  // c_attn has read them by then
    aa.inv = sinv;
    aa.scale = 0.125f;  // 1 / sqrt(64)
    const size_t lds = t3_attn_lds(c.n_ctx);
    // the prompt pass's rows in groups of one slot each (one row or one slot
    // is grouped as it is)
    int n_groups = (n_rows + 15) / 16;
    if (prefill && n_rows > 1 && n_slots > 1) {
        n_groups = group_bound(n_rows, n_slots);
        aa.rows = groups;
        hipLaunchKernelGGL(t3_group_rows, dim3(1), dim3(kGroupThreads), 0, st, act, slots, n_rows,
                           n_groups, groups);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }

    const int kz_a = mc ? min(head_k_split(n_rows, n, n), kMaxKSplit) : 1;
    const int kz_f = mc || !head_uses_gemv(n_rows, false, 4 * n)
                         ? min(head_k_split(n_rows, n, 4 * n), kMaxKSplit) : 1;
    // one or two streams: the residual adds and norms between the layer's
    // products run inside the mat-vec that consumes them (c_fc, and the next
    // layer's c_attn), the residual rows alternating between x and y's
    // second slab (the mat-vec products take no K split)
    const bool fold = !mc && n_rows <= 2 && kz_a == 1 && kz_f == 1;
    float* xcur = x;
    float* const xalt = y + row;
    GemvNorm gn{};
    gn.y = y;
    gn.act = act;
    gn.eps = m.eps;
    // the products of rows already split, from `in`
    auto product = [&](const void* w, const float* b, float* out, int n_out, int n_in,
                       const void* in, int kz, bool gelu, void* out_split,
                       const KvOut& kv = KvOut{}) {
        return head_uses_tiles(n_rows, n_in) && kz == 1
                   ? launch_head_tiles(w, m.wtype, b, out, n_out, n_rows, n_out, n_in, in, unpacked,
                                       st, gelu, out_split, kv)
                   : launch_head_presplit(w, m.wtype, b, out, n_out, n_rows, n_out, n_in, in, st,
                                          kz, gelu, out_split, kv);
    };
    for (int l = 0; l < m.n_layer; ++l) {
        const cbx_t3_layer& L = m.layers[l];
        if (mc) {
            const KvOut kv = prefill ? KvOut{c.k, c.v, positions, slots, act, l, m.n_layer,
                                             m.n_head, c.n_ctx}
                                     : KvOut{};
            e = product(L.attn_w, L.attn_b, qkv, 3 * n, n, split, 1, false, nullptr, kv);
        } else if (fold && l > 0) {  // the previous layer's residual + this ln_1
            gn.x_in = xcur;
            gn.x_out = xcur = xcur == x ? xalt : x;
            gn.g = L.ln_1_g;
            gn.b = L.ln_1_b;
            e = launch_head_gemv_norm(L.attn_w, m.wtype, L.attn_b, gn, qkv, 3 * n, n_rows, 3 * n,
                                      n, st, false);
        } else {
            e = launch_head(L.attn_w, m.wtype, L.attn_b, u, nullptr, n, qkv, nullptr, 3 * n,
                            n_rows, 3 * n, n, split, st);
        }
        if (e != hipSuccess) return e;
        aa.layer = l;
        if (prefill) {
            if (!mc) {
                hipLaunchKernelGGL(t3_kv_append, dim3((unsigned)n_rows, (unsigned)m.n_head),
                                   dim3(kHeadDim), 0, st, aa);
                if ((e = hipGetLastError()) != hipSuccess) return e;
            }
            if ((e = launch_attn_tile(aa, n_rows, n_groups, st)) != hipSuccess) return e;
        } else if (wide) {
            hipLaunchKernelGGL((t3_attn<6, 16>), dim3((unsigned)n_rows, (unsigned)m.n_head),
                               dim3(16 * kHeadDim), lds, st, aa);
        } else {
            hipLaunchKernelGGL((t3_attn<6, 4>), dim3((unsigned)n_rows, (unsigned)m.n_head),
                               dim3(4 * kHeadDim), lds, st, aa);
        }
        if ((e = hipGetLastError()) != hipSuccess) return e;
        // the two products the residual adds take a K split when their grid
        // is narrow (the norm adds the slabs)
        e = mc ? product(L.attn_proj_w, L.attn_proj_b, y, n, n, split, kz_a, false, nullptr)
               : launch_head_k(L.attn_proj_w, m.wtype, L.attn_proj_b, att, nullptr, n, y, nullptr,
                               n, n_rows, n, n, split, st, kz_a, false);
        if (e != hipSuccess) return e;
        NormArgs nb{};
        nb.n_embd = n;
        nb.eps = m.eps;
        nb.x = xcur;
        nb.y = y;
        nb.ny = kz_a;
        nb.ystride = (int64_t)row;
        nb.act = act;
        nb.g = L.ln_2_g;
        nb.b = L.ln_2_b;
        nb.out = u;
        nb.parts = mc ? sparts : nullptr;
        nb.inv = sinv;
        // gelu applied as the mlp rows are stored
        if (fold) {  // the residual + ln_2 inside c_fc
            gn.x_in = xcur;
            gn.x_out = xcur = xcur == x ? xalt : x;
            gn.g = L.ln_2_g;
            gn.b = L.ln_2_b;
            e = launch_head_gemv_norm(L.fc_w, m.wtype, L.fc_b, gn, f, 4 * n, n_rows, 4 * n, n, st,
                                      true);
        } else {
            if ((e = launch_norm(nb, n_rows, st)) != hipSuccess) return e;
            e = mc ? product(L.fc_w, L.fc_b, f, 4 * n, n, split, 1, true, split2)
                   : launch_head_k(L.fc_w, m.wtype, L.fc_b, u, nullptr, n, f, nullptr, 4 * n,
                                   n_rows, 4 * n, n, split, st, 1, true);
        }
        if (e != hipSuccess) return e;
        e = mc ? product(L.fc_proj_w, L.fc_proj_b, y, n, 4 * n, split2, kz_f, false, nullptr)
               : launch_head_k(L.fc_proj_w, m.wtype, L.fc_proj_b, f, nullptr, 4 * n, y, nullptr, n,
                               n_rows, n, 4 * n, split, st, kz_f, false);
        if (e != hipSuccess) return e;
        // the residual, then the next layer's ln_1 or, after the last, ln_f
        // into `hidden` and the positions advanced
        const bool last = l + 1 == m.n_layer;
        if (fold && !last) continue;  // inside the next layer's c_attn
        NormArgs nc = nb;
        nc.x = xcur;
        nc.ny = kz_f;
        nc.g = last ? m.ln_f_g : m.layers[l + 1].ln_1_g;
        nc.b = last ? m.ln_f_b : m.layers[l + 1].ln_1_b;
        nc.out = last ? hidden : u;
        nc.parts = mc && !last ? sparts : nullptr;
        nc.positions = positions;
        nc.advance = last && !prefill ? 1 : 0;
        if ((e = launch_norm(nc, n_rows, st)) != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace cbx
