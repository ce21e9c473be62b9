// cbx_tile.hip -- the matrix products of many rows (the T3 prompt pass) on
// split activations (cbx_split.h): out[r][v] = sum_k W[v][k] x[r][k] + b[v],
// as head_mfma (cbx_head.hip) computes it (fp16 parts of the activations
// against F16 weights or the formats' integers, each block's product scaled
// by d 2^-s in fp32), in tiles large enough to be bound by the matrix cores.
//
// Two launches: head_unpack writes the weights once per product as the fp16
// operands (8 MB of 4096 x 1024, 6 us), so the many workgroups of a column
// neither shift nor convert them again (about 80 VALU instructions per block
// and wave); head_tile multiplies.
// Measured, 14975 rows of the Turbo shape (Q4_0, us, head_mfma -> here): c_fc with
// gelu and split outputs 697 -> 317, the layer's other three 1146 -> 590 (c_attn
// 234, the two c_proj 356), unpacking 25; the prompt pass of 64 x 129-383 rows
// 53.6 -> 31.6 ms.  The products run twice (hi, lo): 18.1 TFLOP, 830 TFLOP/s; a
// library product of 8192^3 in fp16 reaches 1174 on this card.
// What bounds it (counters, of a SIMD's cycles): the matrix cores are busy 36-40%,
// VALU instructions (theirs included) issue in 60% (c_proj) to 81% (c_fc); there
// are no bank conflicts outside the split outputs, and a wave spends a third of
// its time ready but not issued, a third waiting.  F16, without the weights'
// scales, issues 46-70%, its matrix cores are busy 41-47%, in 11-14% fewer cycles:
// the shared issue of scaled adds and matrix products bounds it, with the waits
// at the barrier of each block next.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "cbx_internal.h"
#include "cbx_split.h"
#include "cbx_weights.h"

namespace cbx {
namespace {

constexpr int kTileThreads = 256;
constexpr int kColPad = 256;  // unpacked outputs are padded to this many (zeros)

// ------------------------------------------------------------- the weights
// Lane (g, m) of fragment (C, kb): weights 8g .. 8g + 7 of block kb of output
// 16 C + m as 8 halves at 16 bytes ((C nball + kb) 64 + lane) (the
// matrix-core B operand), the block's scale at float (C nball + kb) 16 + m.
template <int WT>
__global__ __launch_bounds__(kTileThreads) void head_unpack(const void* W, int n_vocab, int nball,
                                                            u4v* wq, float* wd) {
    constexpr int BB = block_bytes<WT>();
    const int lane = threadIdx.x & 63, g = lane >> 4, m = lane & 15;
    const int kb = (int)blockIdx.y * (kTileThreads / 64) + (int)(threadIdx.x >> 6);
    const int C = (int)blockIdx.x, v = 16 * C + m;
    if (kb >= nball) return;
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<void*>(W), (short)0, (int)((int64_t)n_vocab * nball * BB), kBufWord3);
    // outputs past the table read zeros (byte offsets past the range)
    const uint32_t off = (uint32_t)((v < n_vocab ? v : n_vocab) * nball + kb) * (uint32_t)BB;
    auto word = [&](uint32_t at) {
        return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rw, at & ~3u, 0, 0);
    };
    const int64_t frag = (int64_t)C * nball + kb;
    if constexpr (WT == CBX_WTYPE_F16) {
        wq[frag * 64 + lane] = u4v{word(off + 16 * g), word(off + 16 * g + 4),
                                   word(off + 16 * g + 8), word(off + 16 * g + 12)};
    } else {
        const uint32_t qoff = off + (WT == CBX_WTYPE_Q5_0 ? 6 : 2) +
                              (WT == CBX_WTYPE_Q8_0 ? 8 * g : 8 * (g & 1));
        const uint32_t sh = 8u * (qoff & 3u);
        const uint32_t t0 = word(qoff), t1 = word(qoff + 4), t2 = word(qoff + 8);
        uint32_t q[5];
        q[0] = __builtin_amdgcn_alignbit(t1, t0, sh);
        q[1] = __builtin_amdgcn_alignbit(t2, t1, sh);
        if constexpr (WT == CBX_WTYPE_Q5_0) {
            const uint32_t h0 = word(off + 2), h1 = word(off + 6);
            q[2] = __builtin_amdgcn_alignbit(h1, h0, 8u * ((off + 2) & 3u));
        }
        q[4] = (word(off) >> (8u * (off & 3u))) & 0xffffu;
        float d;
        wq[frag * 64 + lane] = int_weights<WT>(q, g, d);
        if (g == 0) wd[frag * 16 + m] = d;
    }
}

// ------------------------------------------------------------- the products
struct TileArgs {
    const u4v* wq;         // head_unpack's operands and scales
    const float* wd;
    const float* bias;
    const uint32_t* parts;  // the rows, split
    const float* inv;
    int n_tiles;           // 16-row tiles
    int n_cg;              // workgroups along the outputs
    float* out;
    int64_t ld_out;
    int n_rows, n_vocab, n_embd;
    int gelu_out;
    uint32_t* out_parts;   // when set, the outputs go there instead, split
    float* out_inv;
    KvOut kv;              // a q|k|v product
};

// What a product's outputs become: fp32 rows, the next product's split rows,
// or q rows beside k and v in the caches.
enum class Out { kRows, kSplit, kQkv };

typedef int32_t i4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ i4 buffer(const void* p, int64_t bytes) {
    const uint64_t at = reinterpret_cast<uint64_t>(p);
    return i4{__builtin_amdgcn_readfirstlane((int)at), __builtin_amdgcn_readfirstlane((int)(at >> 32)) & 0xffff,
              __builtin_amdgcn_readfirstlane((int)bytes), kBufWord3};
}

// 16 bytes per lane from the buffer at voff + soff (4 bytes per lane from an
// address) straight into the LDS at byte lds + 16 lane (4 lane).  As asm: for
// the builtins the compiler waits for all of them before any LDS read, and
// the point is to keep later blocks' loads in flight.  No register is
// written; the waits are wait_stage's.
// (-Winline-asm: that m0 is a reserved register, which holds a load's LDS base
// and is set right before each; the compiler sets it anew for its own uses, told
// by the clobber.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma16(uint32_t lds, uint32_t voff, const i4& rsrc, uint32_t soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 ::"s"(lds), "v"(voff), "s"(rsrc), "s"(soff) : "memory", "m0");
}
__device__ __forceinline__ void dma4(uint32_t lds, uint32_t voff, const i4& rsrc, uint32_t soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds"
                 ::"s"(lds), "v"(voff), "s"(rsrc), "s"(soff) : "memory", "m0");
}
#pragma clang diagnostic pop
// This wave's loads but the last N done, its LDS reads too; then the others'.
template <int N>
__device__ __forceinline__ void wait_stage() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// A workgroup of 4 RW waves computes 16 NT RW rows x 64 NC outputs, wave
// (wr, wc) the wr-th 16 NT rows and the wc-th 16 NC outputs.  The operands of
// a block of 32 along n_embd go straight into the LDS, ST - 1 blocks ahead (a
// block one ahead through registers left a step waiting for the L2, about
// 2000 cycles, where its products take 512), one barrier per block.  Per block and
// 16 x 16 tile a wave issues 2 matrix products of 16 cycles and 8 VALU
// instructions (d 2^-s and the scaled add, 4 cycles each).
// Every kFold blocks the sums join the totals, so that no chain of adds is
// longer than head_mfma's (a chain over all of n_embd had up to 1.3x its
// error after 24 layers).
// DQ: quantized weights (their blocks' scales); F16 weights have none.
constexpr int kFold = 8;

template <bool DQ, int NT, int NC, int RW, int ST, Out OUT>
__global__ __launch_bounds__(256 * RW, 2) void head_tile(TileArgs a) {
    constexpr int W = 4 * RW, WT = NT * RW, WC = 4 * NC;  // waves, row and output tiles
    static_assert(2 * WT % W == 0 && WC % W == 0 && NC % 2 == 0, "whole loads per wave, whole output blocks");
    // one block: the parts, the weights, the scales of both
    constexpr int kScales = 16 * WT + (DQ ? 16 * WC : 0);
    constexpr int NA = 2 * WT / W, NB = WC / W, NS = (kScales + 64 * W - 1) / (64 * W);
    constexpr int kB = 2048 * WT, kS = kB + 1024 * WC, kStage = kS + 256 * W * NS;
    __shared__ __align__(16) char lds[ST * kStage];
    const uint32_t base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, m = lane & 15, wr = wave >> 2, wc = wave & 3;
    // workgroups in order of their outputs, then rows; XCD x (workgroups
    // x, x + 8, ...) takes a contiguous run of that order, so its L2 holds
    // few row groups
    const int nwg = (int)gridDim.x, per = nwg / 8, extra = nwg % 8;
    const int xcd = (int)blockIdx.x % 8, at = (int)blockIdx.x / 8;
    const int wg = xcd * per + min(xcd, extra) + at;
    const int T0 = wg / a.n_cg * WT, C00 = wg % a.n_cg * WC, C0 = C00 + wc * NC;
    const int nball = a.n_embd / 32;
    const int nt = min(WT, a.n_tiles - T0);  // row tiles past the last read the last's
    const i4 ra = buffer(a.parts + (int64_t)T0 * nball * 512, (int64_t)nt * nball * 2048);
    const i4 rs = buffer(a.inv + (int64_t)T0 * nball * 16, (int64_t)nt * nball * 64);
    const i4 rb = buffer(a.wq + (int64_t)C00 * nball * 64, (int64_t)WC * nball * 1024);
    const i4 rd = buffer(DQ ? a.wd + (int64_t)C00 * nball * 16 : nullptr, DQ ? (int64_t)WC * nball * 64 : 0);
    // this lane's offsets: operand W j + wave of the parts (row tile half
    // that, hi or lo) and of the weights; scale 64 (W j + wave) + lane, the
    // rows' first (those past the last are loaded again, and not read)
    uint32_t aoff[NA], boff[NB], soff[NS];
#pragma unroll
    for (int j = 0; j < NA; ++j) {
        const int f = W * j + wave;
        aoff[j] = (uint32_t)(min(f >> 1, nt - 1) * nball * 2048 + (f & 1) * 1024 + lane * 16);
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) boff[j] = (uint32_t)((W * j + wave) * nball * 1024 + lane * 16);
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        const int s = 64 * (W * j + wave) + lane;
        const int tile = s < 16 * WT ? min(s >> 4, nt - 1) : min((s >> 4) - WT, WC - 1);
        soff[j] = (uint32_t)(tile * nball * 64 + m * 4);
    }
    auto load = [&](int kb, int st) {
        const uint32_t to = base + (uint32_t)(st * kStage);
#pragma unroll
        for (int j = 0; j < NA; ++j) dma16(to + 1024 * (W * j + wave), aoff[j], ra, kb * 2048);
#pragma unroll
        for (int j = 0; j < NB; ++j) dma16(to + kB + 1024 * (W * j + wave), boff[j], rb, kb * 1024);
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            static_assert(16 * WT % 64 == 0, "a wave loads the scales of rows or of weights");
            const bool rows = !DQ || 64 * (W * j + wave) < 16 * WT;
            dma4(to + kS + 256 * (W * j + wave), soff[j], rows ? rs : rd, kb * 64);
        }
    };
    f4 acc[NT][NC], tot[NT][NC];
    const f4 z = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[t][c] = tot[t][c] = z;
#pragma unroll
    for (int st = 0; st < ST - 1; ++st) load(min(st, nball - 1), st);
    int cur = 0;
#pragma unroll 1
    for (int k0 = 0; k0 < nball; k0 += kFold) {
#pragma unroll 1
        for (int kb = k0; kb < k0 + kFold; ++kb) {
            // block kb is there for every wave, and every wave has read block
            // kb - 1, whose place the next load takes
            wait_stage<(ST - 2) * (NA + NB + NS)>();
            load(min(kb + ST - 1, nball - 1), cur == 0 ? ST - 1 : cur - 1);
            const char* const from = lds + cur * kStage;
            const u4v* const as = reinterpret_cast<const u4v*>(from) + 128 * NT * wr + lane;
            const u4v* const bs = reinterpret_cast<const u4v*>(from + kB) + 64 * NC * wc + lane;
            const f4* const ss = reinterpret_cast<const f4*>(from + kS) + 4 * NT * wr + g;
            const float* const ds = reinterpret_cast<const float*>(from + kS) + 16 * WT + 16 * NC * wc + m;
            cur = cur == ST - 1 ? 0 : cur + 1;
            u4v b[NC];
            float d[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                b[c] = bs[64 * c];
                d[c] = DQ ? ds[16 * c] : 1.0f;
            }
            u4v hi[2], lo[2];
            f4 sc[2], p[2][NC];
            auto fetch = [&](int t) {
                hi[t & 1] = as[128 * t];
                lo[t & 1] = as[128 * t + 64];
            };
            auto add = [&](int t) {
#pragma unroll
                for (int c = 0; c < NC; ++c)
#pragma unroll
                    for (int i = 0; i < 4; ++i)  // d 2^-s: exact
                        acc[t][c][i] = __fmaf_rn(
                            p[t & 1][c][i], DQ ? __fmul_rn(d[c], sc[t & 1][i]) : sc[t & 1][i],
                            acc[t][c][i]);
            };
            // row tile by row tile: the matrix products of one beside the
            // scaled adds of the one before
            fetch(0);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if (t + 1 < NT) fetch(t + 1);
                sc[t & 1] = ss[4 * t];  // rows 4g .. 4g + 3
#pragma unroll
                for (int c = 0; c < NC; ++c) p[t & 1][c] = mfma_f16(lo[t & 1], b[c], z);
#pragma unroll
                for (int c = 0; c < NC; ++c) p[t & 1][c] = mfma_f16(hi[t & 1], b[c], p[t & 1][c]);
                if (t > 0) add(t - 1);
                __builtin_amdgcn_sched_barrier(0);
            }
            add(NT - 1);
        }
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    tot[t][c][i] = __fadd_rn(tot[t][c][i], acc[t][c][i]);
                    acc[t][c][i] = 0.0f;
                }
    }
    wait_stage<0>();  // the loads past the end too: the LDS is used again
    float bias[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int v = 16 * (C0 + c) + m;
        bias[c] = a.bias && v < a.n_vocab ? a.bias[v] : 0.0f;
    }
    // the stages (no wave reads them any more) turn split outputs into
    // operand order: 16 rows of 32 dwords (hi | lo << 16), padded, per wave
    constexpr int kTurn = 36;
    static_assert(W * 16 * kTurn * 4 <= (int)sizeof(lds), "the turned tiles fit");
    uint32_t* const turn = reinterpret_cast<uint32_t*>(lds) + wave * 16 * kTurn;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int T = wr * NT + t;  // in the workgroup
        float x[NC][4];
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                x[c][i] = __fadd_rn(tot[t][c][i], bias[c]);
                if (a.gelu_out) x[c][i] = t3_gelu_f(x[c][i]);
            }
        if constexpr (OUT == Out::kSplit) {  // n_vocab a multiple of 32: whole blocks in or out
            const int nb_out = a.n_vocab / 32;
#pragma unroll
            for (int c = 0; c < NC; c += 2) {
                const int blk = (C0 + c) / 2;
                const bool in = T < nt && blk < nb_out;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float mx = max16_dpp(fmaxf(fabsf(x[c][i]), fabsf(x[c + 1][i])));
                    float sc, sinv;
                    split_scale(mx, sc, sinv);
                    turn[(4 * g + i) * kTurn + m] = split_pair(__fmul_rn(x[c][i], sc));
                    turn[(4 * g + i) * kTurn + 16 + m] = split_pair(__fmul_rn(x[c + 1][i], sc));
                    if (in && m == 0)
                        a.out_inv[split_inv_index(T0 + T, 4 * g + i, nb_out, blk)] = sinv;
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
                __builtin_amdgcn_wave_barrier();
                // lane (g, m): row m, values 8g .. 8g + 7
                const u4v q0 = *reinterpret_cast<const u4v*>(turn + m * kTurn + 8 * g);
                const u4v q1 = *reinterpret_cast<const u4v*>(turn + m * kTurn + 8 * g + 4);
                u4v hi, lo;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t e = i < 2 ? q0[2 * i] : q1[2 * i - 4];
                    const uint32_t o = i < 2 ? q0[2 * i + 1] : q1[2 * i - 3];
                    hi[i] = __builtin_amdgcn_perm(o, e, 0x05040100u);
                    lo[i] = __builtin_amdgcn_perm(o, e, 0x07060302u);
                }
                if (in) {
                    u4v* const o = reinterpret_cast<u4v*>(a.out_parts) +
                                   ((int64_t)(T0 + T) * nb_out + blk) * 128 + lane;
                    o[0] = hi;
                    o[64] = lo;
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
                __builtin_amdgcn_wave_barrier();
            }
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int rr = 16 * (T0 + T) + 4 * g + i;
                if (rr >= a.n_rows) continue;
                float* const o = a.out + (int64_t)rr * a.ld_out;
                float* kvp = nullptr;
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    const int v = 16 * (C0 + c) + m;
                    if (OUT == Out::kQkv && 3 * 16 * (C0 + c) >= a.n_vocab) {
                        if (c % 2 == 0) kvp = v < a.n_vocab ? kv_place(a.kv, rr, v) : nullptr;
                        if (kvp) kvp[16 * (c % 2)] = x[c][i];
                    } else if (v < a.n_vocab) {
                        o[v] = x[c][i];
                    }
                }
            }
        }
    }
}

int padded_cols(int n_vocab) { return (n_vocab + kColPad - 1) / kColPad * kColPad; }

template <int WT>
void unpack(const void* W, int n_vocab, int nball, u4v* wq, float* wd, hipStream_t st) {
    hipLaunchKernelGGL(head_unpack<WT>,
                       dim3((unsigned)padded_cols(n_vocab) / 16, (unsigned)(nball + 3) / 4),
                       dim3(kTileThreads), 0, st, W, n_vocab, nball, wq, wd);
}

template <bool DQ, int NT, int NC, int RW, int ST>
hipError_t launch_tile(TileArgs a, hipStream_t st) {
    a.n_cg = (a.n_vocab + 64 * NC - 1) / (64 * NC);
    const dim3 grid((unsigned)((a.n_tiles + NT * RW - 1) / (NT * RW)) * (unsigned)a.n_cg);
    if (a.out_parts)
        hipLaunchKernelGGL((head_tile<DQ, NT, NC, RW, ST, Out::kSplit>), grid, dim3(256 * RW), 0, st, a);
    else if (a.kv.kc)
        hipLaunchKernelGGL((head_tile<DQ, NT, NC, RW, ST, Out::kQkv>), grid, dim3(256 * RW), 0, st, a);
    else
        hipLaunchKernelGGL((head_tile<DQ, NT, NC, RW, ST, Out::kRows>), grid, dim3(256 * RW), 0, st, a);
    return hipGetLastError();
}

// 128 x 128 outputs per workgroup of 8 waves (each 64 x 32: twice the products
// per operand read), or 64 x 128 (each 32 x 32) while the larger would leave
// CUs idle: fewer than 384 of them (1.5 per CU).  ms per Q4_0 prompt pass of
// the Turbo shape with the line at 256 / 384 / 512 / 800 workgroups, and with
// 64 x 128 alone: about 2500 rows 7.34 / 7.36 / 7.51 / 7.53 / 7.51, 4900 rows
// 12.19 / 11.99 / 12.00 / 11.99 / 12.82, 10560 rows 22.83 / 22.81 / 22.82 / 23.26 / 24.69.
template <bool DQ>
hipError_t launch_tiles(const TileArgs& a, hipStream_t st) {
    const int64_t large = (int64_t)((a.n_tiles + 7) / 8) * ((a.n_vocab + 127) / 128);
    return large >= 384 ? launch_tile<DQ, 4, 2, 2, 3>(a, st) : launch_tile<DQ, 2, 2, 2, 4>(a, st);
}

}  // namespace

size_t tile_scratch_bytes(int32_t n_rows, int32_t n_vocab, int32_t n_embd) {
    if (!head_uses_tiles(n_rows, n_embd)) return 0;
    const size_t cols = (size_t)padded_cols(n_vocab);
    return cols * n_embd * 2 + cols * (n_embd / 32) * 4;
}

// From 1024 rows (ms per Q4_0 prompt pass, tiles / head_mfma: about 450 rows 3.54 /
// 2.63, 900 4.28 / 4.32, 1400 4.80 / 5.10, 2850 7.81 / 10.39).
bool head_uses_tiles(int32_t n_rows, int32_t n_embd) {
    return n_rows >= 1024 && n_embd % (32 * kFold) == 0;
}

hipError_t launch_head_tiles(const void* W, int32_t wtype, const float* bias, float* out,
                             int64_t ld_out, int32_t n_rows, int32_t n_vocab, int32_t n_embd,
                             const void* split, void* scratch, hipStream_t st, bool gelu_out,
                             void* out_split, const KvOut& kv) {
    if (!split || !scratch || !head_uses_tiles(n_rows, n_embd) || (out_split && n_vocab % 32 != 0) ||
        (kv.kc && (out_split || gelu_out || n_vocab != 3 * 64 * kv.n_head)))
        return hipErrorInvalidValue;
    const int nball = n_embd / 32, n_tiles = (n_rows + 15) / 16;
    u4v* const wq = static_cast<u4v*>(scratch);
    float* const wd = reinterpret_cast<float*>(static_cast<char*>(scratch) +
                                               (size_t)padded_cols(n_vocab) * n_embd * 2);
    switch (wtype) {
        case CBX_WTYPE_F16: unpack<CBX_WTYPE_F16>(W, n_vocab, nball, wq, wd, st); break;
        case CBX_WTYPE_Q4_0: unpack<CBX_WTYPE_Q4_0>(W, n_vocab, nball, wq, wd, st); break;
        case CBX_WTYPE_Q5_0: unpack<CBX_WTYPE_Q5_0>(W, n_vocab, nball, wq, wd, st); break;
        case CBX_WTYPE_Q8_0: unpack<CBX_WTYPE_Q8_0>(W, n_vocab, nball, wq, wd, st); break;
        default: return hipErrorInvalidValue;
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    TileArgs a{};
    a.wq = wq;
    a.wd = wd;
    a.bias = bias;
    a.parts = static_cast<const uint32_t*>(split);
    a.inv = reinterpret_cast<const float*>(static_cast<const char*>(split) +
                                           split_inv_offset(16 * n_tiles, n_embd));
    a.n_tiles = n_tiles;
    a.out = out;
    a.ld_out = ld_out;
    a.n_rows = n_rows;
    a.n_vocab = n_vocab;
    a.n_embd = n_embd;
    a.gelu_out = gelu_out ? 1 : 0;
    a.out_parts = static_cast<uint32_t*>(out_split);
    a.out_inv = out_split ? reinterpret_cast<float*>(static_cast<char*>(out_split) +
                                                     split_inv_offset(16 * n_tiles, n_vocab))
                          : nullptr;
    a.kv = kv;
    return wtype == CBX_WTYPE_F16 ? launch_tiles<false>(a, st) : launch_tiles<true>(a, st);
}

}  // namespace cbx
