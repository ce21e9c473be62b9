// cbx_group.h -- the rows of a prompt pass in groups of 16 for its attention
// tiles (t3_attn_tile, cbx_t3.hip), whatever order the caller gave them in.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cbx {

// A tile walks the positions of one slot at a time for the rows of its group
// that are in it, so a group of 16 slots walks 16 times.  Rows are grouped by
// slot modulo kGroupSlots (LDS counters, whatever the caches hold: a group may
// mix slots that are equal in it, which the tile allows for), skipped rows
// together.
constexpr int kGroupSlots = 4096;
constexpr int kGroupThreads = 1024;

// Groups that n_rows rows in n_slots slots need at most: a part of one per slot
// (and one of skipped rows) beside the whole ones.
inline int group_bound(int n_rows, int n_slots) {
    const int slots = n_slots < kGroupSlots ? n_slots : kGroupSlots;
    const int64_t g = (int64_t)n_rows / 16 + slots + 1;
    return (int)(g < n_rows ? g : n_rows);
}

// rows[16 G + c], G < n_groups = group_bound(..): row c of group G, in the
// caller's order within a slot; -1: none.  One workgroup: rows counted by all
// of its waves, placed by one (64 rows at a time, each after the rows of its
// slot before it, looked up in LDS).  Once per call: 5 us at 251 rows, 12 at 3000,
// 43 at 14975 (with one wave to find the rows of a slot among its 64 too, 24 at
// 3000, 103 at 14975).  us per Q4_0 prompt pass of the Turbo shape
// with groups of consecutive rows / here: one row in each of 16 slots at position
// 1000 9041 / 1418, of 64 slots 9243 / 3232 (a workgroup per row and head: 1764,
// 3357); 64 streams of 200 rows by position 55690 / 26290, one after the other
// 25860 / 26070; one stream of 251 rows in one of 64 slots 1645 / 1671 (64 empty
// groups).
static __global__ __launch_bounds__(kGroupThreads) void t3_group_rows(const int32_t* act,
                                                                      const int32_t* slots,
                                                                      int n_rows, int n_groups,
                                                                      int32_t* rows) {
    constexpr int kPer = kGroupSlots / kGroupThreads, kWaves = kGroupThreads / 64;
    constexpr int kChunk = 16384, kNone = 8191;  // past the last row: no slot's 13 bits
    __shared__ int at[kGroupSlots + 1];  // a slot's rows, then the place of its next
    __shared__ int wave_sum[kWaves];
    // of the rows being placed, 64 at a time: the slot, the rows of it before
    // this one among the 64 and, with the first of them, how many there are
    __shared__ uint32_t unit[kChunk];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    for (int i = tid; i <= kGroupSlots; i += kGroupThreads) at[i] = 0;
    __syncthreads();
    // the chunk from row c0, eight rows of a thread in flight (a wave's 64 are
    // consecutive); the first chunk is counted last and so is there to be placed
    auto load = [&](int c0, bool count) {
        for (int i0 = tid; i0 < kChunk && c0 + i0 - tid < n_rows; i0 += 8 * kGroupThreads) {
            int a[8], s[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int r = min(c0 + i0 + u * kGroupThreads, n_rows - 1);
                a[u] = act[r];
                s[u] = slots[r];
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int i = i0 + u * kGroupThreads;
                if (c0 + i - lane >= n_rows) break;  // the whole wave's
                const int b = c0 + i >= n_rows ? kNone : a[u] ? s[u] & (kGroupSlots - 1) : kGroupSlots;
                uint64_t same = ~0ull;  // the lanes of this lane's slot
#pragma unroll
                for (int bit = 0; bit <= 12; ++bit) {
                    const uint64_t on = __ballot((b >> bit) & 1);
                    same &= (b >> bit) & 1 ? on : ~on;
                }
                const uint32_t rank = __popcll(same & ((1ull << lane) - 1));
                unit[i] = (uint32_t)b | rank << 13 | (rank ? 0u : (uint32_t)__popcll(same) << 19);
                if (count && b != kNone) atomicAdd(&at[b], 1);
            }
        }
    };
    for (int c0 = (n_rows - 1) / kChunk * kChunk; c0 >= 0; c0 -= kChunk) load(c0, true);
    __syncthreads();
    // thread t: slots kPer t .. (the last thread the skipped rows too); the
    // places before its first from a scan over the threads
    const int own = tid == kGroupThreads - 1 ? kPer + 1 : kPer;
    int n[kPer + 1], sum = 0;
#pragma unroll
    for (int i = 0; i <= kPer; ++i) {
        n[i] = i < own ? at[kPer * tid + i] : 0;
        sum += (n[i] + 15) / 16 * 16;
    }
    int before = sum;
    for (int o = 1; o < 64; o <<= 1) {
        const int x = __shfl_up(before, o);
        if (lane >= o) before += x;
    }
    if (lane == 63) wave_sum[w] = before;
    __syncthreads();
    int total = 0;
    for (int i = 0; i < kWaves; ++i) {
        if (i < w) before += wave_sum[i];
        total += wave_sum[i];
    }
    before -= sum;
#pragma unroll
    for (int i = 0; i <= kPer; ++i) {
        if (i < own) at[kPer * tid + i] = before;
        const int next = before + (n[i] + 15) / 16 * 16;
        for (int p = before + n[i]; p < next; ++p) rows[p] = -1;
        before = next;
    }
    for (int p = total + tid; p < 16 * n_groups; p += kGroupThreads) rows[p] = -1;
    for (int c0 = 0; c0 < n_rows; c0 += kChunk) {
        const int here = min(kChunk, n_rows - c0);
        __syncthreads();  // the scan, or the chunk before, done
        if (c0 > 0) {
            load(c0, false);
            __syncthreads();
        }
        if (w > 0) continue;
        uint32_t x = unit[lane];
        for (int i0 = 0; i0 < here; i0 += 64) {
            const uint32_t next = unit[min(i0 + 64, kChunk - 64) + lane];
            const bool in = i0 + lane < here;
            const int s = x & 8191, place = in ? at[s] : 0;
            // every lane has read its place before the first of a slot moves it
            // on, and that is seen by the next 64
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
            __builtin_amdgcn_wave_barrier();
            if (in) rows[place + (x >> 13 & 63)] = c0 + i0 + lane;
            if (in && x >> 19) at[s] = place + (x >> 19);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
            __builtin_amdgcn_wave_barrier();
            x = next;
        }
    }
}

}  // namespace cbx
