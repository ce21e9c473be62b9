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
// slot before it).  Once per call.  us per Q4_0 prompt pass of the Turbo shape
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
    __shared__ int at[kGroupSlots + 1];  // a slot's rows, then the place of its next
    __shared__ int wave_sum[kWaves];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    for (int i = tid; i <= kGroupSlots; i += kGroupThreads) at[i] = 0;
    __syncthreads();
    for (int r = tid; r < n_rows; r += kGroupThreads)
        atomicAdd(&at[act[r] ? slots[r] & (kGroupSlots - 1) : kGroupSlots], 1);
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
    __syncthreads();
    if (w > 0) return;
    auto slot_of = [&](int r) {
        return r >= n_rows ? -1 : act[r] ? slots[r] & (kGroupSlots - 1) : kGroupSlots;
    };
    int s = slot_of(lane);
    for (int r0 = 0; r0 < n_rows; r0 += 64) {
        const int r = r0 + lane, later = slot_of(r + 64);
        uint64_t same = __ballot(s >= 0);  // the lanes of this lane's slot
#pragma unroll
        for (int bit = 0; bit <= 12; ++bit) {
            const uint64_t on = __ballot((s >> bit) & 1);
            same &= (s >> bit) & 1 ? on : ~on;
        }
        if (s >= 0) {
            const int place = at[s], rank = __popcll(same & ((1ull << lane) - 1));
            rows[place + rank] = r;
            if (rank == 0) at[s] = place + __popcll(same);
        }
        s = later;
    }
}

}  // namespace cbx
