// Entries (token * 6 + slot) sorted by expert and cut into token blocks, for the
// kernels that give each block of a routed expert's tokens to workgroups of its
// own (grouped_tiles.h, prefill.hip).
#pragma once
#include "moe_common.h"

namespace fleet_moe {
namespace blocks {

constexpr int kXcds = 8;

struct Table {
    int32_t off[kRouted + 1];     // first sorted entry of an expert
    int32_t blk[kRouted + 1];     // first token block of an expert
};

// One workgroup of 1024 threads, n <= 1024 N entries, blocks of `tok` tokens. Ids
// outside [0, 64) are clamped; true where this thread saw one. An expert's entries
// come in no fixed order.
template <int N, class Ent>
__device__ __forceinline__ bool build(const int32_t* ids, int n, int tok, Table* tab, Ent* ent) {
    __shared__ int cnt[kRouted], at[kRouted];
    const int tid = threadIdx.x;
    if (tid < kRouted) cnt[tid] = 0;
    __syncthreads();
    int id[N];
    bool bad = false;
#pragma unroll
    for (int r = 0; r < N; ++r) {
        const int k = tid + 1024 * r;
        const int raw = k < n ? ids[k] : 0;
        id[r] = min(max(raw, 0), kRouted - 1);
        bad |= raw != id[r];
        if (k < n) atomicAdd(&cnt[id[r]], 1);
    }
    __syncthreads();
    if (tid < kLanes) {
        const int c = cnt[tid], b = (c + tok - 1) / tok;
        const int oi = wave_incl_scan(c), bi = wave_incl_scan(b);
        at[tid] = oi - c;
        tab->off[tid] = oi - c;
        tab->blk[tid] = bi - b;
        if (tid == kRouted - 1) {
            tab->off[kRouted] = oi;
            tab->blk[kRouted] = bi;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < N; ++r) {
        const int k = tid + 1024 * r;
        if (k < n) ent[atomicAdd(&at[id[r]], 1)] = (Ent)k;
    }
    return bad;
}

// Blocks of n entries at most (one partly filled block per selected expert),
// rounded up to whole rounds of the XCDs: the routed workgroups of a launch with
// `tiles` row tiles are `tiles` times as many.
__host__ constexpr int most(int n, int tok) {
    return ((n < kRouted ? n : kRouted) + n / tok + kXcds - 1) / kXcds * kXcds;
}

// The token block of routed workgroup `wg`: row tile `tile` of `tiles`, entries
// [first, first + m) of expert e. The workgroups of one XCD (wg % 8) take a block's
// row tiles in turn, so its token rows are fetched into one L2. False past the last
// block.
__device__ __forceinline__ bool of(const Table* tab, int wg, int tok, int tiles, int& e, int& tile,
                                   int& first, int& m) {
    const int lane = threadIdx.x & (kLanes - 1);
    const int local = wg / kXcds, b = wg % kXcds + kXcds * (local / tiles);
    tile = local % tiles;
    if (b >= tab->blk[kRouted]) return false;
    // the last expert that starts at or before b (one without tokens starts
    // where the next does)
    e = __builtin_popcountll(__ballot(tab->blk[lane] <= b)) - 1;
    first = tab->off[e] + tok * (b - tab->blk[e]);
    m = min(tok, tab->off[e + 1] - first);
    return true;
}

}  // namespace blocks
}  // namespace fleet_moe
