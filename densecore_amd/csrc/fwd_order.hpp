// Longest-first order of the heads under key-padding masks (float32 forwards): workgroups take
// heads in descending order of their live key tiles.
#pragma once

#include "common.hpp"
#include "params.hpp"

namespace dc {
namespace {

// The BN-key tiles of one mask row (S keys) that hold any key whose mask is not -inf, counted by
// one wave.  The loads of 8 x 64 keys are all issued before any is tested, so a row costs one
// memory latency per 512 keys instead of one per 64 (C3's step, order pass plus forward: 90.7 ->
// 90.4 us; the rest of the pass is its launch).
template <int BN>
DEVI int live_tiles(const float *row, int S, int lane) {
    constexpr int U = 8;
    int c = 0;
    for (int k0 = 0; k0 < S; k0 += 64 * U) {
        float x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int key = k0 + 64 * u + lane;
            x[u] = key < S ? row[key] : -INFINITY;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint64_t live = __ballot(x[u] != -INFINITY);
            if (BN == 64) c += live != 0;
            else c += ((live & 0xffffffffull) != 0) + ((live >> 32) != 0);
        }
    }
    return c;
}

// One wave per (b, h) of a query-independent mask: the number of BN-key tiles that hold any key
// whose mask is not -inf (the tiles the forward computes; the others it skips).
template <int BN>
__global__ __launch_bounds__(64) void rowmask_tiles_kernel(FwdArgs a) {
    static_assert(BN == 32 || BN == 64, "one or two tiles per wave-wide pass");
    const AttnShape &s = a.s;
    const int bh = blockIdx.x, lane = threadIdx.x;
    const float *row = s.mask + (int64_t)(bh / s.H) * s.msb + (int64_t)(bh % s.H) * s.msh;
    const int count = live_tiles<BN>(row, s.S, lane);
    if (lane == 0) a.tiles[bh] = count;
}

// One workgroup: a counting sort of the heads by live tiles, descending (ties in any order; the
// results do not depend on the order).
__global__ __launch_bounds__(1024) void rowmask_order_kernel(FwdArgs a, int ntiles) {
    __shared__ int start[kOrderMaxTiles + 1];
    const int BH = a.s.B * a.s.H, tid = threadIdx.x;
    for (int v = tid; v <= ntiles; v += 1024) start[v] = 0;
    __syncthreads();
    for (int i = tid; i < BH; i += 1024) atomicAdd(&start[a.tiles[i]], 1);
    __syncthreads();
    if (tid == 0) {  // start[v] = number of heads with more live tiles than v
        int run = 0;
        for (int v = ntiles; v >= 0; --v) {
            const int c = start[v];
            start[v] = run;
            run += c;
        }
    }
    __syncthreads();
    for (int i = tid; i < BH; i += 1024) a.order[atomicAdd(&start[a.tiles[i]], 1)] = i;
}

// Masks that depend on the batch and the key only (head and query strides 0: key padding, C3):
// one launch instead of the two above.  One workgroup counts the live tiles of each batch's mask
// row, a wave per row, and sorts the heads by their batch's count, descending.
template <int BN>
__global__ __launch_bounds__(1024) void rowmask_batch_order_kernel(FwdArgs a, int ntiles) {
    static_assert(BN == 32 || BN == 64, "one or two tiles per wave-wide pass");
    __shared__ int count[kOrderMaxBatch];
    __shared__ int start[kOrderMaxTiles + 1];
    const AttnShape &s = a.s;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int v = tid; v <= ntiles; v += 1024) start[v] = 0;
    for (int b = wave; b < s.B; b += 16) {
        const int c = live_tiles<BN>(s.mask + (int64_t)b * s.msb, s.S, lane);
        if (lane == 0) count[b] = c;
    }
    __syncthreads();
    const int BH = s.B * s.H;
    for (int i = tid; i < BH; i += 1024) atomicAdd(&start[count[i / s.H]], 1);
    __syncthreads();
    if (tid == 0) {  // start[v] = number of heads with more live tiles than v
        int run = 0;
        for (int v = ntiles; v >= 0; --v) {
            const int c = start[v];
            start[v] = run;
            run += c;
        }
    }
    __syncthreads();
    for (int i = tid; i < BH; i += 1024) a.order[atomicAdd(&start[count[i / s.H]], 1)] = i;
}

// Fills a.order (and a.tiles) for a mask that does not depend on the query, or clears a.order when
// the workspace does not hold it or the problem is too large for one workgroup to sort.
template <int BN>
hipError_t order_heads(FwdArgs &a, hipStream_t st) {
    const int ntiles = (a.s.S + BN - 1) / BN;
    if (!a.order || a.s.B * a.s.H > kOrderMaxHeads || ntiles > kOrderMaxTiles) {
        a.order = nullptr;
        return hipSuccess;
    }
    if (a.s.msh == 0 && a.s.B <= kOrderMaxBatch)
        return launch(rowmask_batch_order_kernel<BN>, dim3(1), dim3(1024), st, a, ntiles);
    return_if(launch(rowmask_tiles_kernel<BN>, dim3(a.s.B * a.s.H), dim3(64), st, a));
    return launch(rowmask_order_kernel, dim3(1), dim3(1024), st, a, ntiles);
}
// The grid for it: the query tiles of one head on one XCD, heads dealt to the 8 XCDs in a.order.
inline dim3 ordered_grid(const FwdArgs &a, int nqt) {
    return dim3(nqt * (a.order ? 8 * ((a.s.B * a.s.H + 7) / 8) : a.s.B * a.s.H));
}

}  // namespace
}  // namespace dc
