// Masks that do not depend on the query (key padding), shared by the attention kernels.
//
// A kernel that reads a mask value per (query, key) from global memory waits for it behind the
// transfers of the next tile it has already issued (loads return in order), so nothing overlaps.
// Where the mask's query stride is 0 a tile of 64 keys has 64 values: each wave loads them a tile
// ahead, one per lane, and tiles whose keys are all masked are neither loaded nor visited.
// Against a value per (query, key) (bf16, B16 H12 L512 E64, lengths 152 to 512): forward 62.9 ->
// 38.3 us, dQ 58.8 -> 36.8, dK / dV 79.9 -> 60.0 (it visits every tile: a masked key's gradient
// still takes a NaN from dO, as the reference's 0 * NaN does).
#pragma once

#include "common.hpp"
#include "params.hpp"

namespace dc {
namespace {

// kNoMask; kFullMask: a mask value per (query, key); kRowMask: the mask does not depend on the query
// (key padding): one value per key.
enum MaskKind { kNoMask, kFullMask, kRowMask };

// The 64-key tiles of one mask row that hold a key whose mask is not -inf, in order.  One wave
// tests 64 tiles at a time (eight loads in flight) and keeps them as bits; every wave of a
// workgroup reads the same row and so walks the same tiles.
struct LiveTiles {
    const float *row;
    int S, ntiles, lane;
    int base = -64;     // tiles [base, base + 64) are in bits
    uint64_t bits = 0;

    DEVI LiveTiles(const float *row_, int S_, int ntiles_, int lane_) : row(row_), S(S_), ntiles(ntiles_), lane(lane_) {}

    // Lane l: the mask of key 64 t + l (-inf past S).
    DEVI float value(int t) const {
        const int key = 64 * t + lane;
        return t < ntiles && key < S ? row[key] : -INFINITY;
    }
    // The first such tile from t on; ntiles when there is none.
    DEVI int next(int t) {
        while (t < ntiles) {
            if (t >= base + 64) {
                base = t & ~63;
                bits = 0;
                for (int u0 = 0; u0 < 64 && base + u0 < ntiles; u0 += 8) {
                    float x[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) x[u] = value(base + u0 + u);
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        bits |= (uint64_t)(__ballot(x[u] != -INFINITY) != 0) << (u0 + u);
                }
            }
            const uint64_t rest = bits >> (t - base);
            if (rest) return t + __builtin_ctzll(rest);
            t = base + 64;
        }
        return ntiles;
    }
};

// Under a row mask a batch's heads all take as long as its live keys, so heads are dealt to the 8
// XCDs (blocks go to them round-robin) one by one: contiguous runs of heads would give one XCD the
// longest batches (B16 H12 L512, lengths 152 to 512).  The tiles of a head stay on one XCD, whose
// L2 holds its K and V.  Below 32 heads an XCD would get few or none: logical_block() then.
constexpr int kDealtHeads = 32;
inline int dealt_heads(int heads) { return heads < kDealtHeads ? heads : (heads + 7) / 8 * 8; }
// This block's (head, tile of the head); false for the blocks past the last head.
DEVI bool dealt_block(int heads, int tiles, int natural, int *head, int *tile) {
    if (heads < kDealtHeads) {
        *head = natural / tiles, *tile = natural % tiles;
        return true;
    }
    const int j = (int)blockIdx.x >> 3;
    *head = j / tiles * 8 + ((int)blockIdx.x & 7), *tile = j % tiles;
    return *head < heads;
}

}  // namespace
}  // namespace dc
