// The float32 backward's tiles and schedules, shared by its float32 kernels (bwd_f32.hip) and its
// split-product kernels (bwd_x3.hip).
#pragma once

#include "common.hpp"
#include "params.hpp"

namespace dc {

// Stream-K schedule: the steps of all key tiles, in (batch * kv head, key tile, step) order, cut
// into `chunks` equal ranges, one per workgroup.  A key tile whose steps fall in more than one
// range is "split": its workgroups add their dK / dV into outputs the pre-kernel cleared.
struct StreamK {
    int64_t total;    // steps of all key tiles
    int64_t per_kvh;  // steps of one (batch, kv head)
    int chunks;       // a multiple of 8
};

// Head dims up to 64 with slots (a.dq_part): whole tiles or stream-K ranges over `grid`, one workgroup
// per CU.
hipError_t launch_bwd_x3(const BwdArgs &a, const StreamK &sk, dim3 grid, hipStream_t st);

namespace {

constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
constexpr int kBN = 32 * kWaves;  // keys per workgroup
constexpr int kBM = 32;           // queries per step

// Query steps of key tile kt (keys kt * kBN ..): (query head of the kv head, 32-query tile)
// pairs, query head outermost; causal skips the query tiles that end before the tile's first key
// (kBN is a multiple of kBM, so the first step starts at that key).
__host__ __device__ inline int tile_m_begin(bool causal, int kt) { return causal ? kt * kBN : 0; }
__host__ __device__ inline int tile_per_head(const AttnShape &s, int kt) {
    const int m_begin = tile_m_begin(s.causal, kt);
    return s.L > m_begin ? (s.L - m_begin + kBM - 1) / kBM : 0;
}
__host__ __device__ inline int tile_steps(const AttnShape &s, int kt) { return tile_per_head(s, kt) * s.repeat; }

// The dQ slots of the deterministic backward: key tile kt's slot holds, for every (batch, head),
// the query rows its steps cover, [slot_from(kt), L) (causal: from the tile's first key; else all
// rows).  slot_before(kt): rows of the slots of tiles 0 .. kt - 1, per (batch, head).
__host__ __device__ inline int slot_from(const AttnShape &s, int kt) {
    return s.causal ? (int)min((int64_t)kt * kBN, (int64_t)s.L) : 0;
}
__host__ __device__ inline int64_t slot_before(const AttnShape &s, int kt) {
    if (!s.causal) return (int64_t)kt * s.L;
    const int64_t j = min((int64_t)kt, ((int64_t)s.L + kBN - 1) / kBN);  // tiles starting before L
    return j * s.L - (int64_t)kBN * j * (j - 1) / 2;
}

// The range holding step p: the largest c with floor(c * total / chunks) <= p.
__host__ __device__ inline int64_t chunk_of(const StreamK &k, int64_t p) {
    return ((p + 1) * k.chunks - 1) / k.total;
}

// The thread index through an empty asm, which the compiler cannot see through.  A key tile's
// prologue (K / V loads) and epilogue (dK / dV stores) derive their lane addresses from such a
// copy: in the stream-K kernel, which runs key tiles in a loop, the compiler would otherwise hoist
// that address arithmetic out of the loop and hold it in registers across every step of every
// tile, and spill (the step loop's own addresses use the thread index directly).
DEVI int opaque_index(int tid) {
    asm volatile("" : "+v"(tid));
    return tid;
}

// Where a stream-K range's share of a key tile it cuts goes: slot 0 of the range for the tile it
// starts in, slot 1 for the tile it ends in (a range cuts at most these two); each slot holds a
// whole tile's dK (times scale) then dV.
DEVI float *kv_slot(const BwdArgs &a, int64_t range, int which) {
    return a.kv_part + (range * 2 + which) * 2 * (int64_t)kBN * a.s.E;
}

// One workgroup per range of the stream-K schedule, ranges dealt to the 8 XCDs in contiguous
// blocks (workgroup w runs on XCD w % 8), so the key tiles of one kv head, which read the same
// Q / dO, share an L2.  tile(bhk, kt, i0, i1, kdst, vdst, atomic) runs steps [i0, i1) of a key tile.
template <typename F>
DEVI void streamk_range(const BwdArgs &a, const StreamK &sk, F tile) {
    const int w = blockIdx.x;
    const int64_t c = (int64_t)(w & 7) * (sk.chunks >> 3) + (w >> 3);
    int64_t pos = c * sk.total / sk.chunks;
    const int64_t end = (c + 1) * sk.total / sk.chunks;
    const int nkt = (a.s.S + kBN - 1) / kBN;
    // The key tile and step of the first position (tiles without steps hold no position).
    int bhk = (int)(pos / sk.per_kvh), kt = 0;
    int64_t r = pos % sk.per_kvh;
    for (; kt < nkt; ++kt) {
        const int n = tile_steps(a.s, kt);
        if (r < n) break;
        r -= n;
    }
    int i = (int)r;
    bool first = true;
    while (pos < end) {
        const int n = tile_steps(a.s, kt);
        const int i1 = (int)min((int64_t)n, i + (end - pos));
        if (!first) __syncthreads();  // the previous tile's last readers of the shared area are done
        const bool whole = i == 0 && i1 == n;
        const int64_t row0 = ((int64_t)bhk * a.s.S + (int64_t)kt * kBN) * a.s.E;
        float *kd = static_cast<float *>(a.dk) + row0, *vd = static_cast<float *>(a.dv) + row0;
        if (!whole && a.kv_part) {
            kd = kv_slot(a, c, first ? 0 : 1);
            vd = kd + (int64_t)kBN * a.s.E;
        }
        tile(bhk, kt, i, i1, kd, vd, !whole && !a.kv_part);
        first = false;
        pos += i1 - i;
        i = 0;
        do {
            if (++kt == nkt) kt = 0, ++bhk;
        } while (pos < end && tile_steps(a.s, kt) == 0);
    }
}

}  // namespace
}  // namespace dc
