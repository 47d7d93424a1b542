// Float32 products on the bf16 matrix cores through an exact three-way split of each operand.
//
// A float32 value is the sum of three bf16 values, x = h + m + l with h = bf16(x), m = bf16(x - h),
// l = bf16(x - h - m): 24 significand bits in three times 8, each remainder exact.  A product is
// then six bf16 products accumulated in float32 (v_mfma_f32_32x32x16_bf16, 16 times the rate of
// v_mfma_f32_32x32x2_f32),
//     x y = xl yh + xh yl + xm ym + xm yh + xh ym + xh yh
// (the splitting of G. Henry, P. T. P. Tang and A. Heinecke, "Leveraging the bfloat16 Artificial
// Intelligence Datatype For Higher-Precision Computations", ARITH 2019), the three dropped ones at most
// 2^-24 of |x y| together (|xm| <= 2^-8, |xl| <= 2^-17 of |x|'s power of two), 2^-27 root mean square.  The sums round less often than the float32 MFMA's
// (every 16 terms and part instead of every 2): measured on random 32 x 32 tiles against float64,
// root mean square error relative to the result's, float32 MFMA / this: depth 16 7.3e-8 / 3.4e-8,
// 64 1.44e-7 / 1.09e-7, 128 2.0e-7 / 1.6e-7, 1024 5.8e-7 / 4.8e-7, 4096 1.15e-6 / 1.00e-6 (normal
// operands; positive ones alike).
//
// What the split costs is VALU work, 5.5 instructions per value, so operands are split once where
// they are staged (tiles on their way into LDS, queries on their way into registers) and only the
// probabilities in the loop; bf16 MFMAs, unlike float32 ones, overlap VALU work.
//
// Small values: the parts of |x| >= 2^-110 are bf16 numbers (subnormal ones, which the MFMA does not
// flush: V scaled by 2^-110 leaves the output's relative error where it was).  Below, a part loses what
// lies under 2^-133, at most 2^-134 of absolute error per element (V scaled by 2^-116: relative error
// 2.4e-6, where the float32 MFMA has 4e-7).
//
// An infinite operand, or a finite one that bf16 rounds to infinity, has NaN remainders, so every
// result it reaches is NaN where float32 might be infinite or finite: kernels test their results and
// redo rows that are not finite in plain float32 arithmetic.  A NaN operand alone makes NaN what float32
// makes NaN: the forward and dc_bmm look for operands of the first kind and keep their results where
// there is none.  (The backward redoes its tile: the probabilities' range is not known.  NaN in one dO
// row of every head, causal B8 H12 L1024 D64: 13.4 ms against 0.23.)
#pragma once

#include <utility>

#include "common.hpp"
#include "tile_bf16.hpp"

namespace dc {
namespace {

struct X3 {
    bf16x8 h, m, l;
};

// x0, x1 split: the packed parts.
DEVI void split3_pair(float x0, float x1, uint32_t &h, uint32_t &m, uint32_t &l) {
    h = cvt_pk_bf16(x0, x1);
    const float r0 = x0 - __uint_as_float(h << 16), r1 = x1 - __uint_as_float(h & 0xffff0000u);
    m = cvt_pk_bf16(r0, r1);
    l = cvt_pk_bf16(r0 - __uint_as_float(m << 16), r1 - __uint_as_float(m & 0xffff0000u));
}
// The same split in three steps, for loops that place them between MFMAs: x -> h, r -> m, r -> l.
struct SplitPair {
    float x0, x1;         // the values, then the remainders
    uint32_t h, m, l;
    DEVI void step(int i) {  // i = 0, 1, 2 in turn
        if (i == 0) {
            h = cvt_pk_bf16(x0, x1);
        } else if (i == 1) {
            x0 -= __uint_as_float(h << 16), x1 -= __uint_as_float(h & 0xffff0000u);
            m = cvt_pk_bf16(x0, x1);
        } else {
            l = cvt_pk_bf16(x0 - __uint_as_float(m << 16), x1 - __uint_as_float(m & 0xffff0000u));
        }
    }
};
// Calls part(0 .. PARTS - 1) in order, spread evenly behind the NM MFMAs mfma(0 .. NM - 1).  The
// scheduler is held to this order: left to itself it issues a run of MFMAs and then the VALU work,
// and since a wave issues in order, neither then hides the other.
// (A fold and not a loop: every index is a constant from the start, so arrays stay in registers.)
template <int Q0, int... Q, typename P>
DEVI void run_parts(P &part, std::integer_sequence<int, Q...>) {
    (part(Q0 + Q), ...);
}
template <int NM, int PARTS, int... I, typename M, typename P>
DEVI void interleave_all(M &mfma, P &part, std::integer_sequence<int, I...>) {
    ((mfma(I),
      run_parts<I * PARTS / NM>(part, std::make_integer_sequence<int, (I + 1) * PARTS / NM - I * PARTS / NM>{}),
      __builtin_amdgcn_sched_barrier(0)),
     ...);
}
template <int NM, int PARTS, typename M, typename P>
DEVI void interleave(M mfma, P part) {
    interleave_all<NM, PARTS>(mfma, part, std::make_integer_sequence<int, NM>{});
}
// use(0, load(0)) .. use(N - 1, load(N - 1)), each load issued before the use ahead of its own (the
// compiler would issue it right before its MFMAs and expose the LDS latency every time).
template <int... I, typename L, typename U>
DEVI void pipelined_all(L &load, U &use, std::integer_sequence<int, I...>) {
    constexpr int N = sizeof...(I);
    X3 f[2] = {load(0), {}};
    ((f[(I + 1) & 1] = I + 1 < N ? load(I + 1 < N ? I + 1 : I) : f[(I + 1) & 1], __builtin_amdgcn_sched_barrier(0),
      use(I, f[I & 1]), __builtin_amdgcn_sched_barrier(0)),
     ...);
}
template <int N, typename L, typename U>
DEVI void pipelined(L load, U use) {
    pipelined_all(load, use, std::make_integer_sequence<int, N>{});
}
template <typename V>
DEVI X3 split3(const V &x, int at) {  // x[at .. at + 7]
    u32x4 h, m, l;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        uint32_t a, b, c;
        split3_pair(x[at + 2 * w], x[at + 2 * w + 1], a, b, c);
        h[w] = a, m[w] = b, l[w] = c;
    }
    return {__builtin_bit_cast(bf16x8, h), __builtin_bit_cast(bf16x8, m), __builtin_bit_cast(bf16x8, l)};
}

// c + a b, smallest products first; mfma_x3_small leaves out the largest, h h.
DEVI f32x16 mfma_x3_small(const X3 &a, const X3 &b, f32x16 c) {
    c = mfma_bf16(a.l, b.h, c);
    c = mfma_bf16(a.h, b.l, c);
    c = mfma_bf16(a.m, b.m, c);
    c = mfma_bf16(a.m, b.h, c);
    return mfma_bf16(a.h, b.m, c);
}
// Product i = 0 .. 5 of mfma_x3.
DEVI f32x16 mfma_x3_part(const X3 &a, const X3 &b, f32x16 c, int i) {
    return i == 0 ? mfma_bf16(a.l, b.h, c) : i == 1 ? mfma_bf16(a.h, b.l, c) : i == 2 ? mfma_bf16(a.m, b.m, c)
         : i == 3 ? mfma_bf16(a.m, b.h, c) : i == 4 ? mfma_bf16(a.h, b.m, c) : mfma_bf16(a.h, b.h, c);
}
DEVI f32x16 mfma_x3(const X3 &a, const X3 &b, f32x16 c) { return mfma_bf16(a.h, b.h, mfma_x3_small(a, b, c)); }

// The same products in the same order with the operands' roles exchanged (a and b swapped): where
// the backward forms the forward's scores with queries as rows.
DEVI f32x16 mfma_x3_small_ba(const X3 &b, const X3 &a, f32x16 c) {
    c = mfma_bf16(b.h, a.l, c);
    c = mfma_bf16(b.l, a.h, c);
    c = mfma_bf16(b.m, a.m, c);
    c = mfma_bf16(b.h, a.m, c);
    return mfma_bf16(b.m, a.h, c);
}

// Product i = 0 .. 5, the sixth being h h.
DEVI f32x16 mfma_x3_part_ba(const X3 &b, const X3 &a, f32x16 c, int i) {
    return i == 0 ? mfma_bf16(b.h, a.l, c) : i == 1 ? mfma_bf16(b.l, a.h, c) : i == 2 ? mfma_bf16(b.m, a.m, c)
         : i == 3 ? mfma_bf16(b.h, a.m, c) : i == 4 ? mfma_bf16(b.m, a.h, c) : mfma_bf16(b.h, a.h, c);
}

// A tile of R rows x D float32 values as three chunk-major bf16 planes (tile_bf16.hpp).
template <int R, int D>
struct X3Tile {
    u32x4 p[3][CMTile<R, D>::SLOTS];
};
template <int R, int D>
DEVI X3 row_frag_x3(const X3Tile<R, D> &t, uint32_t lanebase, int row0, int st) {
    return {row_frag<R, D>(t.p[0], lanebase, row0, st), row_frag<R, D>(t.p[1], lanebase, row0, st),
            row_frag<R, D>(t.p[2], lanebase, row0, st)};
}
template <int R, int D>
DEVI X3 tr_frag_x3(const X3Tile<R, D> &t, uint32_t lanebase, int row0, int dt) {
    return {tr_frag<R, D>(t.p[0], lanebase, row0, dt), tr_frag<R, D>(t.p[1], lanebase, row0, dt),
            tr_frag<R, D>(t.p[2], lanebase, row0, dt)};
}

// 8 consecutive dims of row `row` (d0 a multiple of 8; dims past E are 0).  VEC: E % 4 == 0 and
// 16-byte aligned rows.
template <bool VEC>
DEVI void load_chunk(f32x4 (&x)[2], const float *row, int d0, int E) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int d = d0 + 4 * i;
        if constexpr (VEC) {
            x[i] = d < E ? *reinterpret_cast<const f32x4 *>(row + d) : f32x4{0.f, 0.f, 0.f, 0.f};
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) x[i][e] = d + e < E ? row[d + e] : 0.f;
        }
    }
}
DEVI X3 split_chunk(const f32x4 (&x)[2]) {
    const float v[8] = {x[0][0], x[0][1], x[0][2], x[0][3], x[1][0], x[1][1], x[1][2], x[1][3]};
    return split3(v, 0);
}

// A tile on its way from memory to LDS: each of the THREADS threads carries N chunks (8 dims of a
// row) in registers from load() until store() splits them.  Eight consecutive threads hold two
// chunks of four rows: 64 contiguous bytes of each row from memory, and LDS writes to distinct
// banks.  Rows past the last one read the last (their scores are masked).
template <int R, int D, int THREADS, bool VEC>
struct X3Stage {
    static constexpr int C = D / 8, TOTAL = R * C, N = (TOTAL + THREADS - 1) / THREADS;
    static_assert(C % 2 == 0 && R % 4 == 0, "threads come in groups of two chunks by four rows");
    f32x4 x[N][2];

    DEVI static void place(int j, int tid, int &r, int &c) {
        const int i = tid + THREADS * j, grp = i >> 3;
        c = (i & 1) + 2 * (grp % (C / 2));
        r = ((i >> 1) & 3) + 4 * (grp / (C / 2));
    }
    DEVI void load(const float *base, int n0, int last, int E, int tid) {
#pragma unroll
        for (int j = 0; j < N; ++j) {
            int r, c;
            place(j, tid, r, c);
            if (TOTAL % THREADS != 0 && tid + THREADS * j >= TOTAL) return;
            load_chunk<VEC>(x[j], base + (int64_t)min(n0 + r, last) * E, 8 * c, E);
        }
    }
    DEVI static void put(X3Tile<R, D> &t, int j, int tid, u32x4 h, u32x4 m, u32x4 l) {
        int r, c;
        place(j, tid, r, c);
        if (TOTAL % THREADS != 0 && tid + THREADS * j >= TOTAL) return;
        const int slot = c * CMTile<R, D>::P + r;
        t.p[0][slot] = h, t.p[1][slot] = m, t.p[2][slot] = l;
    }
    DEVI void store(X3Tile<R, D> &t, int tid) const {
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const X3 s = split_chunk(x[j]);
            put(t, j, tid, __builtin_bit_cast(u32x4, s.h), __builtin_bit_cast(u32x4, s.m), __builtin_bit_cast(u32x4, s.l));
        }
    }
    // store() in parts for interleave(): PARTS calls of part(), each a third of a pair's split, the
    // LDS writes with a chunk's last.
    static constexpr int PARTS = 12 * N;
    struct Splitter {
        SplitPair pr;
        u32x4 h, m, l;
    };
    DEVI void part(Splitter &sp, X3Tile<R, D> &t, int tid, int q) const {
        const int j = q / 12, w = q / 3 % 4, i = q % 3;
        if (i == 0) sp.pr.x0 = x[j][w / 2][2 * (w % 2)], sp.pr.x1 = x[j][w / 2][2 * (w % 2) + 1];
        sp.pr.step(i);
        if (i == 2) sp.h[w] = sp.pr.h, sp.m[w] = sp.pr.m, sp.l[w] = sp.pr.l;
        if (q % 12 == 11) put(t, j, tid, sp.h, sp.m, sp.l);
    }
};

// NaN when any of the values is not finite, 0 otherwise.
DEVI float not_finite(const f32x16 &x) {
    float t = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) t = fmaf(x[r], 0.f, t);
    return t;
}

}  // namespace
}  // namespace dc
