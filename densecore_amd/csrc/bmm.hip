// Float32 batched matrix product, C[b] = A[b] B[b], on the bf16 matrix cores (split products, x3.hpp).
//
// The reference registers one bmm kernel, (Cpu, Float32) (src/batched_matmul.rs:28-49), which runs
// PyTorch's bmm on the operands' strided storage (src/torch_blas.rs:404-449): A is (batch, m, k),
// B is (batch, k, n), each read through its own element strides (a transposed view is just other
// strides), and C is a fresh row-major (batch, m, n).  This is the device entry of that table: the
// math attention path's two products (q k^T, a transposed view of k, and weights v) and MHA's.
//
// Blocking (this kernel's own): a workgroup of 4 waves computes a BM x BN tile of one batch item
// (waves 2 x 2, each (BM/2) x (BN/2) as 32 x 32 MFMA tiles), over k in steps of 16, one MFMA's depth.
// A thread loads 8 elements of each operand along its contiguous dimension, splits them and writes
// them to LDS in chunks along that dimension (two buffers, one barrier per step, the next step's
// loads in flight): chunks along k are read as they are, chunks along m or n transposed
// (ds_read_b64_tr_b16), both giving a lane the same eight k.  Six MFMAs per 32 x 32 tile and step,
// smallest products first.  Bound: the MFMAs (24 per wave and step at 128 x 128) beside the splits
// (44 VALU instructions per operand and step); few k steps also by writing C.  On one MI355X, float32
// MFMAs before -> now: 32 items of 2048 x 256 x 2048 588 -> 444 us (155 TFLOP/s), of 2048 x 2048 x
// 256 606 -> 478, 4096^3 1139 -> 826; 256 items of 512 x 64 x 512 121 -> 104, of 512 x 512 x 64 125 ->
// 112 (268 MB of C).  Relative error against float64: depth 64 1.45e-7 -> 1.10e-7, 4096 1.15e-6 ->
// 1.00e-6 (the reference sums the products in k order).  The launcher also serves the attention path
// of head dims above 128 (wide.hip), which writes C through strides and can add A B into C.
#include "common.hpp"
#include "params.hpp"
#include "x3.hpp"

namespace dc {
namespace {

constexpr int kThreads = 256;
constexpr int BK = 16;  // one MFMA's depth

// How an operand's tile is loaded: CONTIG_K: 16-byte loads along k; CONTIG_MN: 16-byte loads along
// m (A) or n (B); SCALAR: one element at a time, any strides.  RAGGED: the two operands' loads are
// 4-byte aligned only and the last of a row may be cut short (rows of a length that is not a multiple of
// 4: loads of one element each took 256 items of 511 x 64 x 511 259 us and, A transposed, 151; now 114
// and 90).
enum Layout { CONTIG_K = 0, CONTIG_MN = 1, SCALAR = 2 };
typedef f32x4 f32x4_ragged __attribute__((aligned(4)));

// One operand's tile: R rows (m or n) by BK, as three chunk-major bf16 planes (x3.hpp), its chunks
// of 8 along the dimension it is loaded along.
template <int R, int L, bool RAGGED>
struct Operand {
    static constexpr bool ALONG_K = L != CONTIG_MN;
    typedef X3Tile<ALONG_K ? R : BK, ALONG_K ? BK : R> Tile;
    typedef CMTile<ALONG_K ? R : BK, ALONG_K ? BK : R> Shape;
    static constexpr int CHUNKS = R * BK / 8;  // at most one per thread
    static_assert(CHUNKS <= kThreads, "a thread stages one chunk");
    f32x4 x[2];

    // This thread's chunk (row or k index r of the tile, chunk c), and whether it has one.
    DEVI static bool place(int tid, int &r, int &c) {
        const int grp = tid >> 3;  // two chunks of four rows per eight threads (X3Stage)
        c = (tid & 1) + 2 * (grp % (Shape::C / 2));
        r = ((tid >> 1) & 3) + 4 * (grp / (Shape::C / 2));
        return CHUNKS == kThreads || tid < CHUNKS;
    }
    // Four elements from q on, `left` (at least one) of which exist.
    DEVI static void part(f32x4 &y, const float *q, int left) {
        if (!RAGGED) {
            y = *reinterpret_cast<const f32x4 *>(q);
        } else if (left >= 4) {
            y = *reinterpret_cast<const f32x4_ragged *>(q);
        } else {
#pragma unroll
            for (int e = 0; e < 3; ++e)
                if (e < left) y[e] = q[e];
        }
    }
    // From `p` (the batch item's base) with strides (s_r along the rows, s_k along k); rows past
    // `rows` and k past `kk` read zero.
    DEVI void load(const float *p, int64_t s_r, int64_t s_k, int r0, int rows, int k0, int kk, int tid) {
        int r, c;
        if (!place(tid, r, c)) return;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            x[h] = f32x4{0.f, 0.f, 0.f, 0.f};
            if constexpr (L == CONTIG_K) {
                const int k = k0 + 8 * c + 4 * h;
                if (r0 + r < rows && k < kk) part(x[h], p + (r0 + r) * s_r + k, kk - k);
            } else if constexpr (L == CONTIG_MN) {
                const int rr = r0 + 8 * c + 4 * h;
                if (rr < rows && k0 + r < kk) part(x[h], p + (k0 + r) * s_k + rr, rows - rr);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int k = k0 + 8 * c + 4 * h + e;
                    if (r0 + r < rows && k < kk) x[h][e] = p[(r0 + r) * s_r + k * s_k];
                }
            }
        }
    }
    DEVI void store(Tile &t, int tid) const {
        int r, c;
        if (!place(tid, r, c)) return;
        const X3 v = split_chunk(x);
        const int slot = c * Shape::P + r;
        t.p[0][slot] = __builtin_bit_cast(u32x4, v.h);
        t.p[1][slot] = __builtin_bit_cast(u32x4, v.m);
        t.p[2][slot] = __builtin_bit_cast(u32x4, v.l);
    }
    // The MFMA operand of rows row0 + (l % 32): k in the order {4g..4g+3, 8+4g..8+4g+3} (g = l / 32),
    // which is what a transposed read gives.
    DEVI static uint32_t lanebase(int lane) {
        if constexpr (ALONG_K) return (uint32_t)((lane & 31) * 16 + (lane >> 5) * 8);
        else return tr_lanebase<BK, R>(lane);
    }
    DEVI static bf16x8 plane(const u32x4 *t, uint32_t base, int row0) {
        if constexpr (ALONG_K) {
            const char *q = reinterpret_cast<const char *>(t) + base + row0 * 16;
            const uint2 lo = *reinterpret_cast<const uint2 *>(q), hi = *reinterpret_cast<const uint2 *>(q + Shape::CS);
            return __builtin_bit_cast(bf16x8, u32x4{lo.x, lo.y, hi.x, hi.y});
        } else {
            return tr_frag<BK, R>(t, base, 0, row0 / 32);
        }
    }
    DEVI static X3 frag(const Tile &t, uint32_t base, int row0) {
        return {plane(t.p[0], base, row0), plane(t.p[1], base, row0), plane(t.p[2], base, row0)};
    }
};

// Three workgroups per CU, two where the 128 x 128 tile reads an operand transposed (their registers).
constexpr int waves_per_simd(int BN, int LA, int LB) { return BN == 128 && (LA == CONTIG_MN || LB == CONTIG_MN) ? 2 : 3; }

template <int BM, int BN, int LA, int LB, bool RAGGED>
__global__ __launch_bounds__(kThreads)
__attribute__((amdgpu_waves_per_eu(waves_per_simd(BN, LA, LB), waves_per_simd(BN, LA, LB)))) void bmm_f32_kernel(BmmArgs g) {
    constexpr int TM = BM / 64, TN = BN / 64;  // 32 x 32 MFMA tiles per wave along m, n
    static_assert(TM >= 1 && TN >= 1, "a wave covers at least 32 x 32");
    typedef Operand<BM, LA, RAGGED> OpA;
    typedef Operand<BN, LB, RAGGED> OpB;
    __shared__ typename OpA::Tile ta[2];
    __shared__ typename OpB::Tile tb[2];
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, gh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave >> 1, wn = wave & 1;
    const int mt = (g.m + BM - 1) / BM, nt = (g.n + BN - 1) / BN, per = mt * nt;
    // The tiles of one batch item run on one XCD (workgroup w goes to XCD w % 8), so its A and B
    // panels are read from one L2.
    const int n = gridDim.x, bid = blockIdx.x;
    const int w = (n & 7) == 0 ? (bid & 7) * (n >> 3) + (bid >> 3) : bid;
    const int bt = w / per, r = w % per, m0 = (r / nt) * BM, n0 = (r % nt) * BN;
    const float *ap = g.a + (int64_t)bt * g.sab;
    const float *bp = g.b + (int64_t)bt * g.sbb;
    // Causal products: the largest query index among rows [r0, r1] of the block (rows across a
    // head boundary: L - 1).
    auto max_query = [&](int r0, int r1) {
        const int64_t j0 = (int64_t)g.causal_row0 + r0, j1 = (int64_t)g.causal_row0 + r1;
        return j0 / g.causal_L != j1 / g.causal_L ? g.causal_L - 1 : (int)(j1 % g.causal_L);
    };
    int kk = g.k;
    if (g.causal_mode == 1 && n0 > max_query(m0, min(m0 + BM, g.m) - 1)) return;  // no key visible
    if (g.causal_mode == 2) kk = min(kk, max_query(m0, min(m0 + BM, g.m) - 1) + 1);
    const int nk = (kk + BK - 1) / BK;
    // The first k tile at or after kt that contributes (mode 3: some row of it sees key m0).
    auto next_live = [&](int kt) {
        if (g.causal_mode == 3)
            while (kt < nk && max_query(kt * BK, min((kt + 1) * BK, g.k) - 1) < m0) ++kt;
        return kt;
    };

    OpA sa;
    OpB sb;
    const int first = next_live(0);
    int kt = first;
    // B's "rows" are its n columns: its row stride is the n stride, its k stride the k stride.
    auto load = [&](int t) {
        sa.load(ap, g.sam, g.sak, m0, g.m, t * BK, kk, tid);
        sb.load(bp, g.sbn, g.sbk, n0, g.n, t * BK, kk, tid);
    };
    load(kt);
    sa.store(ta[0], tid);
    sb.store(tb[0], tid);
    int next = next_live(kt + 1);
    if (next < nk) load(next);

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    const uint32_t abase = OpA::lanebase(lane), bbase = OpB::lanebase(lane);
    for (int buf = 0; kt < nk; buf ^= 1) {
        __syncthreads();  // tile kt is in LDS; everyone is done with the one before
        X3 fa[TM], fb[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) fa[i] = OpA::frag(ta[buf], abase, wm * (BM / 2) + 32 * i);
#pragma unroll
        for (int j = 0; j < TN; ++j) fb[j] = OpB::frag(tb[buf], bbase, wn * (BN / 2) + 32 * j);
#pragma unroll
        for (int t = 0; t < 6; ++t)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] = mfma_x3_part(fa[i], fb[j], acc[i][j], t);
        if (next < nk) {
            sa.store(ta[buf ^ 1], tid);
            sb.store(tb[buf ^ 1], tid);
        }
        kt = next;
        next = next_live(kt + 1);
        if (next < nk) load(next);
    }

    // Sums that are not finite again in plain float32: an infinite element may have met NaN
    // remainders (x3.hpp).  Where every element of the tile's operands is NaN or below 2^48 they are
    // final: no sum overflows, and NaN parts make the sums NaN that a NaN element makes NaN.  (Softmax
    // rows of fully masked queries are NaN and go through products: with a NaN row in
    // every tile, 256 items of 512 x 64 x 512, 159 us, redoing each tile 1583, without NaN 95.)
    float bad = 0.f;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) bad += not_finite(acc[i][j]);
    auto beyond = [&]() {
        float peak = 0.f;  // of what is not NaN
        for (int q = first; q < nk; q = next_live(q + 1)) {
            OpA ca[kThreads / 64];
            OpB cb[kThreads / 64];
#pragma unroll
            for (int u = 0; u < kThreads / 64; ++u) {  // this wave alone: every thread's chunks
                const int id = lane + 64 * u;
                ca[u].load(ap, g.sam, g.sak, m0, g.m, q * BK, kk, id);
                cb[u].load(bp, g.sbn, g.sbk, n0, g.n, q * BK, kk, id);
            }
#pragma unroll
            for (int u = 0; u < kThreads / 64; ++u)
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    if (64 * u < OpA::CHUNKS) peak = fmaxf(peak, fabsf(ca[u].x[i / 4][i % 4]));
                    if (64 * u < OpB::CHUNKS) peak = fmaxf(peak, fabsf(cb[u].x[i / 4][i % 4]));
                }
        }
        return __any(peak >= 0x1p48f);
    };
    if (__any(bad != 0.f) && beyond()) {
        for (int i = 0; i < TM; ++i)
            for (int j = 0; j < TN; ++j) {
                const int col = min(n0 + wn * (BN / 2) + 32 * j + lr, g.n - 1);
                f32x16 t;
#pragma unroll
                for (int e = 0; e < 16; ++e) t[e] = 0.f;
                for (int q = first; q < nk; q = next_live(q + 1))
                    for (int k = q * BK; k < min((q + 1) * BK, kk); ++k) {
                        const float b = bp[col * g.sbn + k * g.sbk];
#pragma unroll
                        for (int e = 0; e < 16; ++e) {
                            const int row = min(m0 + wm * (BM / 2) + 32 * i + acc_row(e, gh), g.m - 1);
                            t[e] = fmaf(ap[row * g.sam + k * g.sak], b, t[e]);
                        }
                    }
#pragma unroll
                for (int ii = 0; ii < TM; ++ii)
#pragma unroll
                    for (int jj = 0; jj < TN; ++jj)
                        if (ii == i && jj == j) acc[ii][jj] = t;
            }
    }

    float *cp = g.c + (int64_t)bt * g.scb;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int col = n0 + wn * (BN / 2) + 32 * j + lr;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int row = m0 + wm * (BM / 2) + 32 * i + acc_row(e, gh);
                if (row < g.m && col < g.n) {
                    float *dst = cp + (int64_t)row * g.scm + col;
                    *dst = g.acc ? *dst + acc[i][j][e] : acc[i][j][e];
                }
            }
        }
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// The load layout of an operand: along the dimension whose stride is 1 (`whole`: its extent and the
// other strides keep 16-byte loads whole and aligned).
int layout(const float *p, int64_t sb, int64_t s_r, int rows, int64_t s_k, int kk, bool &whole) {
    const bool along_k = s_k == 1, along_r = s_r == 1;
    whole = whole && aligned16(p) && sb % 4 == 0;
    if (along_k && (!along_r || kk > 1)) {
        whole = whole && kk % 4 == 0 && s_r % 4 == 0;
        return CONTIG_K;
    }
    if (along_r) {
        whole = whole && rows % 4 == 0 && s_k % 4 == 0;
        return CONTIG_MN;
    }
    return SCALAR;
}

template <int BM, int BN, int LA, int LB>
hipError_t launch_r(const BmmArgs &g, bool whole, dim3 grid, hipStream_t st) {
    if constexpr (LA != SCALAR && LB != SCALAR)
        if (whole) return launch(bmm_f32_kernel<BM, BN, LA, LB, false>, grid, dim3(kThreads), st, g);
    return launch(bmm_f32_kernel<BM, BN, LA, LB, true>, grid, dim3(kThreads), st, g);
}

template <int BM, int BN, int LA>
hipError_t launch_b(const BmmArgs &g, int lb, bool whole, dim3 grid, hipStream_t st) {
    if (lb == CONTIG_K) return launch_r<BM, BN, LA, CONTIG_K>(g, whole, grid, st);
    if (lb == CONTIG_MN) return launch_r<BM, BN, LA, CONTIG_MN>(g, whole, grid, st);
    return launch_r<BM, BN, LA, SCALAR>(g, whole, grid, st);
}

template <int BM, int BN>
hipError_t launch_t(const BmmArgs &g, hipStream_t st) {
    const int64_t tiles = (int64_t)((g.m + BM - 1) / BM) * ((g.n + BN - 1) / BN) * g.batch;
    const dim3 grid((unsigned)tiles);
    bool whole = true;
    const int la = layout(g.a, g.sab, g.sam, g.m, g.sak, g.k, whole), lb = layout(g.b, g.sbb, g.sbn, g.n, g.sbk, g.k, whole);
    if (la == CONTIG_K) return launch_b<BM, BN, CONTIG_K>(g, lb, whole, grid, st);
    if (la == CONTIG_MN) return launch_b<BM, BN, CONTIG_MN>(g, lb, whole, grid, st);
    return launch_b<BM, BN, SCALAR>(g, lb, whole, grid, st);
}

// Zeroes C when k == 0 (the reference returns zeros); C is (batch, m, n) through its strides.
__global__ __launch_bounds__(256) void bmm_zero_kernel(BmmArgs g) {
    const int64_t count = (int64_t)g.batch * g.m * g.n;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < count; i += (int64_t)gridDim.x * 256) {
        const int64_t bt = i / ((int64_t)g.m * g.n), r = i % ((int64_t)g.m * g.n);
        g.c[bt * g.scb + (r / g.n) * g.scm + r % g.n] = 0.f;
    }
}

}  // namespace

hipError_t launch_bmm(const BmmArgs &g, hipStream_t st) {
    if (g.batch == 0 || g.m == 0 || g.n == 0) return hipSuccess;
    if (g.k == 0) {
        if (g.acc) return hipSuccess;
        const int64_t count = (int64_t)g.batch * g.m * g.n;
        const int64_t blocks = (count + 255) / 256 < 65536 ? (count + 255) / 256 : 65536;
        return launch(bmm_zero_kernel, dim3((unsigned)blocks), dim3(256), st, g);
    }
    // 128 x 64 tiles when n is narrow (the weights-times-v product of attention, n = head dim).
    if (g.n <= 64) return launch_t<128, 64>(g, st);
    return launch_t<128, 128>(g, st);
}

}  // namespace dc
