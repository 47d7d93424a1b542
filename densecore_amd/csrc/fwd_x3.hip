// Float32 attention forward on CDNA4 MFMA, its products on the bf16 matrix cores (x3.hpp), for
// head dims up to 127 (fwd_f32.hip chooses).
//
// Computes what DenseCore's torch_attention::forward computes (src/torch_attention.rs:143-284):
// out = softmax(scale * q k^T + mask, causal) v and lse = max + ln(sum), with fully masked
// rows giving out = 0 and lse = 0 (:223-226, :258-264).  The blocking is this kernel's own:
//
//   * one workgroup = 4 waves = 128 queries of one (batch, head); each wave owns 32 queries, split
//     into their three bf16 parts in registers as the B operand of S^T = K Q^T (keys x queries), so
//     every lane owns one query column and the online-softmax state (max, sum) is a scalar per lane;
//   * K and V tiles of 32 keys go through registers, where each thread splits its 8 dims of a row,
//     into double-buffered LDS planes (x3.hpp, tile_bf16.hpp);
//   * P = exp2(S * scale * log2 e - m) is split in registers: the S^T accumulator's rows are the
//     reduction index of O^T += V^T P^T, whose V operand is read transposed from LDS.
//
// Bound: the bf16 MFMAs, six per product; at 32 keys and D = 64 a wave issues 48 of them (1536
// matrix-pipe cycles) against about 300 VALU instructions, so the tile loop keeps both busy (see
// step() below).  Measured on one MI355X, with float32 MFMAs before -> now: causal B8 H12 L1024 D64
// 124.7 -> 79.5 us, B2 H12 L4096 D64 439 -> 273, full B6 H16 L1024 D64 198 -> 131 us (197 TFLOP/s;
// times six, 0.9 of the 1260 TFLOP/s a large bf16 matrix product reaches on this part), B4 H8 L1001
// D80 185 -> 68.  (float32 MFMAs reach 135 TFLOP/s here at best, and no VALU instruction runs beside
// one.)  Short rows (B64 H6 L256 D64: 41 -> 38) are held by each workgroup's first tiles: queries,
// two tiles of K and one of V from memory before the first MFMA.
//
// Head dims below the instantiated D are zero-padded on load; keys past S and (causal) keys
// past the query are -inf before the softmax.
#include <type_traits>

#include "common.hpp"
#include "fwd_order.hpp"
#include "fwd_split.hpp"
#include "params.hpp"
#include "row_mask.hpp"
#include "x3.hpp"

namespace dc {
namespace {

constexpr int kX3BN = 32;      // keys per tile
constexpr int kX3Waves = 4;    // 32 queries each
constexpr int kX3Threads = 64 * kX3Waves;
constexpr int kX3M = 32 * kX3Waves;

// At D = 128 the queries' parts and the output take 160 registers and the tiles 110 KB of LDS: one
// workgroup per CU, one wave per SIMD (two of single-buffered tiles: causal B2 H16 L2048 224 us
// against 193).
constexpr int fwd_waves_per_simd(int D) { return D <= 64 ? 2 : 1; }

template <int D, bool CAUSAL, int MASK, bool VEC, bool SPLIT>
__global__ __launch_bounds__(kX3Threads)
__attribute__((amdgpu_waves_per_eu(fwd_waves_per_simd(D), fwd_waves_per_simd(D)))) void fwd_x3_kernel(FwdArgs a) {
    constexpr int BN = kX3BN, KSTEP = D / 16, NDT = D / 32, DH = D / 2;
    constexpr bool LIST = MASK == kRowMask;
    __shared__ X3Tile<BN, D> sk[2], sv[2];
    __shared__ float mslot[LIST ? kX3Waves : 1][32];
    __shared__ uint16_t list[LIST ? kOrderMaxTiles : 1];  // row masks: the tiles with any visible key
    __shared__ uint8_t open_tile[LIST ? kOrderMaxTiles : 1];
    __shared__ int list_len;

    const AttnShape &s = a.s;
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: branches stay scalar
    const int BH = s.B * s.H;
    const int nqt = (s.L + kX3M - 1) / kX3M;
    const int bid = blockIdx.x;
    int qt = CAUSAL ? nqt - 1 - bid / BH : bid / BH;  // longest causal tiles first
    int bh = bid % BH;
    // Split key ranges: blocks run over (head, query tile longest first, piece), the pieces of a
    // head dealt to one XCD (blocks go to XCD bid % 8) so that its K/V stays in one L2.
    int piece = 0, npieces = 1;
    if constexpr (SPLIT) {
        const int n = gridDim.x, w = (n & 7) == 0 ? (bid & 7) * (n >> 3) + (bid >> 3) : bid;
        if (!split_block(s, kX3M, BN, a.split_chunk, w, &qt, &bh, &piece, &npieces)) return;
    }
    if (LIST && a.order) {
        // Heads in descending order of live key tiles, dealt to the 8 XCDs round-robin (blocks
        // go to XCD bid % 8), the query tiles of one head on one XCD: its K/V stays in one L2.
        const int x = bid & 7, slot = bid >> 3;
        const int r = 8 * (slot / nqt) + x;
        if (r >= BH) return;
        bh = a.order[r];
        qt = slot % nqt;
    }
    const int b = bh / s.H, h = bh % s.H, hk = h / s.repeat;
    const int q0 = qt * kX3M;
    const int wave_q0 = q0 + wave * 32, wave_last_q = wave_q0 + 31;
    const int qi = wave_q0 + lr;  // this lane's query
    const float *kb = static_cast<const float *>(a.k) + (int64_t)(b * s.Hkv + hk) * s.S * s.E;
    const float *vb = static_cast<const float *>(a.v) + (int64_t)(b * s.Hkv + hk) * s.S * s.E;
    const float *qrow = static_cast<const float *>(a.q) + ((int64_t)bh * s.L + min(qi, s.L - 1)) * s.E;
    const float *mrow = nullptr;
    if (MASK) mrow = s.mask + (int64_t)b * s.msb + (int64_t)h * s.msh + (int64_t)qi * s.msl;

    // This block's key tiles [t_begin, t_end): all of them, or its piece's (the query tile's
    // tiles cut into npieces near-equal ranges).
    const int kv_end = CAUSAL ? min(q0 + kX3M, s.S) : s.S;
    const int ntiles = (kv_end + BN - 1) / BN;
    const int t_begin = SPLIT ? piece * ntiles / npieces : 0;
    const int t_end = SPLIT ? (piece + 1) * ntiles / npieces : ntiles;

    // Row masks: the tiles with any visible key, listed, so that the others (padding) are neither
    // staged nor computed; kOrderMaxTiles tiles from w0 on at a time.
    int w0 = 0;
    int n = t_end - t_begin;
    auto list_tiles = [&]() {
        const int w1 = min(ntiles, w0 + kOrderMaxTiles);
        for (int seg = w0 / 2 + wave; 2 * seg < w1; seg += kX3Waves) {
            const int key = seg * 64 + lane;
            const uint64_t open = __ballot(key < s.S && mrow[key] != -INFINITY);
            if (lane < 2 && 2 * seg + lane < w1) open_tile[2 * seg + lane - w0] = ((open >> (32 * lane)) & 0xffffffffull) != 0;
        }
        __syncthreads();
        if (wave == 0) {
            int count = 0;
            for (int t0 = 0; t0 < w1 - w0; t0 += 64) {
                const bool open = t0 + lane < w1 - w0 && open_tile[t0 + lane] != 0;
                const uint64_t set = __ballot(open);
                if (open) list[count + __popcll(set & ((1ull << lane) - 1))] = (uint16_t)(t0 + lane);
                count += __popcll(set);
            }
            if (lane == 0) list_len = count;
        }
        __syncthreads();
        n = list_len;
    };
    if constexpr (LIST) list_tiles();
    n = __builtin_amdgcn_readfirstlane(n);
    auto key0 = [&](int i) { return (LIST ? w0 + __builtin_amdgcn_readfirstlane((int)list[i]) : t_begin + i) * BN; };

    // The first tiles' loads go out before the queries are split.
    X3Stage<BN, D, kX3Threads, VEC> kst, vst;
    X3Stage<BN, D, kX3Threads, VEC> k1;
    auto load_first = [&]() {
        kst.load(kb, key0(0), s.S - 1, s.E, tid);
        vst.load(vb, key0(0), s.S - 1, s.E, tid);
        k1.load(kb, key0(min(1, n - 1)), s.S - 1, s.E, tid);
    };
    if (n > 0) load_first();
    // Without a mask the scale is applied after the tile max and inside each exponent's FMA: for a
    // positive scale the max of the rounded products equals the rounded product of the max, and the
    // exponent is rounded once instead of twice.  A negative scale enters as its magnitude with the
    // queries negated; a zero scale as the smallest normal float (every visible score then gives
    // exp2 of a value below 2^-100, which is 1, as it is with 0).
    const bool neg = !MASK && s.scale_log2 < 0.f;
    const float csc = MASK ? 0.f : fmaxf(fabsf(s.scale_log2), 0x1p-126f);
    X3 q3[KSTEP];  // step t, half g: dims 16t + 8g + 0..7 of the lane's query
#pragma unroll
    for (int t = 0; t < KSTEP; ++t) {
        f32x4 x[2];
        load_chunk<VEC>(x, qrow, 16 * t + 8 * g, s.E);
        if (neg) x[0] = -x[0], x[1] = -x[1];
        q3[t] = split_chunk(x);
    }

    f32x16 oacc[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[dt][r] = 0.f;
    float m_run = -INFINITY, l_part = 0.f;  // l_part: this half-wave's keys only
    const uint32_t rowb = row_lanebase<BN, D>(lane), trb = tr_lanebase<BN, D>(lane);

    // A wave's tiles are 0 .. wlast (causal tiles past its last query are only staged); only tile
    // wlast can hold keys to mask out at the diagonal or the end.
    int wlast = n - 1;
    if (CAUSAL) wlast = min(wlast, wave_last_q / BN - t_begin);
    wlast = __builtin_amdgcn_readfirstlane(wlast);

    // S^T of tile i.  Smallest products first: the h h products, last, round the sum KSTEP times
    // where the float32 MFMA chain rounded it D / 2 times.
    auto scores = [&](int i, f32x16 &acc) {
        const auto &ck = sk[i & 1];
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
        for (int st = 0; st < KSTEP; ++st) acc = mfma_x3_small(row_frag_x3(ck, rowb, 0, st), q3[st], acc);
#pragma unroll
        for (int st = 0; st < KSTEP; ++st) acc = mfma_bf16(row_frag<BN, D>(ck.p[0], rowb, 0, st), q3[st].h, acc);
    };
    // Tile i's scores into exponent form: masked, and the running max (and, rarely, O and l) moved.
    auto settle = [&](int i, f32x16 &acc, float mrow_lane) {
        if constexpr (MASK == kRowMask) {
            // Lane l holds key l % 32's mask, times log2 e; through the wave's LDS slot it reaches
            // the accumulator layout (registers 4j .. 4j + 3: keys 8j + 4g + 0..3).
            float *slot = mslot[wave];
            if (g == 0) slot[lr] = mrow_lane;
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const f32x4 x = *reinterpret_cast<const f32x4 *>(&slot[8 * j + 4 * g]);
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[4 * j + e] = fmaf(acc[4 * j + e], s.scale_log2, x[e]);
            }
            __builtin_amdgcn_wave_barrier();
        }
        if (i == wlast) {
            const int n0 = key0(i);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int key = n0 + acc_row(r, g);
                if (key >= s.S || (CAUSAL && key > qi)) acc[r] = -INFINITY;
            }
        }
        float mx = acc[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) mx = fmaxf(mx, acc[r]);
        mx = xor32_max(mx);
        if constexpr (!MASK) mx *= csc;
        // Lazy rescaling: the exponent reference m_run moves (and O, l are rescaled) only when
        // some lane's tile max exceeds it by more than 8, so P <= 2^8 and most tiles skip the
        // rescale of the accumulator; out = O / l and lse = m_run + log2(l) are unchanged.
        if (__any(mx > m_run + 8.f)) {
            const float m_new = fmaxf(m_run, mx);
            const float alpha = exp2_fast(m_run - (m_new == -INFINITY ? 0.f : m_new));
            l_part *= alpha;
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) oacc[dt][r] *= alpha;
            m_run = m_new;
        }
    };
    // Scores to probabilities, summed and split: the B operand of P V, 16 keys each.
    auto probabilities = [&](f32x16 &acc, X3 (&p3)[2]) {
        const float m_use = m_run == -INFINITY ? 0.f : m_run;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            acc[r] = exp2_fast(MASK ? acc[r] - m_use : fmaf(acc[r], csc, -m_use));
            l_part += acc[r];
        }
        p3[0] = split3(acc, 0);
        p3[1] = split3(acc, 8);
    };
    auto values = [&](int i, const X3 (&p3)[2]) {  // O^T += V^T P^T of tile i
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
                oacc[dt] = mfma_x3(tr_frag_x3(sv[i & 1], trb, 16 * u, dt), p3[u], oacc[dt]);
    };

    if constexpr (MASK != kFullMask) {
        // Software pipeline, one barrier per tile.  Step i: S of tile i + 1 (MFMA) beside the
        // probabilities of tile i (VALU), then P V of tile i (MFMA) beside the splitting of the tiles
        // to come (VALU): K(i + 2) takes the buffer K(i) left in step i - 1, V(i + 1) that of V(i - 1).
        // (One S and one P V after the other in each step: causal B8 H12 L1024 88.3 against 78.1 us.)
        // STEADY steps hold no conditions, so that each half is one straight run for the scheduler.
        float mcur = 0.f, mnext = 0.f;  // row mask of tiles i and i + 1 (lane: key % 32)
        auto row_mask = [&](int i) -> float {
            if constexpr (MASK != kRowMask) return 0.f;
            const int key = key0(i) + lr;
            return key < s.S ? mrow[key] * kLog2e : -INFINITY;
        };
        // scores(i) with probabilities(acc) in between, and values(i) with the stores of K(i + 2) and
        // V(i + 1): the same sums, in interleave()'s order; LDS operands are read a group ahead.
        auto steady_scores = [&](int i, f32x16 &next, f32x16 &acc, X3 (&p3)[2]) {
            const auto &ck = sk[i & 1];
            const float m_use = m_run == -INFINITY ? 0.f : m_run;
            auto expo = [&](int r) { acc[r] = exp2_fast(MASK ? acc[r] - m_use : fmaf(acc[r], csc, -m_use)); };
#pragma unroll
            for (int r = 0; r < 16; ++r) next[r] = 0.f;
            X3 kf[2];
            bf16x8 kh[KSTEP];
            kf[0] = row_frag_x3(ck, rowb, 0, 0), kh[0] = kf[0].h;
            expo(0), expo(1);
            SplitPair pr;
            u32x4 ph, pm, pl;
            interleave<6 * KSTEP, 24>(
                [&](int m) {
                    const int st = m / 5, ty = m % 5;
                    if (m >= 5 * KSTEP) {
                        next = mfma_bf16(kh[m - 5 * KSTEP], q3[m - 5 * KSTEP].h, next);
                        return;
                    }
                    if (ty == 0 && st + 1 < KSTEP) kf[(st + 1) & 1] = row_frag_x3(ck, rowb, 0, st + 1), kh[st + 1] = kf[(st + 1) & 1].h;
                    next = mfma_x3_part(kf[st & 1], q3[st], next, ty);
                },
                [&](int q) {
                    const int c = q / 3, i = q % 3;
                    if (i == 0) {
                        pr.x0 = acc[2 * c], pr.x1 = acc[2 * c + 1];
                        l_part += pr.x0, l_part += pr.x1;
                        if (c + 1 < 8) expo(2 * c + 2), expo(2 * c + 3);
                    }
                    pr.step(i);
                    if (i == 2) {
                        ph[c % 4] = pr.h, pm[c % 4] = pr.m, pl[c % 4] = pr.l;
                        if (c % 4 == 3)
                            p3[c / 4] = {__builtin_bit_cast(bf16x8, ph), __builtin_bit_cast(bf16x8, pm), __builtin_bit_cast(bf16x8, pl)};
                    }
                });
        };
        auto steady_values = [&](int i, const X3 (&p3)[2], auto &kx, auto &vx) {
            const auto &cv = sv[i & 1];
            X3 vf[2];
            vf[0] = tr_frag_x3(cv, trb, 0, 0);
            constexpr int NG = 2 * NDT, KP = decltype(kst)::PARTS;
            typename decltype(kst)::Splitter sp;
            interleave<6 * NG, 2 * KP>(
                [&](int m) {
                    const int gi = m / 6, ty = m % 6;
                    if (ty == 0 && gi + 1 < NG) vf[(gi + 1) & 1] = tr_frag_x3(cv, trb, 16 * ((gi + 1) / NDT), (gi + 1) % NDT);
                    oacc[gi % NDT] = mfma_x3_part(vf[gi & 1], p3[gi / NDT], oacc[gi % NDT], ty);
                },
                [&](int q) {
                    if (q < KP) kx.part(sp, sk[i & 1], tid, q);
                    else vx.part(sp, sv[(i + 1) & 1], tid, q - KP);
                });
        };
        f32x16 sacc;
        auto step = [&](int i, auto steady) {
            constexpr bool STEADY = decltype(steady)::value;
            const bool live = STEADY || i <= wlast, next = STEADY || i < wlast;
            __syncthreads();
            f32x16 snext;
            X3 p3[2];
            if (MASK == kRowMask && next) mcur = mnext, mnext = row_mask(min(i + 2, n - 1));
            if constexpr (STEADY) {
                steady_scores(i + 1, snext, sacc, p3);
                steady_values(i, p3, kst, vst);
                kst.load(kb, key0(min(i + 3, n - 1)), s.S - 1, s.E, tid);
                vst.load(vb, key0(i + 2), s.S - 1, s.E, tid);
            } else {
                if (next) scores(i + 1, snext);
                if (live) probabilities(sacc, p3);
                if (live) values(i, p3);
                if (i + 2 < n) kst.store(sk[i & 1], tid);
                if (i + 1 < n) vst.store(sv[(i + 1) & 1], tid);
                if (i + 3 < n) kst.load(kb, key0(i + 3), s.S - 1, s.E, tid);
                if (i + 2 < n) vst.load(vb, key0(i + 2), s.S - 1, s.E, tid);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (next) {
                sacc = snext;
                settle(i + 1, sacc, mcur);
            }
        };
        for (;;) {
            if (n > 0) {
                kst.store(sk[0], tid);
                vst.store(sv[0], tid);
                k1.store(sk[1], tid);
                if (n > 2) kst.load(kb, key0(2), s.S - 1, s.E, tid);
                if (n > 1) vst.load(vb, key0(1), s.S - 1, s.E, tid);
                if constexpr (MASK == kRowMask) mcur = row_mask(0), mnext = row_mask(min(1, n - 1));
                __syncthreads();
                if (wlast >= 0) {
                    scores(0, sacc);
                    settle(0, sacc, mcur);
                }
                const int steady = min(wlast, n - 2);
                int i = 0;
                for (; i < steady; ++i) step(i, std::true_type{});
                for (; i < n; ++i) step(i, std::false_type{});
            }
            if constexpr (LIST) {
                w0 += kOrderMaxTiles;
                if (w0 >= ntiles) break;
                __syncthreads();  // everyone is done with the list and the last tiles
                list_tiles();
                n = __builtin_amdgcn_readfirstlane(n);
                wlast = n - 1;
                if (n > 0) load_first();
            } else {
                break;
            }
        }
    } else {
        // A mask value per (query, key): tiles one after the other, a tile whose mask is -inf for
        // every (query, key) of the wave skipped (its probabilities are exactly 0).
        if (n > 0) {
            kst.store(sk[0], tid);
            vst.store(sv[0], tid);
            if (n > 1) {
                kst.load(kb, key0(1), s.S - 1, s.E, tid);
                vst.load(vb, key0(1), s.S - 1, s.E, tid);
            }
        }
        for (int i = 0; i < n; ++i) {
            __syncthreads();  // tile i is in LDS; everyone is done with tile i - 1
            const int n0 = key0(i);
            float mv[16];
            bool any_open = false;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int key = n0 + acc_row(r, g);
                mv[r] = (i <= wlast && key < s.S && qi < s.L) ? mrow[key] : -INFINITY;
                any_open |= mv[r] != -INFINITY;
            }
            const bool live = __any(any_open);
            f32x16 sacc;
            if (live) scores(i, sacc);
            if (i + 1 < n) {
                kst.store(sk[(i + 1) & 1], tid);
                vst.store(sv[(i + 1) & 1], tid);
                if (i + 2 < n) {
                    kst.load(kb, key0(i + 2), s.S - 1, s.E, tid);
                    vst.load(vb, key0(i + 2), s.S - 1, s.E, tid);
                }
            }
            if (live) {
#pragma unroll
                for (int r = 0; r < 16; ++r) sacc[r] = (sacc[r] * s.scale + mv[r]) * kLog2e;
                settle(i, sacc, 0.f);
                X3 p3[2];
                probabilities(sacc, p3);
                values(i, p3);
            }
        }
    }

    float l_run = xor32_add(l_part);
    const int64_t row = (int64_t)bh * s.L + qi;
    const bool partial = SPLIT && npieces > 1;
    float *orow = partial ? a.split_o + (row * a.split_max + piece) * s.E : static_cast<float *>(a.out) + row * s.E;
    // NaN when anything this wave summed was not finite: then an infinite operand may have met the
    // split's NaN remainders, and the wave's rows are redone in float32 (rare, and slow: every lane
    // goes through the keys of its query, its half-wave's dims at a time, reading the mask and
    // skipping masked-out tiles as above).  Not where all that the wave's tiles hold is NaN or below
    // 2^56: then no product or sum overflows, and NaN parts reach what a NaN reaches (NaN in one
    // visible key of every head, causal B8 H12 L1024 D64: 98 us; redone 9204; without NaN 75).
    float bad = l_run * 0.f;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) bad += not_finite(oacc[dt]);
    auto beyond = [&]() {
        float peak = 0.f;  // of what is not NaN
        auto scan = [&](const float *p, int count, int from, int stride) {
            constexpr int U = 8;
            for (int i = from; i < count; i += U * stride)
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    f32x4 x = {0.f, 0.f, 0.f, 0.f};
                    const int at = i + u * stride;
                    if constexpr (VEC) {
                        if (at < count) x = *reinterpret_cast<const f32x4 *>(p + at);
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (at + e < count) x[e] = p[at + e];
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) peak = fmaxf(peak, fabsf(x[e]));
                }
        };
        const int k_end = min(t_end * BN, CAUSAL ? min(wave_last_q + 1, s.S) : s.S);
        scan(qrow, s.E, 4 * g, 8);
        for (int k = t_begin * BN; k < k_end; k += 1024) {  // rows k .. k + 1023 lie behind one another
            const int64_t at = (int64_t)k * s.E;
            const int count = min(1024, k_end - k) * s.E;
            scan(kb + at, count, 4 * lane, 256);
            scan(vb + at, count, 4 * lane, 256);
        }
        return __any(peak >= 0x1p56f);
    };
    if (__any(qi < s.L && bad != 0.f) && beyond()) {
        const int d0 = g * DH;
        float acc[DH];
#pragma unroll
        for (int j = 0; j < DH; ++j) acc[j] = 0.f;
        const int end = CAUSAL ? min(wave_last_q + 1, s.S) : s.S;
        const int k_end = min(t_end * BN, min(s.S, (end + BN - 1) / BN * BN));
        float mx = -INFINITY, sum = 0.f;
        for (int pass = 0; pass < 2; ++pass) {
            const float m_use = mx == -INFINITY ? 0.f : mx;
            for (int n0 = t_begin * BN; n0 < k_end; n0 += BN) {
                if (MASK) {
                    bool any_open = false;
                    for (int key = n0; key < min(n0 + BN, k_end); ++key) any_open |= qi < s.L && mrow[key] != -INFINITY;
                    if (!__any(any_open)) continue;
                }
                for (int key = n0; key < min(n0 + BN, k_end); ++key) {
                    const float *kr = kb + (int64_t)key * s.E, *vr = vb + (int64_t)key * s.E;
                    float dot = 0.f;
#pragma unroll 4
                    for (int j = 0; j < DH; ++j)
                        if (d0 + j < s.E) dot = fmaf(neg ? -qrow[d0 + j] : qrow[d0 + j], kr[d0 + j], dot);
                    dot = xor32_add(dot);
                    if (MASK) dot = ((dot * s.scale) + (qi < s.L ? mrow[key] : -INFINITY)) * kLog2e;
                    else dot *= csc;
                    if (CAUSAL && key > qi) dot = -INFINITY;
                    if (pass == 0) {
                        mx = fmaxf(mx, dot);
                        continue;
                    }
                    const float p = exp2_fast(dot - m_use);
                    sum += p;
#pragma unroll
                    for (int j = 0; j < DH; ++j)
                        if (d0 + j < s.E) acc[j] = fmaf(p, vr[d0 + j], acc[j]);
                }
            }
        }
        m_run = mx, l_run = sum;
        const float inv = l_run == 0.f ? 0.f : 1.f / l_run;
        if (qi < s.L)
#pragma unroll
            for (int j = 0; j < DH; ++j)
                if (d0 + j < s.E) orow[d0 + j] = acc[j] * inv;
    } else if (qi < s.L) {
        const float inv = l_run == 0.f ? 0.f : 1.f / l_run;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int r = 0; r < 16; r += 4) {
                const int d = dt * 32 + acc_row(r, g);
                if (VEC) {
                    if (d < s.E)
                        *reinterpret_cast<f32x4 *>(orow + d) = f32x4{oacc[dt][r] * inv, oacc[dt][r + 1] * inv,
                                                                     oacc[dt][r + 2] * inv, oacc[dt][r + 3] * inv};
                } else {
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (d + u < s.E) orow[d + u] = oacc[dt][r + u] * inv;
                }
            }
    }
    if (qi < s.L && g == 0) {
        const bool empty = l_run == 0.f;
        if (partial) a.split_lse[row * a.split_max + piece] = empty ? -INFINITY : (m_run + log2_fast(l_run)) * kLn2;
        else a.lse[row] = empty ? 0.f : (m_run + log2_fast(l_run)) * kLn2;
    }
}

template <int D, bool CAUSAL, int MASK>
hipError_t launch_rows(const FwdArgs &a, dim3 grid, bool split, hipStream_t st) {
    const dim3 block(kX3Threads);
    if constexpr (MASK == kNoMask) {
        if (split)
            return a.s.vec ? launch(fwd_x3_kernel<D, CAUSAL, MASK, true, true>, grid, block, st, a)
                           : launch(fwd_x3_kernel<D, CAUSAL, MASK, false, true>, grid, block, st, a);
    }
    return a.s.vec ? launch(fwd_x3_kernel<D, CAUSAL, MASK, true, false>, grid, block, st, a)
                   : launch(fwd_x3_kernel<D, CAUSAL, MASK, false, false>, grid, block, st, a);
}

// How a grid of few query tiles splits the keys.  Pieces of 4 tiles of 32 keys, as for the float32
// MFMA's tiles (of 64 keys up to head dim 32), are short ones here: on one MI355X, pieces of 4 -> one per
// CU where that is estimated faster, B7 H2 L253 S1260 E32 22.8 -> 19.5 us (float32 MFMA 22.7), B8 H4 L128
// S4096 E32 42.1 -> 33.7 (36.6), E64 42.7 -> 37.2, B1 H1 L128 S16384 E32 79.9 -> 46.8 (55.3), E64 80.2 ->
// 49.5, E96 127 -> 82, causal B1 H16 L1000 E64 33.0 -> 30.1; one per CU wherever it fits, causal B1 H4 L4096
// E32 62 -> 78.  Up to head dim 32, 256 keys are not worth a second launch (B1 H1 L864 S172 16.3 -> 13.8).
template <int D>
FwdSplitPlan plan(const AttnShape &s) {
    if (D == 32 && s.S <= 256) return FwdSplitPlan{};
    const int64_t blocks = (int64_t)(s.L + kX3M - 1) / kX3M * s.B * s.H;
    const int64_t slots = split_slots(reinterpret_cast<const void *>(&fwd_x3_kernel<D, true, kNoMask, true, true>),
                                      kX3Threads, blocks);
    // Microseconds per tile in a workgroup with a CU to itself: L128 S16384 whole, 620 us at E32, 658 at
    // E64, 1213 at E96.
    return plan_split(s, kX3M, kX3BN, slots, D <= 64 ? 1.2f : 2.4f);
}

template <int D>
hipError_t launch_d(const FwdArgs &args, hipStream_t st) {
    FwdArgs a = args;
    a.s.vec = args.s.vec && args.s.E % 4 == 0;  // the ABI checked alignment; rows of whole 16-byte parts
    const int nqt = (a.s.L + kX3M - 1) / kX3M;
    const dim3 grid(nqt * a.s.B * a.s.H);
    if (a.split_o) {
        const FwdSplitPlan p = plan<D>(a.s);
        if (p.chunk > 0 && p.bytes <= a.split_bytes) {
            record_schedule(split_chunk, p.chunk);
            record_schedule(split_pieces, p.max_pieces);
            a.split_chunk = p.chunk, a.split_max = p.max_pieces;
            a.split_lse = a.split_o + (size_t)a.s.B * a.s.H * a.s.L * p.max_pieces * a.s.E;
            const dim3 sgrid((unsigned)p.blocks);
            if (a.s.causal) return_if((launch_rows<D, true, kNoMask>(a, sgrid, true, st)));
            else return_if((launch_rows<D, false, kNoMask>(a, sgrid, true, st)));
            const int64_t rows = (int64_t)a.s.B * a.s.H * a.s.L;
            return launch(fwd_split_merge_kernel<float>, dim3((unsigned)((rows + 15) / 16)), dim3(256), st, a,
                          kX3M, kX3BN);
        }
    }
    if (!a.s.mask)
        return a.s.causal ? launch_rows<D, true, kNoMask>(a, grid, false, st)
                          : launch_rows<D, false, kNoMask>(a, grid, false, st);
    if (a.s.causal) return launch_rows<D, true, kFullMask>(a, grid, false, st);
    if (a.s.msl != 0) return launch_rows<D, false, kFullMask>(a, grid, false, st);
    return_if(order_heads<kX3BN>(a, st));
    return launch_rows<D, false, kRowMask>(a, ordered_grid(a, nqt), false, st);
}

template <typename F>
auto with_head_dim(int E, F f) {
    if (E <= 32) return f.template operator()<32>();
    if (E <= 64) return f.template operator()<64>();
    return f.template operator()<128>();
}

struct SplitBytes {
    const AttnShape &s;
    template <int D>
    size_t operator()() const { return plan<D>(s).bytes; }
};

struct Launch {
    const FwdArgs &a;
    hipStream_t st;
    template <int D>
    hipError_t operator()() const { return launch_d<D>(a, st); }
};

}  // namespace

size_t fwd_x3_split_bytes(const AttnShape &s) { return with_head_dim(s.E, SplitBytes{s}); }

hipError_t launch_fwd_x3(const FwdArgs &a, hipStream_t st) { return with_head_dim(a.s.E, Launch{a, st}); }

}  // namespace dc
