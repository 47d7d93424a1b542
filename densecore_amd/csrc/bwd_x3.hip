// Float32 attention backward for head dims up to 64 whose workspace holds the dQ slots: products on the
// bf16 matrix cores (x3.hpp).  What it computes, the tiles, steps and slots are bwd_f32.hip's.
#include "bwd_common.hpp"
#include "bwd_tiles.hpp"
#include "common.hpp"
#include "params.hpp"
#include "x3.hpp"

namespace dc {
namespace {

// The steps [i0, i1) of a key tile in plain float32 arithmetic, for key_tile_x3's tiles whose sums
// were not finite: the wave's accumulator (dV of its keys for the first four waves, dK for the
// others, in MFMA layout) and the tile's dQ slot rows.  Slow and rare.
template <int D, bool CAUSAL, int MASK>
DEVI void redo_key_tile(const BwdArgs &a, int tid, int bhk, int kt, int i0, int i1, f32x16 (&acc)[D / 32]) {
    const AttnShape &s = a.s;
    const int wave = tid >> 6, lane = tid & 63, lr = lane & 31, g = lane >> 5;
    const int b = bhk / s.Hkv, hk = bhk % s.Hkv, n0 = kt * kBN;
    const float *kb = static_cast<const float *>(a.k) + (int64_t)bhk * s.S * s.E;
    const float *vb = static_cast<const float *>(a.v) + (int64_t)bhk * s.S * s.E;
    const int m_begin = tile_m_begin(CAUSAL, kt), per_head = tile_per_head(s, kt);
    const int rf = slot_from(s, kt);
    const int64_t slot0 = slot_before(s, kt) * ((int64_t)s.B * s.H);
    // P and dS of (query row, key), every lane its own pair.
    auto pair = [&](int bh, int qq, int key, float &p, float &ds) {
        const int64_t row = (int64_t)bh * s.L + qq;
        const float *q = static_cast<const float *>(a.q) + row * s.E, *go = static_cast<const float *>(a.dout) + row * s.E;
        const int kk = min(key, s.S - 1);
        const float *kr = kb + (int64_t)kk * s.E, *vr = vb + (int64_t)kk * s.E;
        float x = 0.f, dp = 0.f;
#pragma unroll 4
        for (int d = 0; d < s.E; ++d) x = fmaf(q[d], kr[d], x), dp = fmaf(go[d], vr[d], dp);
        x *= s.scale;
        if (MASK) x += s.mask[(int64_t)b * s.msb + (int64_t)(bh - b * s.H) * s.msh + (int64_t)qq * s.msl + kk];
        p = exp2_fast((x - a.lse[row]) * kLog2e);
        if (key >= s.S || (CAUSAL && key > qq)) p = 0.f;
        ds = p * (dp - a.dsum[row]);
    };
    const bool values = wave < 4;  // this wave's accumulator: dV, or dK
    const int kw0 = n0 + (wave & 3) * 32;
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[dt][r] = 0.f;
    for (int i = i0; i < i1; ++i) {
        const int bh = b * s.H + hk * s.repeat + i / per_head, m0 = m_begin + (i % per_head) * kBM;
        for (int qq = m0; qq < min(m0 + kBM, s.L); ++qq) {
            const int64_t row = (int64_t)bh * s.L + qq;
            // dQ: the waves take the rows in turn, lanes the tile's keys, then lanes the dims.
            if ((qq & 7) == wave) {
                float p, d0, d1, t = 0.f;
                pair(bh, qq, n0 + lane, p, d0);
                pair(bh, qq, n0 + 64 + lane, p, d1);
                for (int j = 0; j < kBN && n0 + j < s.S; ++j) {
                    if (CAUSAL && n0 + (j & ~31) > m0 + kBM - 1) break;  // keys no query of the step sees
                    const float dj = __shfl(j < 64 ? d0 : d1, j & 63, 64);
                    if (lane < s.E) t = fmaf(dj, kb[(int64_t)(n0 + j) * s.E + lane], t);
                }
                if (lane < s.E) a.dq_part[(slot0 + (int64_t)bh * (s.L - rf) + (qq - rf)) * s.E + lane] = t;
            }
            if (kw0 >= s.S || (CAUSAL && m0 + kBM - 1 < kw0)) continue;
            float p, ds;
            pair(bh, qq, kw0 + lr, p, ds);
            const float *x = static_cast<const float *>(values ? a.dout : a.q) + row * s.E;
            const float w = values ? p : ds;
#pragma unroll
            for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int d = 32 * dt + acc_row(r, g);
                    if (d < s.E) acc[dt][r] = fmaf(w, x[d], acc[dt][r]);
                }
        }
    }
}

// key_tile on the bf16 matrix cores (x3.hpp), for head dims up to 64: the same tile, steps and
// slots, eight waves in two groups that ping-pong.  Waves w and w + 4 share a SIMD and the same 32
// keys; wave w (group A) forms S, P and dV, wave w + 4 (group B) dP, dS, dK and dQ:
//
//   phase 1 of step i   A: P(i), split, to LDS; stages dO(i + 1)     B: dQ, dK of i - 1, dP(i)  (MFMA)
//   phase 2             A: dV(i), S(i + 1)                 (MFMA)    B: dS(i), split; stages Q(i + 2)
//
// with a barrier after each, so that in every phase one wave of a SIMD feeds the matrix cores (72
// MFMAs in phase 1, 48 in phase 2 at D = 64) while the other has the VALU.  A wave alone does not
// overlap the two well: an MFMA holds its wave's issue for half of its own time, and a dependent
// VALU instruction waits 8 cycles.  (All of it in each of four waves, one per SIMD at 512 registers,
// S and dP of the next step between the VALU work of this one: B8 H16 L1024 D64 full 681 us,
// 35% of the matrix cores' time; this: 530 us, 46%.  On float32 MFMAs, with dS
// shared by four waves through LDS: 655 us.  Issue priorities for the MFMA phases, or dQ in group A:
// no faster, 2% slower.)
//
//   * K (A), V and K^T (B) of the wave's keys are split once and stay in registers; Q and dO are
//     split on their way into LDS (three buffers of Q: S reads one ahead, dK one behind);
//   * P goes from A to B in the accumulators' own layout; dS goes through B's own LDS tile to be
//     read back with queries on lanes, so that each wave forms its 32 keys' share of dQ; the four
//     shares are added in wave order through LDS, one phase later;
//   * S takes the forward's products in the forward's order, so P = exp(S - lse) normalizes
//     exactly as the forward's did.
constexpr int kX3Threads = 2 * kThreads;

template <int D>
struct alignas(16) BwdSmemX3 {
    X3Tile<kBM, D> q[3], o[2];
    float p[kWaves][16][64];         // P, accumulator registers by lane
    X3Tile<32, 32> ds[kWaves];       // dS: rows are keys, columns the step's queries
    float part[kWaves][kBM][D + 4];  // a wave's share of dQ
    float lse[2][kBM], dsum[2][kBM];
    int seen[2 * kWaves];            // row masks: bit 0, the wave's keys have one that is not -inf; bit 1, tame
};

// MASK: 0 none, 1 a value per (query, key), 2 the same for every query (key padding).
template <int D, bool CAUSAL, int MASK, bool VEC>
DEVI void key_tile_x3(const BwdArgs &a, BwdSmemX3<D> &sm, int tid, int bhk, int kt, int i0, int i1, float *kdst,
                      float *vdst) {
    constexpr int KSTEP = D / 16, NDT = D / 32;
    const AttnShape &s = a.s;
    const int wave8 = __builtin_amdgcn_readfirstlane(tid >> 6), wave = wave8 & 3;
    const bool group_a = wave8 < 4;
    const int lane = tid & 63, lr = lane & 31, g = lane >> 5, gtid = tid & (kThreads - 1);
    const int b = bhk / s.Hkv, hk = bhk % s.Hkv;
    const int n0 = kt * kBN;
    const int kw0 = n0 + wave * 32;  // this wave's first key
    const int key = kw0 + lr;        // this lane's key column
    const uint32_t rowb = row_lanebase<kBM, D>(lane), trb = tr_lanebase<kBM, D>(lane);
    const float *mbase = MASK ? s.mask + (int64_t)b * s.msb : nullptr;

    // Steps as (query head, first query), advanced without divisions.
    const int m_begin = tile_m_begin(CAUSAL, kt), per_head = tile_per_head(s, kt);
    struct Pos {
        int bh, m0;
    };
    auto next_pos = [&](Pos p) {
        p.m0 += kBM;
        if (p.m0 >= s.L) p.m0 = m_begin, ++p.bh;
        return p;
    };
    const int rf = slot_from(s, kt);
    const int64_t slot0 = slot_before(s, kt) * ((int64_t)s.B * s.H);
    auto dq_dst = [&](Pos p) -> float * {
        return a.dq_part + (slot0 + (int64_t)p.bh * (s.L - rf) + (p.m0 - rf)) * s.E;
    };
    // Padding: a wave none of whose keys is visible to any query does no work where that is exact
    // (masks that differ between heads are not looked at).  The visit would add P = exp(-inf - lse) = 0
    // times dO to dV and 0 times (dO V - dsum), Q and K to the others: zeros, unless a score, dO V or an
    // operand is not finite (the reference's 0 * NaN).  So the rows must be tame (bwd_pre_block) and the
    // masked keys' K and V too; otherwise every key of the tile is visited.
    int open = 15;
    auto look = [&](bool &any, bool &tame) {  // this wave's part
        any = __any(key < s.S && mbase[min(key, s.S - 1)] != -INFINITY);
        tame = true;
        const int ltid = opaque_index(tid), llane = ltid & 63;
        for (int j = ltid; j < (i1 - i0) * kBM; j += kX3Threads) {
            const int i = i0 + j / kBM, qq = m_begin + (i % per_head) * kBM + j % kBM;
            if (qq < s.L) tame &= a.tame[(int64_t)(b * s.H + hk * s.repeat + i / per_head) * s.L + qq] != 0;
        }
        if (!any && kw0 < s.S) {  // the wave's 32 rows of K (group A) or V (group B)
            const float *rows = static_cast<const float *>(group_a ? a.k : a.v) + ((int64_t)bhk * s.S + kw0) * s.E;
            const int count = min(32, s.S - kw0) * s.E;
            if constexpr (VEC) {
#pragma unroll 8
                for (int j = 4 * llane; j < count; j += 256) {
                    const f32x4 x = *reinterpret_cast<const f32x4 *>(rows + j);
#pragma unroll
                    for (int e = 0; e < 4; ++e) tame &= fabsf(x[e]) <= kTame;
                }
            } else {
#pragma unroll 8
                for (int j = llane; j < count; j += 64) tame &= fabsf(rows[j]) <= kTame;
            }
        }
        tame = __all(tame);
    };
    // Wave w works in a step if some query of the step sees one of its keys.
    auto live_at = [&](int w, int m0) {
        return ((open >> w) & 1) && n0 + 32 * w < s.S && (!CAUSAL || m0 + kBM - 1 >= n0 + 32 * w);
    };

    f32x16 acc[NDT];  // dV^T (group A) or dK^T (group B) of this lane's key
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[dt][r] = 0.f;
    const Pos first{b * s.H + hk * s.repeat + (i0 < i1 ? i0 / per_head : 0), m_begin + (i0 < i1 ? i0 % per_head : 0) * kBM};

    // The waves' shares of the dQ of the step at p, added and stored.
    auto reduce_dq = [&](Pos p) {
        float *dst = dq_dst(p);
        const int rows = min(kBM, s.L - p.m0);
        const int otid = opaque_index(tid);
        const int r = otid / (D / 4), d = otid % (D / 4) * 4;
        if (kBM * D / 4 < kX3Threads && tid >= kBM * D / 4) return;
        f32x4 t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < kWaves; ++w)
            if (live_at(w, p.m0)) t += *reinterpret_cast<const f32x4 *>(&sm.part[w][r][d]);
        if (r >= rows) return;
        if ((s.E & 3) == 0) {  // slots start 16-byte aligned and rows are whole parts
            if (d < s.E) *reinterpret_cast<f32x4 *>(dst + (int64_t)r * s.E + d) = t;
            return;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (d + e < s.E) dst[(int64_t)r * s.E + d + e] = t[e];
    };

    if (i0 < i1) {
        // Group A stages dO (with lse and dsum), group B Q: a step at a time, in registers until the
        // buffer it goes to is free.
        X3Stage<kBM, D, kThreads, VEC> stage;
        float lse_next = 0.f, dsum_next = 0.f;
        Pos load_pos = first;
        const float *sbase = static_cast<const float *>(group_a ? a.dout : a.q);
        auto load_step = [&]() {
            stage.load(sbase + (int64_t)load_pos.bh * s.L * s.E, load_pos.m0, s.L - 1, s.E, gtid);
            if (group_a) {  // every thread its row modulo 32; queries past L: lse +inf, so P = 0
                const int qq = load_pos.m0 + (gtid & (kBM - 1));
                const int64_t at = (int64_t)load_pos.bh * s.L + min(qq, s.L - 1);
                lse_next = qq < s.L ? a.lse[at] : INFINITY;
                dsum_next = qq < s.L ? a.dsum[at] : 0.f;
            }
            load_pos = next_pos(load_pos);
        };
        auto store_do = [&](int buf) {
            stage.store(sm.o[buf], gtid);
            sm.lse[buf][gtid & (kBM - 1)] = lse_next, sm.dsum[buf][gtid & (kBM - 1)] = dsum_next;
        };
        // The keys' rows, through LDS tiles where dS and the dQ shares will be (waves w and w + 4 share
        // tile w): K as A's row operand and B's transposed one, then V as B's row operand.  The first
        // steps' Q and dO are on their way meanwhile.
        X3 kv[KSTEP], kT[NDT][2];
        static_assert(kWaves * sizeof(X3Tile<kBM, D>) <= sizeof(sm.ds) + sizeof(sm.part), "the rows fit");
        X3Tile<kBM, D> &wt = reinterpret_cast<X3Tile<kBM, D> *>(&sm.ds[0])[wave];
        X3Stage<kBM, D, 64, VEC> rows;
        rows.load((static_cast<const float *>(group_a ? a.k : a.v)) + (int64_t)bhk * s.S * s.E, kw0, s.S - 1, s.E, opaque_index(lane));
        load_step();
        bool any = true, tame = true;
        if (MASK == 2 && a.tame) look(any, tame);
        __syncthreads();  // a previous tile's last readers of these areas are done
        if (MASK == 2 && lane == 0) sm.seen[wave8] = (any ? 1 : 0) | (tame ? 2 : 0);
        if (group_a) {
            rows.store(wt, opaque_index(lane));
            store_do(0);
        } else {
            stage.store(sm.q[0], gtid);
        }
        if (i0 + 1 < i1) load_step();
        __syncthreads();
        if (MASK == 2 && a.tame) {
            int all = 2, seen = 0;
#pragma unroll
            for (int w = 0; w < 2 * kWaves; ++w) {
                const int x = sm.seen[w];
                all &= x, seen |= (x & 1) << (w & 3);
            }
            open = __builtin_amdgcn_readfirstlane(all ? seen : 15);
        }
        if (open == 0) {  // nothing visible: the tile's dQ shares are zero
            Pos p = first;
            for (int i = i0; i < i1; ++i, p = next_pos(p)) {
                float *dst = dq_dst(p);
                const int count = min(kBM, s.L - p.m0) * s.E;
                for (int j = tid; j < count; j += kX3Threads) dst[j] = 0.f;
            }
        } else {
            if (group_a) {
#pragma unroll
                for (int st = 0; st < KSTEP; ++st) kv[st] = row_frag_x3(wt, rowb, 0, st);
            } else {
#pragma unroll
                for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                    for (int u = 0; u < 2; ++u) kT[dt][u] = tr_frag_x3(wt, trb, 16 * u, dt);
            }
            __syncthreads();
            if (!group_a) {
                rows.store(wt, opaque_index(lane));
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int st = 0; st < KSTEP; ++st) kv[st] = row_frag_x3(wt, rowb, 0, st);
                if (i0 + 1 < i1) {
                    stage.store(sm.q[1], gtid);
                    if (i0 + 2 < i1) load_step();
                }
            }
            __syncthreads();  // Q of the first two steps, dO of the first

            Pos pos = first, prev{-1, 0};
            bool live = live_at(wave, pos.m0);
            if (group_a) {
                float mrow = 0.f;
                int mrow_bh = -1;
                float mfull[MASK == 1 ? 16 : 1];
                auto full_mask = [&](Pos p) {  // the mask of the step at p
                    if constexpr (MASK == 1) {
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const int qq = p.m0 + acc_row(r, g);
                            mfull[r] = (qq < s.L && key < s.S) ? mbase[(int64_t)(p.bh - b * s.H) * s.msh + (int64_t)qq * s.msl + key] : 0.f;
                        }
                    }
                };
                f32x16 sacc;
                X3 p3[2];
                // S = Q K^T (queries are rows, the wave's keys columns), in k-step groups; and dV += P^T dO,
                // in groups of 32 dims by 16 queries.
                auto score_group = [&](int st, const X3 &q) {
                    if (st == 0) {
#pragma unroll
                        for (int r = 0; r < 16; ++r) sacc[r] = 0.f;
                    }
                    sacc = mfma_x3_small_ba(q, kv[st], sacc);
                };
                auto score_rest = [&](int buf) {
#pragma unroll
                    for (int st = 0; st < KSTEP; ++st)
                        sacc = mfma_bf16(row_frag<kBM, D>(sm.q[buf].p[0], rowb, 0, st), kv[st].h, sacc);
                };
                auto value_group = [&](int gi, const X3 &o) { acc[gi % NDT] = mfma_x3(o, p3[gi / NDT], acc[gi % NDT]); };
                auto scores = [&](int buf) {
                    pipelined<KSTEP>([&](int st) { return row_frag_x3(sm.q[buf], rowb, 0, st); }, score_group);
                    score_rest(buf);
                };
                if (live) {
                    full_mask(pos);
                    scores(0);
                }
                int qb = 0;  // buffer of Q(i)
                for (int i = i0; i < i1; ++i) {
                    const Pos npos = next_pos(pos);
                    const bool nlive = i + 1 < i1 && live_at(wave, npos.m0);
                    const int ob = (i - i0) & 1;
                    qb = qb == 2 ? 0 : qb + 1;  // of Q(i + 1)
                    if (live) {
                        if (MASK == 2 && pos.bh != mrow_bh) {
                            mrow = key < s.S ? mbase[(int64_t)(pos.bh - b * s.H) * s.msh + key] : 0.f;
                            mrow_bh = pos.bh;
                        }
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const f32x4 l4 = *reinterpret_cast<const f32x4 *>(&sm.lse[ob][8 * j + 4 * g]);
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                // scale * q.k (+ mask) - lse in natural-log units, as the reference forms
                                // it, then one conversion to base 2 for v_exp_f32.
                                const int r = 4 * j + e;
                                float x = sacc[r] * s.scale;
                                if (MASK == 1) x += mfull[MASK == 1 ? r : 0];
                                if (MASK == 2) x += mrow;
                                sacc[r] = exp2_fast((x - l4[e]) * kLog2e);
                            }
                        }
                        // Keys past the end or (causal) past a query only occur when the wave's keys reach
                        // the end of the sequence or cross the diagonal of this query tile.
                        if (kw0 + 31 >= s.S || (CAUSAL && kw0 + 31 > pos.m0)) {
                            asm volatile("" ::: "memory");  // keeps the branch: not if-converted into selects
#pragma unroll
                            for (int r = 0; r < 16; ++r)
                                if (key >= s.S || (CAUSAL && key > pos.m0 + acc_row(r, g))) sacc[r] = 0.f;
                        }
#pragma unroll
                        for (int r = 0; r < 16; ++r) sm.p[wave][r][lane] = sacc[r];
                        p3[0] = split3(sacc, 0);
                        p3[1] = split3(sacc, 8);
                    }
                    if (i + 1 < i1) {
                        store_do(ob ^ 1);
                        if (i + 2 < i1) load_step();
                    }
                    __syncthreads();
                    if (nlive) full_mask(npos);
                    auto read_do = [&](int gi) { return tr_frag_x3(sm.o[ob], trb, 16 * (gi / NDT), gi % NDT); };
                    if (live && nlive) {
                        pipelined<2 * NDT + KSTEP>(
                            [&](int k) { return k < 2 * NDT ? read_do(k) : row_frag_x3(sm.q[qb], rowb, 0, k - 2 * NDT); },
                            [&](int k, const X3 &f) {
                                if (k < 2 * NDT) value_group(k, f);
                                else score_group(k - 2 * NDT, f);
                            });
                        score_rest(qb);
                    } else {
                        if (live) pipelined<2 * NDT>(read_do, value_group);
                        if (nlive) scores(qb);
                    }
                    if (prev.bh >= 0) reduce_dq(prev);
                    live = nlive;
                    prev = pos, pos = npos;
                    __syncthreads();
                }
                __syncthreads();
            } else {
                const uint32_t dstrb = tr_lanebase<32, 32>(lane);
                f32x16 pacc;
                X3 d3[2];
                auto dq_share = [&]() {  // of the step whose dS is in the wave's tile
                    const X3 dsT[2] = {tr_frag_x3(sm.ds[wave], dstrb, 0, 0), tr_frag_x3(sm.ds[wave], dstrb, 16, 0)};
#pragma unroll
                    for (int dt = 0; dt < NDT; ++dt) {
                        f32x16 dq;
#pragma unroll
                        for (int r = 0; r < 16; ++r) dq[r] = 0.f;
#pragma unroll
                        for (int u = 0; u < 2; ++u) dq = mfma_x3(kT[dt][u], dsT[u], dq);
#pragma unroll
                        for (int r = 0; r < 16; r += 4)
                            *reinterpret_cast<f32x4 *>(&sm.part[wave][lr][32 * dt + acc_row(r, g)]) =
                                f32x4{dq[r], dq[r + 1], dq[r + 2], dq[r + 3]};
                        __builtin_amdgcn_sched_barrier(0);
                    }
                };
                auto key_group = [&](int gi, const X3 &q) { acc[gi % NDT] = mfma_x3(q, d3[gi / NDT], acc[gi % NDT]); };
                auto prob_group = [&](int st, const X3 &o) { pacc = mfma_x3(o, kv[st], pacc); };
                int pb = 2;  // buffer of Q(i - 1)
                bool plive = false;
                for (int i = i0; i < i1; ++i) {
                    const Pos npos = next_pos(pos);
                    const bool nlive = i + 1 < i1 && live_at(wave, npos.m0);
                    const int ob = (i - i0) & 1;
                    // dK += dS^T Q of the step before, and dP = dO V^T.
                    auto read_q = [&](int gi) { return tr_frag_x3(sm.q[pb], trb, 16 * (gi / NDT), gi % NDT); };
                    auto read_do = [&](int st) { return row_frag_x3(sm.o[ob], rowb, 0, st); };
                    if (plive) dq_share();
#pragma unroll
                    for (int r = 0; r < 16; ++r) pacc[r] = 0.f;
                    if (plive && live) {
                        pipelined<2 * NDT + KSTEP>([&](int k) { return k < 2 * NDT ? read_q(k) : read_do(k - 2 * NDT); },
                                                   [&](int k, const X3 &f) {
                                                       if (k < 2 * NDT) key_group(k, f);
                                                       else prob_group(k - 2 * NDT, f);
                                                   });
                    } else {
                        if (plive) pipelined<2 * NDT>(read_q, key_group);
                        if (live) pipelined<KSTEP>(read_do, prob_group);
                    }
                    __syncthreads();
                    if (live) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const f32x4 d4 = *reinterpret_cast<const f32x4 *>(&sm.dsum[ob][8 * j + 4 * g]);
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const int r = 4 * j + e;
                                pacc[r] = sm.p[wave][r][lane] * (pacc[r] - d4[e]);
                            }
                        }
                        // Into the dS tile: rows are keys, columns queries (registers 8u .. 8u + 7 hold
                        // queries 16u + 4g + 0..3 and 16u + 8 + 4g + 0..3).
#pragma unroll
                        for (int u = 0; u < 2; ++u) {
                            d3[u] = split3(pacc, 8 * u);
                            const bf16x8 parts[3] = {d3[u].h, d3[u].m, d3[u].l};
#pragma unroll
                            for (int pl = 0; pl < 3; ++pl) {
                                const u32x4 w = __builtin_bit_cast(u32x4, parts[pl]);
                                uint32_t *row = reinterpret_cast<uint32_t *>(&sm.ds[wave].p[pl][2 * u * CMTile<32, 32>::P + lr]) + 2 * g;
                                *reinterpret_cast<uint64_t *>(row) = (uint64_t)w[0] | ((uint64_t)w[1] << 32);
                                *reinterpret_cast<uint64_t *>(row + CMTile<32, 32>::P * 4) = (uint64_t)w[2] | ((uint64_t)w[3] << 32);
                            }
                        }
                    }
                    if (prev.bh >= 0) reduce_dq(prev);
                    if (i + 2 < i1) {
                        stage.store(sm.q[pb], gtid);  // Q(i + 2) where Q(i - 1) was
                        if (i + 3 < i1) load_step();
                    }
                    pb = pb == 2 ? 0 : pb + 1;
                    plive = live, live = nlive;
                    prev = pos, pos = npos;
                    __syncthreads();
                }
                if (plive) {
                    dq_share();
                    pipelined<2 * NDT>([&](int gi) { return tr_frag_x3(sm.q[pb], trb, 16 * (gi / NDT), gi % NDT); }, key_group);
                }
                __syncthreads();
            }
            reduce_dq(prev);

            // Not finite: the tile's steps again in plain float32 (x3.hpp).
            float bad = 0.f;
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) bad += not_finite(acc[dt]);
            if (__syncthreads_or(bad != 0.f)) {
                __syncthreads();  // the dQ slots' first stores are ordered before the second
                redo_key_tile<D, CAUSAL, MASK>(a, opaque_index(tid), bhk, kt, i0, i1, acc);
            }
        }
    }

    // dV, or dK times scale, of this lane's key.
    const float mul = group_a ? 1.f : s.scale;
    float *tile_dst = group_a ? vdst : kdst;
    const int etid = opaque_index(tid), ekey = kw0 + (etid & 31), eg = (etid & 63) >> 5;
    if (ekey < s.S) {
        float *dst = tile_dst + (int64_t)(ekey - n0) * s.E;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int r = 0; r < 16; r += 4) {
                const int d = dt * 32 + acc_row(r, eg);
                if (VEC) {
                    if (d < s.E)
                        *reinterpret_cast<f32x4 *>(dst + d) =
                            f32x4{acc[dt][r] * mul, acc[dt][r + 1] * mul, acc[dt][r + 2] * mul, acc[dt][r + 3] * mul};
                } else {
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (d + u < s.E) dst[d + u] = acc[dt][r + u] * mul;
                }
            }
    }
}

template <int D, bool CAUSAL, int MASK, bool VEC>
__global__ __launch_bounds__(kX3Threads) __attribute__((amdgpu_waves_per_eu(2, 2))) void bwd_x3_kernel(BwdArgs a) {
    __shared__ BwdSmemX3<D> sm;
    const int BHk = a.s.B * a.s.Hkv;
    const int kt = blockIdx.x / BHk;  // tile 0 has the most causal work, so it goes first
    const int bhk = blockIdx.x % BHk;
    const int64_t row0 = ((int64_t)bhk * a.s.S + (int64_t)kt * kBN) * a.s.E;
    key_tile_x3<D, CAUSAL, MASK, VEC>(a, sm, threadIdx.x, bhk, kt, 0, tile_steps(a.s, kt),
                                      static_cast<float *>(a.dk) + row0, static_cast<float *>(a.dv) + row0);
}

template <int D, bool CAUSAL, int MASK, bool VEC>
__global__ __launch_bounds__(kX3Threads) __attribute__((amdgpu_waves_per_eu(2, 2))) void bwd_x3_streamk_kernel(BwdArgs a, StreamK sk) {
    __shared__ BwdSmemX3<D> sm;
    streamk_range(a, sk, [&](int bhk, int kt, int i0, int i1, float *kd, float *vd, bool) {
        key_tile_x3<D, CAUSAL, MASK, VEC>(a, sm, threadIdx.x, bhk, kt, i0, i1, kd, vd);
    });
}

// Head dims up to 64 (split products on the bf16 matrix cores).
template <int D, int MASK, bool VEC>
hipError_t launch_x3(const BwdArgs &a, const StreamK &sk, dim3 grid, hipStream_t st) {
    const dim3 block(kX3Threads);
    if (sk.chunks > 0) {
        if (a.s.causal) return launch(bwd_x3_streamk_kernel<D, true, MASK, VEC>, grid, block, st, a, sk);
        return launch(bwd_x3_streamk_kernel<D, false, MASK, VEC>, grid, block, st, a, sk);
    }
    if (a.s.causal) return launch(bwd_x3_kernel<D, true, MASK, VEC>, grid, block, st, a);
    return launch(bwd_x3_kernel<D, false, MASK, VEC>, grid, block, st, a);
}

template <int D, bool VEC>
hipError_t launch_mask(const BwdArgs &a, const StreamK &sk, dim3 grid, hipStream_t st) {
    if (!a.s.mask) return launch_x3<D, 0, VEC>(a, sk, grid, st);
    return a.s.msl == 0 ? launch_x3<D, 2, VEC>(a, sk, grid, st) : launch_x3<D, 1, VEC>(a, sk, grid, st);
}

}  // namespace

hipError_t launch_bwd_x3(const BwdArgs &a, const StreamK &sk, dim3 grid, hipStream_t st) {
    if (a.s.E <= 32) return a.s.vec ? launch_mask<32, true>(a, sk, grid, st) : launch_mask<32, false>(a, sk, grid, st);
    return a.s.vec ? launch_mask<64, true>(a, sk, grid, st) : launch_mask<64, false>(a, sk, grid, st);
}

}  // namespace dc
