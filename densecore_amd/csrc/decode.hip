// Single-query (decode) attention over a contiguous KV cache: split-KV partials + merge.
//
// The reference has no decode kernel: a decode step is torch_attention::forward with L = 1,
// non-causal (src/torch_attention.rs:157, 176-180), i.e. for each (batch, head)
//     out = softmax(scale * q k^T) v,  lse = max + ln(sum).
// That is a streaming read of K and V with a few flops per byte, so this path is bound by HBM
// bandwidth, not by the matrix cores.  Layout and work split:
//
//   * grid = B*H*splits workgroups: each owns split_len consecutive keys of one head;
//   * a lane loads 16 bytes per row (4 floats or 8 bf16), D/VEC lanes cover one key row, so
//     every global load instruction of a wave reads whole, contiguous 64-byte-aligned rows;
//   * pass 1 streams the split's K rows, reduces q.k across the row's lanes with butterflies
//     and keeps the split's scores (log2 units) in LDS; pass 2 streams V rows and accumulates
//     p * v per lane, reduced across row groups and waves through LDS;
//   * each split writes (acc[E], max, sum) to the workspace; a merge kernel rescales and sums
//     the splits per head and writes out and lse;
//   * grouped heads (H > Hkv) take a kernel of their own, in which a workgroup serves up to 8 query
//     heads of one kv head from one read of its keys and values (decode_group_kernel).
#include <algorithm>
#include <mutex>

#include "common.hpp"
#include "params.hpp"

namespace dc {
namespace {

// Scratch of the allocation-free entry point (dc_sdpa_decode_noalloc): the split partials live
// in this file-scope array instead of a caller's workspace.  Each GPU the library runs on holds
// its own copy, at its own address, until the process ends.  Host code never passes the array's
// name to a kernel (on the host it is only a stand-in): it passes the device address that
// hipGetSymbolAddress returns for the current device, looked up once per device.
static __device__ __align__(256) float scratch[kDecodeScratchBytes / sizeof(float)];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
float *g_scratch[kMaxDevices];

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kMaxSplitLen = 2048;
constexpr int kUnroll = 8;

// Query heads a workgroup of grouped heads serves: 2, 4 or 8 (more heads than 8: groups of 8).
inline int group_heads(int repeat) { return repeat <= 2 ? 2 : repeat <= 4 ? 4 : 8; }

// Keys a wave of decode_group_kernel takes at a time.
constexpr int group_chunk_keys(int D, int elem) {
    const int n = 64 * 16 * 8 / (D * elem);
    return n > 64 ? 64 : n < 16 ? 16 : n;
}
constexpr int padded_head_dim(int E) { return E <= 32 ? 32 : E <= 64 ? 64 : E <= 128 ? 128 : 256; }

template <typename T> struct Vec16;
template <> struct Vec16<float> {
    static constexpr int N = 4;
    typedef f32x4 type;
};
template <> struct Vec16<__bf16> {
    static constexpr int N = 8;
    typedef bf16x8 type;
};

// Part of a key or value row (read once: nontemporal loads, B32 H32 S4096 D128 6.1 -> 6.9 TB/s).
// vec: rows are 16-byte aligned and hold a whole number of parts (E % N == 0).
template <typename T, int N>
DEVI void load_row_part(float (&x)[N], const T *row, int d0, int E, bool vec) {
    if (vec) {
        if (d0 >= E) {
#pragma unroll
            for (int i = 0; i < N; ++i) x[i] = 0.f;
            return;
        }
        const auto v = load_nt(reinterpret_cast<const typename Vec16<T>::type *>(row + d0));
#pragma unroll
        for (int i = 0; i < N; ++i) x[i] = to_f32<T>(v[i]);
    } else {
#pragma unroll
        for (int i = 0; i < N; ++i) x[i] = d0 + i < E ? to_f32<T>(row[d0 + i]) : 0.f;
    }
}

template <typename T, int D>
__global__ __launch_bounds__(kThreads) void decode_split_kernel(DecodeArgs a) {
    constexpr int VEC = Vec16<T>::N;
    constexpr int LPR = D / VEC;          // lanes per key row
    constexpr int RPW = 64 / LPR;         // rows per wave per step
    constexpr int RPS = RPW * kWaves;     // rows per workgroup per step
    __shared__ float sc[kMaxSplitLen];
    __shared__ float red[kWaves][RPW][D];
    __shared__ float wred[kWaves];

    const AttnShape &s = a.s;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int sub = lane / LPR, part = lane % LPR, d0 = part * VEC;
    const int split = blockIdx.x % a.splits, bh = blockIdx.x / a.splits;
    const int b = bh / s.H, h = bh % s.H, hk = h / s.repeat;
    const int k0 = split * a.split_len, k1 = min(s.S, k0 + a.split_len);
    const int n = max(0, k1 - k0);
    const T *kb = static_cast<const T *>(a.k) + ((int64_t)(b * s.Hkv + hk) * s.S) * s.E;
    const T *vb = static_cast<const T *>(a.v) + ((int64_t)(b * s.Hkv + hk) * s.S) * s.E;

    float qv[VEC];
    load_row_part<T, VEC>(qv, static_cast<const T *>(a.q) + (int64_t)bh * s.E, d0, s.E, s.vec);
#pragma unroll
    for (int i = 0; i < VEC; ++i) qv[i] *= s.scale_log2;

    // Pass 1: scores for rows k0 + step*RPS + wave*RPW + sub.
    const int my_row0 = wave * RPW + sub;
    for (int base = 0; base < n; base += RPS * kUnroll) {
        float kx[kUnroll][VEC];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const int r = base + u * RPS + my_row0;
            if (r < n)
                load_row_part<T, VEC>(kx[u], kb + (int64_t)(k0 + r) * s.E, d0, s.E, s.vec);
            else
#pragma unroll
                for (int i = 0; i < VEC; ++i) kx[u][i] = 0.f;
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            float dot = 0.f;
#pragma unroll
            for (int i = 0; i < VEC; ++i) dot = fmaf(qv[i], kx[u][i], dot);
#pragma unroll
            for (int off = 1; off < LPR; off <<= 1) dot += __shfl_xor(dot, off, 64);
            const int r = base + u * RPS + my_row0;
            if (part == 0 && r < n) sc[r] = dot;
        }
    }
    __syncthreads();

    // Split max and sum of exp2(score - max).
    float mx = -INFINITY;
    for (int r = tid; r < n; r += kThreads) mx = fmaxf(mx, sc[r]);
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
    if (lane == 0) wred[wave] = mx;
    __syncthreads();
    mx = wred[0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) mx = fmaxf(mx, wred[w]);
    const float m_use = mx == -INFINITY ? 0.f : mx;
    float sum = 0.f;
    for (int r = tid; r < n; r += kThreads) {
        const float p = exp2_fast(sc[r] - m_use);
        sc[r] = p;
        sum += p;
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) sum += __shfl_xor(sum, off, 64);
    __syncthreads();  // everyone read wred (max) and wrote sc (p)
    if (lane == 0) wred[wave] = sum;
    __syncthreads();
    sum = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) sum += wred[w];

    // Pass 2: acc[d] = sum_r p[r] * V[r][d].
    float acc[VEC];
#pragma unroll
    for (int i = 0; i < VEC; ++i) acc[i] = 0.f;
    for (int base = 0; base < n; base += RPS * kUnroll) {
        float vx[kUnroll][VEC];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const int r = base + u * RPS + my_row0;
            if (r < n)
                load_row_part<T, VEC>(vx[u], vb + (int64_t)(k0 + r) * s.E, d0, s.E, s.vec);
            else
#pragma unroll
                for (int i = 0; i < VEC; ++i) vx[u][i] = 0.f;
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const int r = base + u * RPS + my_row0;
            const float p = r < n ? sc[r] : 0.f;
#pragma unroll
            for (int i = 0; i < VEC; ++i) acc[i] = fmaf(p, vx[u][i], acc[i]);
        }
    }
#pragma unroll
    for (int i = 0; i < VEC; ++i) red[wave][sub][d0 + i] = acc[i];
    __syncthreads();
    float *out = a.part + ((int64_t)bh * a.splits + split) * (s.E + 2);
    for (int d = tid; d < s.E; d += kThreads) {
        float t = 0.f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w)
#pragma unroll
            for (int r = 0; r < RPW; ++r) t += red[w][r][d];
        out[d] = t;
    }
    if (tid == 0) {
        out[s.E] = mx;
        out[s.E + 1] = sum;
    }
}

// Grouped heads: one workgroup reads a range of one kv head's keys and values once for HG of the
// query heads that share it.  HBM-bound like the kernel above, but per byte there are now HG times
// the products and, on K, HG times the reductions, which on the VALU (8 FMAs and 4 shuffles per 16
// bytes and head in bf16) would pass the time the bytes take from four heads up.  So the scores
// run on the matrix cores, keys as rows and the heads as the 16 columns: a lane's 16 bytes of a
// key row are its MFMA operand as they come from memory, and the sum over the head dim needs no
// shuffles.  The value product stays on the VALU: a lane owns 16 bytes of a row's dims for all HG
// heads (an MFMA would need V transposed).  Waves take chunks of CK keys in turn and keep an
// online softmax each, so nothing in the loop waits for another wave; the waves' sums are merged
// through LDS at the end, in wave order.
// B16 H32 Hkv8 S8192 D128 bf16: 349 us with one workgroup per query head (its four readers of a
// kv head took K and V from L2 and the last-level cache at 1.6 TB/s of distinct bytes) ->
// 103 us (5.2 TB/s).
// A chunk is 8 16-byte vectors of K (and of V) per lane, 16 to 64 keys (16 vectors: 107 us at the
// shape above, but 145 against 89 us at H64 Hkv8 D256, whose registers then leave one wave per SIMD).
template <typename T, int D>
constexpr int kChunkKeys = group_chunk_keys(D, sizeof(T));

// Sixteen keys' scores from a lane's N parts of their rows.  Float32: chains of two products of four
// dims, summed in pairs as a tree (one chain through the accumulator: 1.5 to 3.5 times the error
// against float64 of the split kernel, whose lanes sum their dims as a tree).  The barriers keep the
// chains of one pair of parts in registers at a time.
template <int I, int W, int N>
DEVI f32x4 tree_rows(const f32x4 (&k)[N], const f32x4 (&q)[N]) {
    if constexpr (W <= 2) {
        f32x4 c[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) c[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = I; i < I + W; ++i)
#pragma unroll
            for (int u = 0; u < 4; ++u) c[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i][u], q[i][u], c[u], 0, 0, 0);
        const f32x4 t = (c[0] + c[1]) + (c[2] + c[3]);
        __builtin_amdgcn_sched_barrier(0);
        return t;
    } else {
        const f32x4 lo = tree_rows<I, W / 2>(k, q);
        return lo + tree_rows<I + W / 2, W / 2>(k, q);
    }
}
template <int N>
DEVI f32x4 mfma_rows(const f32x4 (&k)[N], const f32x4 (&q)[N]) {
    static_assert((N & (N - 1)) == 0, "halved down to pairs");
    return tree_rows<0, N>(k, q);
}
template <int N>
DEVI f32x4 mfma_rows(const bf16x8 (&k)[N], const bf16x8 (&q)[N]) {
    f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < N; ++i) c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[i], q[i], c, 0, 0, 0);
    return c;
}

template <typename T, int D, int HG, bool FULL>
__global__ __launch_bounds__(kThreads) void decode_group_kernel(DecodeArgs a) {
    typedef typename Vec16<T>::type vec_t;
    constexpr int VEC = Vec16<T>::N;
    constexpr int KS = D / (4 * VEC);      // 16-byte vectors of a key row per lane (4 lanes per row)
    constexpr int CK = kChunkKeys<T, D>;   // keys per chunk: at most 16 vectors of K (or V) per lane
    constexpr int NG = CK / 16;            // MFMA row groups per chunk
    constexpr int LPR = D / VEC, RPW = 64 / LPR, NV = CK / RPW;
    static_assert(HG <= 16 && NG >= 1 && CK % RPW == 0, "chunk shape");
    __shared__ __attribute__((aligned(16))) float pbuf[kWaves][CK][HG];  // probabilities, then alpha in row 0
    __shared__ float red[kWaves][HG][D];
    __shared__ float wmax[kWaves][HG], wsum[kWaves][HG];

    const AttnShape &s = a.s;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int hgroups = (s.repeat + HG - 1) / HG;
    const int hg = blockIdx.x % hgroups, split = blockIdx.x / hgroups % a.splits;
    const int bk = blockIdx.x / hgroups / a.splits;  // b * Hkv + kv head
    const int bh0 = bk * s.repeat + hg * HG;         // first query head's row (b * H + h)
    const int heads = min(HG, s.repeat - hg * HG);
    const int k0 = split * a.split_len, k1 = min(s.S, k0 + a.split_len);
    const int n = max(0, k1 - k0);
    const T *kb = static_cast<const T *>(a.k) + ((int64_t)bk * s.S + k0) * s.E;
    const T *vb = static_cast<const T *>(a.v) + ((int64_t)bk * s.S + k0) * s.E;

    // 16 bytes of a row at dim d; dims past E are 0.  FULL (E == D, aligned rows): no tests.
    auto load_part = [&](const T *row, int d) -> vec_t {
        // Ordinary loads: an instruction takes half a 128-byte line of each key row, and its other half
        // is read by the next one (nontemporal: 113 against 107 us at the shape above).
        if constexpr (FULL) return *reinterpret_cast<const vec_t *>(row + d);
        vec_t x;
        if (s.vec) {
            if (d < s.E) return *reinterpret_cast<const vec_t *>(row + d);
#pragma unroll
            for (int i = 0; i < VEC; ++i) x[i] = from_f32<T>(0.f);
            return x;
        }
#pragma unroll
        for (int i = 0; i < VEC; ++i) x[i] = d + i < s.E ? row[d + i] : from_f32<T>(0.f);
        return x;
    };

    const int col = lane & 15, quad = lane >> 4;  // MFMA column (head) and reduction quarter
    vec_t qv[KS];
#pragma unroll
    for (int i = 0; i < KS; ++i) {
#pragma unroll
        for (int e = 0; e < VEC; ++e) qv[i][e] = from_f32<T>(0.f);
        if (col < heads)
            qv[i] = load_part(static_cast<const T *>(a.q) + (int64_t)(bh0 + col) * s.E, (4 * i + quad) * VEC);
    }
    const int sub = lane / LPR, d0 = (lane % LPR) * VEC;
    float acc[HG][VEC];
#pragma unroll
    for (int h = 0; h < HG; ++h)
#pragma unroll
        for (int i = 0; i < VEC; ++i) acc[h][i] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;  // of head `col` (per lane: l_run of this lane's keys)

    for (int c0 = wave * CK; c0 < n; c0 += kWaves * CK) {
        const int rows = min(CK, n - c0);
        const T *kc = kb + (int64_t)c0 * s.E, *vc = vb + (int64_t)c0 * s.E;
        vec_t kx[NG][KS];
#pragma unroll
        for (int gi = 0; gi < NG; ++gi) {
            const int r = min(16 * gi + col, rows - 1);  // past the end: any key (its score is dropped)
#pragma unroll
            for (int i = 0; i < KS; ++i) kx[gi][i] = load_part(kc + (int64_t)r * s.E, (4 * i + quad) * VEC);
        }
        f32x4 sc[NG];
#pragma unroll
        for (int gi = 0; gi < NG; ++gi) sc[gi] = mfma_rows(kx[gi], qv);
        // V's loads go out before the softmax: its latency hides part of theirs.
        vec_t vx[NV];
#pragma unroll
        for (int j = 0; j < NV; ++j) vx[j] = load_part(vc + (int64_t)min(j * RPW + sub, rows - 1) * s.E, d0);
        if (rows < CK) {  // rows past the end enter as 0, not as the key they were read from
#pragma unroll
            for (int j = 0; j < NV; ++j)
#pragma unroll
                for (int i = 0; i < VEC; ++i)
                    if (j * RPW + sub >= rows) vx[j][i] = from_f32<T>(0.f);
        }
        float mx = -INFINITY;
#pragma unroll
        for (int gi = 0; gi < NG; ++gi)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                sc[gi][r] = 16 * gi + 4 * quad + r < rows ? sc[gi][r] * s.scale_log2 : -INFINITY;
                mx = fmaxf(mx, sc[gi][r]);
            }
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = xor32_max(mx);
        if (__any(mx > m_run)) {
            const float m_new = fmaxf(m_run, mx);
            const float alpha = exp2_fast(m_run - (m_new == -INFINITY ? 0.f : m_new));
            m_run = m_new;
            l_run *= alpha;
            if (quad == 0 && col < HG) pbuf[wave][0][col] = alpha;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int h = 0; h < HG; ++h) {
                const float al = pbuf[wave][0][h];
#pragma unroll
                for (int i = 0; i < VEC; ++i) acc[h][i] *= al;
            }
            __builtin_amdgcn_wave_barrier();
        }
        const float m_use = m_run == -INFINITY ? 0.f : m_run;
        float l_chunk = 0.f;
#pragma unroll
        for (int gi = 0; gi < NG; ++gi)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float p = exp2_fast(sc[gi][r] - m_use);
                l_chunk += p;
                if (col < HG) pbuf[wave][16 * gi + 4 * quad + r][col] = p;
            }
        l_run += l_chunk;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();  // the wave's probabilities are in LDS (its accesses stay in order)
        // Above 128 dims a wave's lane takes every key of the wave: summed by chunk, then over the chunks.
        constexpr bool BY_CHUNK = D > 128;
        float part[BY_CHUNK ? HG : 1][VEC] = {};
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            float p[HG];
#pragma unroll
            for (int h = 0; h < HG; ++h) p[h] = pbuf[wave][j * RPW + sub][h];
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                const float x = to_f32<T>(vx[j][i]);
#pragma unroll
                for (int h = 0; h < HG; ++h) {
                    if constexpr (BY_CHUNK) part[h][i] = fmaf(p[h], x, part[h][i]);
                    else acc[h][i] = fmaf(p[h], x, acc[h][i]);
                }
            }
        }
        if constexpr (BY_CHUNK)
#pragma unroll
            for (int h = 0; h < HG; ++h)
#pragma unroll
                for (int i = 0; i < VEC; ++i) acc[h][i] += part[h][i];
        __builtin_amdgcn_wave_barrier();
    }

    // Merge: each wave's sums over its row lanes, then the waves at the common max.
    l_run += __shfl_xor(l_run, 16, 64);
    l_run = xor32_add(l_run);
    if (quad == 0 && col < HG) wmax[wave][col] = m_run, wsum[wave][col] = l_run;
#pragma unroll
    for (int h = 0; h < HG; ++h)
#pragma unroll
        for (int i = 0; i < VEC; ++i) {
            float t = acc[h][i];
#pragma unroll
            for (int off = LPR; off < 64; off <<= 1) t += __shfl_xor(t, off, 64);
            if (sub == 0) red[wave][h][d0 + i] = t;
        }
    __syncthreads();
    for (int i = tid; i < heads * D; i += kThreads) {
        const int h = i / D, d = i % D;
        float m = wmax[0][h];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) m = fmaxf(m, wmax[w][h]);
        const float m_use = m == -INFINITY ? 0.f : m;
        float t = 0.f, l = 0.f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const float e = exp2_fast(wmax[w][h] - m_use);
            t = fmaf(red[w][h][d], e, t);
            l = fmaf(wsum[w][h], e, l);
        }
        float *out = a.part + ((int64_t)(bh0 + h) * a.splits + split) * (s.E + 2);
        if (d < s.E) out[d] = t;
        if (d == 0) out[s.E] = m, out[s.E + 1] = l;
    }
}

// One workgroup per (batch, head): rescale the splits to the global max and sum them.  Bound by the
// latency of reading a few hundred KB spread over the partials: the splits are dealt over the
// workgroup's thread groups (one per head-dim row of threads), whose sums are added in order.
constexpr int kMergeThreads = 256;
template <typename T>
__global__ __launch_bounds__(kMergeThreads) void decode_merge_kernel(DecodeArgs a) {
    const AttnShape &s = a.s;
    __shared__ float part_sum[kMergeThreads], wred[kMergeThreads / 64];
    const int bh = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ld = s.E + 2;
    const float *p = a.part + (int64_t)bh * a.splits * ld;
    float m = -INFINITY;
    for (int i = lane; i < a.splits; i += 64) m = fmaxf(m, p[(int64_t)i * ld + s.E]);
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    const float m_use = m == -INFINITY ? 0.f : m;
    // The sum l: each thread its splits, then over the workgroup.
    float l = 0.f;
    for (int i = tid; i < a.splits; i += kMergeThreads)
        l += p[(int64_t)i * ld + s.E + 1] * exp2_fast(p[(int64_t)i * ld + s.E] - m_use);
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) l += __shfl_xor(l, off, 64);
    if (lane == 0) wred[wave] = l;
    // Thread groups of `dims` threads (a power of two covering E): group g sums splits g, g + ng, ...
    const int dims = padded_head_dim(s.E);
    const int d = tid & (dims - 1), g = tid / dims, ng = kMergeThreads / dims;
    float t = 0.f;
    if (d < s.E) {
        int i = g;
        for (; i + 3 * ng < a.splits; i += 4 * ng) {
            float x[4], w[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float *row = p + (int64_t)(i + u * ng) * ld;
                x[u] = row[d], w[u] = row[s.E];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) t = fmaf(x[u], exp2_fast(w[u] - m_use), t);
        }
        for (; i < a.splits; i += ng) t = fmaf(p[(int64_t)i * ld + d], exp2_fast(p[(int64_t)i * ld + s.E] - m_use), t);
    }
    part_sum[tid] = t;
    __syncthreads();
    l = 0.f;
#pragma unroll
    for (int w = 0; w < kMergeThreads / 64; ++w) l += wred[w];
    const bool empty = l == 0.f;
    const float inv = empty ? 0.f : 1.f / l;
    if (g == 0 && d < s.E) {
        for (int k = 1; k < ng; ++k) t += part_sum[k * dims + d];
        static_cast<T *>(a.out)[(int64_t)bh * s.E + d] = from_f32<T>(t * inv);
    }
    if (tid == 0) a.lse[bh] = empty ? 0.f : (m_use + log2_fast(l)) * kLn2;
}

template <typename T, int D, int HG>
hipError_t launch_group(const DecodeArgs &a, bool full, hipStream_t st) {
    const dim3 grid((int64_t)a.splits * a.s.B * a.s.Hkv * ((a.s.repeat + HG - 1) / HG));
    return full ? launch(decode_group_kernel<T, D, HG, true>, grid, dim3(kThreads), st, a)
                : launch(decode_group_kernel<T, D, HG, false>, grid, dim3(kThreads), st, a);
}

template <typename T, int D>
hipError_t launch_t(const DecodeArgs &args, hipStream_t st) {
    DecodeArgs a = args;
    // 16-byte row parts: aligned tensors whose rows hold a whole number of them.
    a.s.vec = args.s.vec && args.s.E % Vec16<T>::N == 0;
    const int64_t BH = (int64_t)a.s.B * a.s.H;
    const int rep = a.s.repeat;
    if (rep > 1) {
        const bool full = a.s.vec && a.s.E == D;
        const int hg = group_heads(rep);
        return_if((hg == 2 ? launch_group<T, D, 2> : hg == 4 ? launch_group<T, D, 4> : launch_group<T, D, 8>)(a, full, st));
    } else {
        return_if(launch(decode_split_kernel<T, D>, dim3((int64_t)a.splits * BH), dim3(kThreads), st, a));
    }
    return_if(launch(decode_merge_kernel<T>, dim3(BH), dim3(kMergeThreads), st, a));
    return hipSuccess;
}

template <typename T>
hipError_t launch_dtype(const DecodeArgs &a, hipStream_t st) {
    if (a.s.E <= 32) return launch_t<T, 32>(a, st);
    if (a.s.E <= 64) return launch_t<T, 64>(a, st);
    if (a.s.E <= 128) return launch_t<T, 128>(a, st);
    return launch_t<T, 256>(a, st);
}

}  // namespace

// Enough splits for ~4K workgroups (16 per CU on 256 CUs), at most kMaxSplitLen keys each.
// Measured on C4 (B32 H32 S4096 D128 fp32, per call): 2K workgroups 6087 GB/s, 4K 6117-6121,
// 6K 6085, 8K 6051-6063, 16K 5820.
// Grouped heads count a workgroup per kv head and head group: about 2K of them, none of under 16
// chunks of keys (four per wave) unless that leaves CUs idle, and then none of under four.  A
// workgroup's partials are HG heads wide, so short ranges make the merge the larger part (bf16 B2
// H32 Hkv4 S16000 D128: 125 splits 55 us, 32 splits 24.5 us; B16 H32 Hkv8 S8192: 2K workgroups 103,
// 4K 106, 8K 148 us).  The splits are also held to what the scratch of the allocation-free entry
// point takes, so that it refuses no call for having grouped heads; with a workspace too, because both
// entry points give the same bits.  It binds at batch * heads * head dim in the millions, where workgroups
// are plenty (B188 H64 Hkv8 S1000 E256 bf16, 1 split or the 2 of a larger scratch: 298.3 us both; B16
// H128 Hkv8 S2000 E256 float32 189 both).
int decode_splits(const AttnShape &s, bool bf16, int *split_len) {
    const int64_t BH = (int64_t)s.B * s.H;
    const int64_t max_splits = (s.S + 63) / 64;
    auto near = [&](int64_t groups) { return groups > 0 ? (4096 + groups - 1) / groups : 1; };
    int64_t splits = std::max<int64_t>(1, std::min(near(BH), max_splits));
    int64_t len = (s.S + splits - 1) / splits;
    if (len > kMaxSplitLen) {
        len = kMaxSplitLen;
        splits = (s.S + len - 1) / len;
    }
    if (s.repeat > 1) {
        const int64_t hg = group_heads(s.repeat), groups = (int64_t)s.B * s.Hkv * ((s.repeat + hg - 1) / hg);
        const int elem = bf16 ? 2 : 4;
        const int64_t room = BH > 0 ? (int64_t)(kDecodeScratchBytes / ((s.E + 2) * sizeof(float))) / BH : 1;
        const int64_t ck = group_chunk_keys(padded_head_dim(s.E), elem);
        auto pieces = [&](int64_t keys) { return (s.S + keys - 1) / keys; };
        auto near_groups = [&](int64_t n) { return groups > 0 ? (n + groups - 1) / groups : 1; };
        splits = std::min(std::max(std::min(near_groups(2048), pieces(16 * ck)), near_groups(256)), pieces(4 * ck));
        splits = std::max<int64_t>(1, std::min(splits, room));
        len = (s.S + splits - 1) / splits;
    }
    *split_len = (int)(len < 1 ? 1 : len);
    return (int)splits;
}

hipError_t launch_decode(const DecodeArgs &a, bool bf16, hipStream_t st) {
    return bf16 ? launch_dtype<__bf16>(a, st) : launch_dtype<float>(a, st);
}

hipError_t decode_scratch(float **ptr) {
    int dev = -1;
    return_if(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch[dev] == nullptr) {
        void *p = nullptr;
        return_if(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        g_scratch[dev] = static_cast<float *>(p);
    }
    *ptr = g_scratch[dev];
    return hipSuccess;
}

}  // namespace dc
