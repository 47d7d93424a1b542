// The reference's CPU generator stream (src/torch_random.rs:9-98, PyTorch's mt19937) drawn on
// the GPU, for dropout masks that are bit-identical to Generator::bernoulli
// (src/torch_random.rs:241-254): element e keeps iff the double built from outputs 2e and
// 2e + 1, (hi << 32 | lo) & (2^53 - 1) times 2^-53, is below p.
//
// The engine's untempered words satisfy x[t + 624] = x[t + 397] ^ twist(x[t], x[t + 1]) for every
// t >= 0 (the in-place update of next_state, src/torch_random.rs:66-77), so the stream is one
// linear recurrence over GF(2).  A window of 624 consecutive words that follows at least one
// update lies in the 19937-dimensional subspace on which that recurrence has the primitive
// characteristic polynomial phi (degree 19937), so the window d words later is
//     W(t + d) = sum_i g_i W(t + i),   g = z^d mod phi,
// a XOR of shifted copies of the sequence (the standard jump-ahead of F2-linear generators).
//
// Layout of one draw of n elements (positions relative to the start of the engine's current
// block of 624 words, r = position of the next output):
//   head      elements [0, Eh), Eh = 64: generated from the current block by one workgroup
//             (mt_base_kernel), which also writes the window at A0 = r + 2 Eh (A0 >= 1, so that
//             window follows an update even when the block is a freshly seeded one);
//   chunks    chunk c covers elements [Eh + c J/2, Eh + (c + 1) J/2), J = 2^17 words; its window
//             is W(A0 + c J), reached from W(A0) through a radix-64 tree of jumps (c = 64 c1 + c0:
//             a jump by c1 2^23, then one by c0 2^17; mt_jump_kernel), and a workgroup of four
//             waves takes it from there: two generate its words from that window, two temper and
//             test them (mt_chunk_kernel).
// Keep bits: element e is bit e % 32 of word e / 32 (heads and chunks write whole words).  The
// engine block that holds the last output drawn is written back to the state (by the base
// workgroup or by the chunk whose range holds the block's first word), and the host moves
// (left, next) the way next_state/random do.
//
// The jump polynomials (128 of them) are computed once on the host: phi by Berlekamp-Massey on
// 2 * 19937 bits of the stream, then z^(digit * 2^(17 + 6 level)) mod phi by squaring and
// multiplying; the caller uploads them into its own device buffer (dc_mt19937_table_init).
#include <climits>
#include <type_traits>
#include <cstring>
#include <mutex>
#include <vector>

#include "common.hpp"
#include "params.hpp"

namespace dc {
namespace mt {

namespace {

// ---------------------------------------------------------------- host: GF(2) polynomials

constexpr int kPW = kTableWords / 2;  // 312 uint64 words: 19968 bits, degree < 19937 fits

inline uint32_t twist(uint32_t u, uint32_t v) {
    return (((u & 0x80000000u) | (v & 0x7fffffffu)) >> 1) ^ ((v & 1u) ? 0x9908b0dfu : 0u);
}

typedef std::vector<uint64_t> Bits;  // bit i of a polynomial = coefficient of z^i

inline bool bit(const Bits &a, int i) { return (a[i >> 6] >> (i & 63)) & 1u; }
inline void flip(Bits &a, int i) { a[i >> 6] ^= 1ull << (i & 63); }

// a ^= b << s (b has nb words; a is large enough).
void xor_shifted(Bits &a, const Bits &b, int nb, int s) {
    const int ws = s >> 6, bs = s & 63;
    for (int i = 0; i < nb; ++i) {
        if (!b[i]) continue;
        a[i + ws] ^= b[i] << bs;
        if (bs) a[i + ws + 1] ^= b[i] >> (64 - bs);
    }
}

// Characteristic polynomial of the engine: Berlekamp-Massey on bit 0 of the untempered words
// x[624 .. 624 + 2 * 19937) of the engine seeded with 5489.
Bits char_poly() {
    const int n = 2 * kDegree;
    std::vector<uint32_t> x(kState + n + 1);
    x[0] = 5489u;
    for (int j = 1; j < kState; ++j) x[j] = 1812433253u * (x[j - 1] ^ (x[j - 1] >> 30)) + (uint32_t)j;
    for (int t = 0; t + kState < (int)x.size(); ++t)
        x[t + kState] = x[t + kM] ^ twist(x[t], x[t + 1]);
    const int W = kPW + 1;
    Bits C(W + 1, 0), B(W + 1, 0), R(W + 1, 0), T;
    C[0] = B[0] = 1;
    int L = 0, m = 1;
    for (int k = 0; k < n; ++k) {
        // R bit j = s[k - j]: shift in s[k].
        for (int w = W; w > 0; --w) R[w] = (R[w] << 1) | (R[w - 1] >> 63);
        R[0] = (R[0] << 1) | (x[kState + k] & 1u);
        int d = 0;
        for (int w = 0; w <= W; ++w) d ^= __builtin_popcountll(C[w] & R[w]) & 1;
        if (!d) {
            ++m;
        } else if (2 * L <= k) {
            T = C;
            xor_shifted(C, B, W + 1 - (m >> 6) - 1, m);
            L = k + 1 - L;
            B = T;
            m = 1;
        } else {
            xor_shifted(C, B, W + 1 - (m >> 6) - 1, m);
            ++m;
        }
    }
    // phi(z) = z^L C(1/z).
    Bits phi(kPW, 0);
    if (L != kDegree) return Bits();
    for (int i = 0; i <= L; ++i)
        if (bit(C, i)) flip(phi, L - i);
    return phi;
}

struct Field {
    Bits phi;

    // a * b mod phi, both of degree < 19937.
    Bits mul(const Bits &a, const Bits &b) const {
        Bits tab[16];
        for (int w = 0; w < 16; ++w) {
            tab[w].assign(kPW + 1, 0);
            for (int s = 0; s < 4; ++s)
                if (w >> s & 1) xor_shifted(tab[w], b, kPW, s);
        }
        Bits r(2 * kPW + 2, 0);
        for (int p = 0; p < kPW * 16; ++p) {
            const int nib = (int)(a[p >> 4] >> (4 * (p & 15))) & 15;
            if (nib) xor_shifted(r, tab[nib], kPW + 1, 4 * p);
        }
        return reduce(r);
    }

    // r mod phi for any length of r (top-down: each step clears bit i and touches no bit above).
    Bits reduce(Bits r) const {
        const int top = (int)r.size() * 64 - 1;
        r.resize(r.size() + kPW + 2, 0);
        for (int i = top; i >= kDegree; --i)
            if (bit(r, i)) xor_shifted(r, phi, kPW, i - kDegree);
        r.resize(kPW);
        return r;
    }

    // z^e mod phi (square and multiply from the top set bit of e).
    Bits pow_z(uint64_t e) const {
        Bits r(kPW, 0);
        r[0] = 1;
        for (int b = 63 - (e ? __builtin_clzll(e) : 63); b >= 0; --b) {
            r = mul(r, r);
            if (e >> b & 1) {
                Bits s(kPW + 1, 0);
                xor_shifted(s, r, kPW, 1);
                r = reduce(s);
            }
        }
        return r;
    }
};

struct Tables {
    bool ok = false;
    Field f;
    std::vector<uint32_t> words;  // kTablePolys polynomials of kTableWords uint32 words
};

const Tables &tables() {
    static Tables t;
    static std::once_flag once;
    std::call_once(once, [] {
        t.f.phi = char_poly();
        if (t.f.phi.empty()) return;
        t.words.assign((size_t)kTablePolys * kTableWords, 0);
        Bits base = t.f.pow_z(1ull << kChunkLog2);  // z^(2^17)
        for (int level = 0; level < kJumpLevels; ++level) {
            Bits p(kPW, 0);
            p[0] = 1;
            for (int digit = 0; digit < kRadix; ++digit) {
                uint32_t *dst = &t.words[((size_t)level * kRadix + digit) * kTableWords];
                std::memcpy(dst, p.data(), kTableWords * sizeof(uint32_t));
                p = t.f.mul(p, base);
            }
            base = p;  // base^16
        }
        t.ok = true;
    });
    return t;
}

// The window d words after `win` (which must follow at least one engine update).
void jump_host(const Field &f, const uint32_t *win, uint64_t d, uint32_t *out) {
    const Bits g = f.pow_z(d);
    std::vector<uint32_t> seq(kState + kDegree + 1);
    std::memcpy(seq.data(), win, kState * sizeof(uint32_t));
    for (int t = 0; t + kState < (int)seq.size(); ++t)
        seq[t + kState] = seq[t + kM] ^ twist(seq[t], seq[t + 1]);
    std::vector<uint32_t> acc(kState, 0);
    for (int i = 0; i < kDegree; ++i)
        if (bit(g, i))
            for (int j = 0; j < kState; ++j) acc[j] ^= seq[i + j];
    std::memcpy(out, acc.data(), kState * sizeof(uint32_t));
}

// ---------------------------------------------------------------- device

DEVI uint32_t twist_d(uint32_t u, uint32_t v) {
    return (((u & 0x80000000u) | (v & 0x7fffffffu)) >> 1) ^ ((v & 1u) ? 0x9908b0dfu : 0u);
}

// src/torch_random.rs:86-89.
DEVI uint32_t temper(uint32_t y) {
    y ^= y >> 11;
    y ^= (y << 7) & 0x9d2c5680u;
    y ^= (y << 15) & 0xefc60000u;
    y ^= y >> 18;
    return y;
}

// uniform_f64 (src/torch_random.rs:106-110) of the pair (hi, lo) compared with p: with
// r = (hi << 32 | lo) & (2^53 - 1), r * 2^-53 < p exactly when r < ceil(p * 2^53) (both sides
// scaled by a power of two, r an integer), the threshold the host computes.
DEVI bool keep(uint32_t hi, uint32_t lo, uint64_t thr) {
    const uint64_t r = (((uint64_t)hi << 32) | lo) & ((1ull << 53) - 1);
    return r < thr;
}

// One workgroup: the current block `state` (positions 0..623), the words after it up to
// A0 + 623, the head's keep bits, the window at A0, and (when the last drawn output lies before
// A0) the engine block that holds it.
constexpr int kBaseWords = 2048;

__global__ __launch_bounds__(256) void mt_base_kernel(MtArgs a) {
    __shared__ uint32_t x[kBaseWords];
    const int tid = threadIdx.x;
    for (int i = tid; i < kState; i += 256) x[i] = a.state[i];
    __syncthreads();
    const int total = a.a0 + kState;  // positions [0, total) are needed
    for (int base = kState; base < total; base += 128) {
        const int u = base + tid;
        if (tid < 128 && u < total) x[u] = x[u - 227] ^ twist_d(x[u - 624], x[u - 623]);
        __syncthreads();
    }
    // Head elements [0, min(Eh, n)): outputs r + 2e, r + 2e + 1, 64 elements per wave pass.
    const int lane = tid & 63, wave = tid >> 6;
    const int64_t head = a.n < a.eh ? a.n : a.eh;
    for (int e0 = wave * 64; e0 < a.eh; e0 += 256) {
        const int e = e0 + lane;
        bool k = false;
        if (e < head) k = keep(temper(x[a.r + 2 * e]), temper(x[a.r + 2 * e + 1]), a.thr);
        const uint64_t m = __ballot(k);
        if (e0 < head) {
            if (lane == 0) a.bits[e0 >> 5] = (uint32_t)m;
            if (lane == 1 && e0 + 32 < head) a.bits[(e0 >> 5) + 1] = (uint32_t)(m >> 32);
        }
    }
    for (int i = tid; i < kState; i += 256) a.win[i] = x[a.a0 + i];
    if (a.state_block >= 0 && a.state_block * kState < a.a0)
        for (int i = tid; i < kState; i += 256) a.state[i] = x[a.state_block * kState + i];
}

// dst window w = W(src window w / 64 + digit * step), digit = w % 64, with g = table[level][digit],
// by `split` workgroups: each generates the sequence seq[i] = x[src + i] into LDS as far as it needs
// it and its eight waves sum g's terms over a 1/(8 split) part of [0, 19937); lanes < 52 own 12
// consecutive output words each and read a 20-word window of seq per group of 8 terms.  The eight
// partial windows are XORed, and the workgroups' ones stand side by side in dst (`src_split` of
// them in src), XORed by whoever reads them.
// Bound: VALU (about 6 M XORs per jump) and, in a launch of few jumps, one workgroup's latency, so
// the level-1 jumps (at most 64) are split over 8 workgroups each.  The sequence is 20576 words, 96 more than half of a CU's LDS: its last words are made
// after the terms that read the first ones are summed, in their place, and two workgroups share a
// CU.  Both launches for 25 M draws (6 level-1, 384 level-0 jumps): 300 -> 143 us.
constexpr int kSeqWords = 20480;  // LDS: half a CU's
constexpr int kTailWords = 96;    // words past it that the last terms read (kDegree - 1 + 12 * 51 + 19)
constexpr int kJumpWaves = 8;
constexpr int kOwn = 12, kOwners = kState / kOwn;       // 52 owner lanes per wave
constexpr int kTailTerms = 620 * 32;                    // terms from here on read past kSeqWords
static_assert(kTailTerms - 1 + kOwn * (kOwners - 1) + kOwn + 8 < kSeqWords, "terms before the tail stay inside");
static_assert(kDegree - 1 + kOwn * (kOwners - 1) + kOwn + 8 < kSeqWords + kTailWords && kTailWords <= 227, "one step makes the tail");

__global__ __launch_bounds__(512) void mt_jump_kernel(const uint32_t *src, int src_split, uint32_t *dst,
                                                      const uint32_t *table, int level, int count, int split) {
    __shared__ __align__(16) uint32_t seq[kSeqWords];
    const int w = blockIdx.x / split, part = blockIdx.x % split;
    if (w >= count) return;
    const int digit = w % kRadix;
    const uint32_t *in = src + (size_t)(w / kRadix) * src_split * kState;
    uint32_t *out = dst + ((size_t)w * split + part) * kState;
    const int tid = threadIdx.x;
    auto first = [&](int i) {
        uint32_t x = 0;
        for (int k = 0; k < src_split; ++k) x ^= in[(size_t)k * kState + i];
        return x;
    };
    if (digit == 0) {
        for (int i = tid; i < kState; i += 512) out[i] = part == 0 ? first(i) : 0u;
        return;
    }
    const uint32_t *g = table + ((size_t)level * kRadix + digit) * kTableWords;
    // Words of g (32 terms each) per wave; this wave's are [w0, w1).
    const int per_wave = (kTableWords + kJumpWaves * split - 1) / (kJumpWaves * split);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int w0 = min(kTableWords, (part * kJumpWaves + wave) * per_wave), w1 = min(kTableWords, w0 + per_wave);
    const int block_end = min(kTableWords, (part + 1) * kJumpWaves * per_wave);
    const int need = min(kSeqWords, 32 * block_end + kState + 16);
    for (int i = tid; i < kState; i += 512) seq[i] = first(i);
    __syncthreads();
    for (int base = kState; base < need; base += 227) {  // x[u] needs x[u - 227]: 227 at a time
        const int u = base + tid;
        if (tid < 227 && u < kSeqWords) seq[u] = seq[u - 227] ^ twist_d(seq[u - 624], seq[u - 623]);
        __syncthreads();
    }
    // Every lane runs the sum (lanes past the owners repeat the last owner's words and store
    // nothing), so the group index and the polynomial bits are wave-uniform: the bits come from
    // two VGPRs loaded up front (word w of this wave's at lane w % 64 of gw[w / 64]) through
    // readlane, and the term tests are scalar branches.
    const int j0 = kOwn * (lane < kOwners ? lane : kOwners - 1);
    const uint32_t gw0 = w0 + lane < w1 ? g[w0 + lane] : 0u;
    const uint32_t gw1 = w0 + 64 + lane < w1 ? g[w0 + 64 + lane] : 0u;
    uint32_t acc[kOwn];
#pragma unroll
    for (int u = 0; u < kOwn; ++u) acc[u] = 0;
    auto terms = [&](int wi, bool wrap) {  // word w0 + wi of g
        const uint32_t word = wi < 64 ? __builtin_amdgcn_readlane(gw0, wi) : __builtin_amdgcn_readlane(gw1, wi - 64);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t gb = (word >> (8 * k)) & 0xffu;
            if (gb == 0) continue;
            const int base = 32 * (w0 + wi) + 8 * k + j0;
            uint32_t win[kOwn + 8];  // seq[base + 0 .. 19]: five 16-byte reads
#pragma unroll
            for (int u = 0; u < kOwn + 8; u += 4) {
                const int at = base + u - (wrap && base + u >= kSeqWords ? kSeqWords : 0);
                const u32x4 x = *reinterpret_cast<const u32x4 *>(&seq[at]);
                win[u] = x[0], win[u + 1] = x[1], win[u + 2] = x[2], win[u + 3] = x[3];
            }
#pragma unroll
            for (int d = 0; d < 8; ++d)
                if (gb >> d & 1u)
#pragma unroll
                    for (int u = 0; u < kOwn; ++u) acc[u] ^= win[d + u];
        }
    };
    constexpr int kTailWord = kTailTerms / 32;
    for (int wi = 0; wi < min(w1, kTailWord) - w0; ++wi) terms(wi, false);
    __syncthreads();  // every wave is done with the sequence's start
    if (block_end > kTailWord) {
        if (tid < kTailWords) {
            const int u = kSeqWords + tid;
            seq[tid] = seq[u - 227] ^ twist_d(seq[u - 624], seq[u - 623]);
        }
        __syncthreads();
        for (int wi = max(0, kTailWord - w0); wi < w1 - w0; ++wi) terms(wi, true);
        __syncthreads();
    }
    if (lane < kOwners)  // seq is free: the waves' partial windows
#pragma unroll
        for (int u = 0; u < kOwn; ++u) seq[wave * kState + j0 + u] = acc[u];
    __syncthreads();
    for (int j = tid; j < kState; j += 512) {
        uint32_t x = 0;
#pragma unroll
        for (int v = 0; v < kJumpWaves; ++v) x ^= seq[v * kState + j];
        out[j] = x;
    }
}

// One workgroup per chunk, which makes kStep words (96 elements, three words of keep bits) per step
// from its window, in an LDS ring: a word depends on the word 227 before it, so a step's words
// depend only on earlier steps'.  Bound by the latency of a step (LDS read, twist, LDS write,
// barrier), so two waves do nothing else, and two more temper and test the words of the step
// before.  (Two chunks per wave, three times 32 elements between LDS ordering points: 371 us for 25 M
// draws, at an eighth of the waves the device holds; two waves that do both: 204 us; now 128 us.)
constexpr int kStep = 192;

__global__ __launch_bounds__(256) void mt_chunk_kernel(MtArgs a, const uint32_t *wins) {
    __shared__ __align__(16) uint32_t ring[1024];
    const int tid = threadIdx.x & 127, lane = tid & 63;  // of the generating, or the testing, pair of waves
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool generate = __builtin_amdgcn_readfirstlane(threadIdx.x >> 7) == 0;
    const int c = blockIdx.x;
    const int64_t e_begin = a.eh + (int64_t)c * (kChunkWords / 2);  // first element, a multiple of 64
    const int n = (int)min(a.n - e_begin, (int64_t)(kChunkWords / 2));
    int words = 2 * n;  // words to make: all elements', or up to the end of the engine block it writes back
    int sb = -1;        // that block's first word
    const int64_t chunk_pos = a.a0 + (int64_t)c * kChunkWords;  // relative position of word 0
    if (a.state_block >= 0 && a.state_block * (int64_t)kState >= a.a0) {
        const int64_t at = a.state_block * (int64_t)kState - chunk_pos;
        if (at >= 0 && at < kChunkWords) {
            sb = (int)at;
            words = max(words, sb + kState);
        }
    }
    for (int i = threadIdx.x; i < kState; i += 256) ring[i] = wins[(size_t)c * kState + i];
    __syncthreads();
    uint32_t *bits = a.bits + (e_begin >> 5);
    const uint64_t thr = a.thr;
    const int pair = min(tid, kStep / 2 - 1);  // this lane's element of a step (the last 32 lanes repeat one)
    // Steps start at words 0, 192, 384 (the window's), 576 (its last 48 and the first made from it),
    // 768, ..., `last`.
    const int last = words <= 576 + kStep ? 576 : 576 + (words - 577) / kStep * kStep;
    if (generate) {
        const int u0 = 576 + 2 * pair;
        // The last 32 lanes write their element's words again: the same values.
        auto make = [&](int u) {
            const uint32_t x0 = ring[(u - 624) & 1023], x1 = ring[(u - 623) & 1023], x2 = ring[(u - 622) & 1023];
            const uint32_t y0 = ring[(u - 227) & 1023], y1 = ring[(u - 226) & 1023];
            *reinterpret_cast<uint2 *>(&ring[u & 1023]) = make_uint2(y0 ^ twist_d(x0, x1), y1 ^ twist_d(x1, x2));
        };
        if (u0 >= kState) make(u0);
        __syncthreads();
        for (int u = u0 + kStep; u <= last + 2 * pair; u += kStep) {
            make(u);
            __syncthreads();
        }
        return;
    }
    // Keep bits of the step at `base`: wave 0 holds 64 elements, wave 1 the other 32; lanes 0 and 1 (lane
    // 0 of wave 1) store a word each.  FULL: every element of the step is the chunk's.
    auto emit = [&](int base, auto full) {
        constexpr bool FULL = decltype(full)::value;
        const uint2 x = *reinterpret_cast<const uint2 *>(&ring[(base + 2 * pair) & 1023]);
        const uint64_t r = (((uint64_t)temper(x.x) << 32) | temper(x.y)) & ((1ull << 53) - 1);
        const bool valid = FULL | (base / 2 + tid < n);
        const uint64_t m = __ballot(valid & (r < thr));
        const int word = base / 64 + 2 * wave + lane;
        if (lane < 2 - wave && (FULL || 32 * word < n)) bits[word] = (uint32_t)(m >> (32 * lane));
    };
    const std::true_type whole;
    const std::false_type cut;
    // The step after which the ring holds the whole engine block this chunk writes back (it is copied
    // then: at most 624 + 191 words were made since its first, and the next step's take older places).
    const int block_at = sb < 0 ? INT_MAX : max(576, 576 + (sb + kState - kStep - 576 + kStep - 1) / kStep * kStep);
    const int full_end = n >= kStep / 2 ? 2 * n - kStep : -1;  // the last base whose elements are all the chunk's
    for (int base = 0; base < 576; base += kStep) emit(base, cut);
    __syncthreads();
    int base = 576;  // made: its step, while the next one's is being made
    for (;;) {
        for (; base < min(last, block_at) && base <= full_end; base += kStep) {
            emit(base, whole);
            __syncthreads();
        }
        if (base == block_at)
            for (int i = tid; i < kState; i += 128) a.state[i] = ring[(sb + i) & 1023];
        emit(base, cut);
        if (base >= last) break;
        __syncthreads();
        base += kStep;
    }
}

// y = x * (keep ? scale : 0): the reference's input * noise, noise = bernoulli / float32(1 - p)
// (python/densecore/functional.py:244, 638-641).  Four elements per thread (one 16-byte load
// and store, four bits of one word) when the tensors allow it.
__global__ __launch_bounds__(256) void dropout_apply_kernel(const uint32_t *bits, int64_t n, float scale,
                                                            const float *x, float *y) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const bool k = (bits[i >> 5] >> (i & 31)) & 1u;
    y[i] = x[i] * (k ? scale : 0.0f);
}

__global__ __launch_bounds__(256) void dropout_apply4_kernel(const uint32_t *bits, int64_t n4, float scale,
                                                             const f32x4 *x, f32x4 *y) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= n4) return;
    const uint32_t b = bits[t >> 3] >> (4 * (t & 7));
    f32x4 v = load_nt(x + t);  // x and y stream through once
#pragma unroll
    for (int c = 0; c < 4; ++c) v[c] = v[c] * ((b >> c & 1u) ? scale : 0.0f);
    __builtin_nontemporal_store(v, y + t);
}

}  // namespace

// Workgroups per level-1 jump.
constexpr int kLevel1Split = 8;

size_t window_words(int chunks) {
    if (chunks == 0) return kState;
    const int n1 = (chunks + kRadix - 1) / kRadix;
    return (size_t)(1 + n1 * kLevel1Split + chunks) * kState;
}

bool tables_ready() { return tables().ok; }

const uint32_t *table_words() { return tables().ok ? tables().words.data() : nullptr; }

bool jump_window_host(const uint32_t *win, uint64_t d, uint32_t *out) {
    const Tables &t = tables();
    if (!t.ok) return false;
    jump_host(t.f, win, d, out);
    return true;
}

void twist_block_host(const uint32_t *in, uint32_t *out) {
    uint32_t x[2 * kState];
    std::memcpy(x, in, kState * sizeof(uint32_t));
    for (int t = 0; t < kState; ++t) x[t + kState] = x[t + kM] ^ twist(x[t], x[t + 1]);
    std::memcpy(out, x + kState, kState * sizeof(uint32_t));
}

hipError_t launch_bernoulli(const MtArgs &a, const uint32_t *table, int chunks, uint32_t *wins,
                            hipStream_t st) {
    return_if(launch(mt_base_kernel, dim3(1), dim3(256), st, a));
    if (chunks == 0) return hipSuccess;
    // Radix-64 tree: level 1 (c1), then level 0 (c0).  Window arrays are carved from `wins`
    // (window_words(chunks) words): [W(A0)] [n1 level-1 windows, in parts] [chunk windows].
    const int n1 = (chunks + kRadix - 1) / kRadix;
    uint32_t *l1 = wins + kState, *l0 = l1 + (size_t)n1 * kLevel1Split * kState;
    return_if(launch(mt_jump_kernel, dim3(n1 * kLevel1Split), dim3(512), st, (const uint32_t *)wins, 1, l1, table, 1, n1,
                     kLevel1Split));
    return_if(launch(mt_jump_kernel, dim3(chunks), dim3(512), st, (const uint32_t *)l1, kLevel1Split, l0, table, 0, chunks, 1));
    return launch(mt_chunk_kernel, dim3(chunks), dim3(256), st, a, (const uint32_t *)l0);
}

hipError_t launch_dropout_apply(const uint32_t *bits, int64_t n, float scale, const float *x, float *y,
                                hipStream_t st) {
    if (n % 4 == 0 && ((uintptr_t)x & 15) == 0 && ((uintptr_t)y & 15) == 0) {
        const int64_t n4 = n / 4;
        return launch(dropout_apply4_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), st, bits, n4,
                      scale, reinterpret_cast<const f32x4 *>(x), reinterpret_cast<f32x4 *>(y));
    }
    return launch(dropout_apply_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), st, bits, n, scale, x, y);
}

}  // namespace mt
}  // namespace dc
