// Token sampling after the lm_head (UnifiedSampling,
// crates/stark-engine/src/backends/cpu/kernel/sampling/unified_sampling.rs:14-117;
// noise crates/stark-engine/src/encodable_block/sampling/gumbel.rs):
// non-finite rows give u32::MAX; the bitmask sends masked tokens to -inf; the
// temperature scales (after a uniform shift that puts the maximum at zero when
// scaling would overflow a finite logit); top-k / top-p / min-p keep a prefix
// of the logits sorted by value (ties: lower index first); a seeded row adds
// Gumbel noise -ln(-ln u), u from Philox4x32-10; the result is the argmax
// (ties: lower index), or u32::MAX when no finite logit is left.
//
// Two forms. Sampled rows, and greedy rows of many logits, are cut into
// 4096-logit pieces, one workgroup each, in three to seven short launches (see
// "Split form" below); the other rows (sample_split, dispatch_rules.h), and the
// rare ones the split form hands back, take the row form: one workgroup of 1024
// threads per row, in passes over the row:
//  - the prefix kept by the filters has length L, the minimum of top_k, the
//    count of logits at or above max + ln(min_p), and for top-p the first
//    prefix whose mass reaches p. Top-p follows the reference's f32 sums in
//    its order: only terms exp(x - max) of at least 2^-27 can move them, and
//    when at most 4096 logits carry such terms they are sorted in LDS and
//    summed in order on one thread (exact_top_p_prefix). Rows with more
//    significant terms (very flat rows) take a radix descent over the
//    order-preserving key with per-digit mass histograms in 2^-40 fixed
//    point (integer atomics: independent of thread timing), which differs
//    from the sequential f32 sums only where the prefix mass lands within
//    their rounding error of p;
//  - the kept set, the first L logits in (value desc, index asc) order, is
//    located by a second radix select over the key (and over the index among
//    equal keys);
//  - the final pass scores kept logits (+ noise) and takes the argmax.
// Without noise the filters cannot change the argmax (the maximum is always
// kept), so a greedy row is one max/argmax pass.
#include <cmath>

#include "qmm_common.h"

// The reference rounds x * (1 / temperature) and the differences exp takes; no contraction into fma here.
#pragma clang fp contract(off)

namespace qmm {
namespace {

constexpr int kST = 1024;  // threads per row

// A second 1024-thread workgroup fits a CU up to 80 scalar registers: at 82, 512
// greedy rows of 16384 logits took 25.0 us in place of 17.5.
#define QMM_TWO_PER_CU __attribute__((amdgpu_num_sgpr(80)))

struct SampleArgs {
    const void* logits;
    uint32_t* out;
    const uint64_t* seeds;
    const uint32_t* bitmask;
    uint32_t vocab, dt;
    uint32_t has_temperature, has_top_k, has_top_p, has_min_p;
    float temperature, top_p, min_p;
    uint32_t top_k;
};

struct SampleLds {
    unsigned long long hist[256];  // mass (fixed point) or counts per digit
    unsigned long long acc64[2];
    float redf[kST / 64];
    uint32_t redi[kST / 64];
    uint32_t flag;
    uint32_t scal[4];
};

// Philox4x32-10 (Salmon et al., SC'11; the constants are the published ones)
__device__ __forceinline__ uint32_t philox_word(uint32_t offset, uint32_t word, uint64_t seed) {
    uint32_t c0 = offset, c1 = 0, c2 = 0, c3 = 0;
    uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        if (r) {
            k0 += 0x9E3779B9u;
            k1 += 0xBB67AE85u;
        }
        const uint64_t p0 = (uint64_t)0xD2511F53u * c0, p1 = (uint64_t)0xCD9E8D57u * c2;
        const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c1 ^ k0, n2 = (uint32_t)(p0 >> 32) ^ c3 ^ k1;
        c1 = (uint32_t)p1;
        c3 = (uint32_t)p0;
        c0 = n0;
        c2 = n2;
    }
    return word == 0 ? c0 : word == 1 ? c1 : word == 2 ? c2 : c3;
}

// gumbel.rs:49-79 (revidx maps a logit to its Philox counter and word)
__device__ __forceinline__ float gumbel(uint64_t seed, uint32_t i, uint32_t vocab) {
    const uint32_t t = i % 1024u, blk = i / 1024u;
    const uint32_t offset = ((vocab + 4095u) / 4096u) * t + blk / 4u;
    uint32_t v = philox_word(offset, blk % 4u, seed) >> 8;
    v = v < 1u ? 1u : v;
    const float u = (float)v * (1.0f / 16777216.0f);
    return -logf(-logf(u));
}

// Top-p in the reference's order: terms of at least 2^-27 (times the maximum's)
// sorted in LDS, at most kExactCap of them.
constexpr int kExactCap = 4096;
constexpr float kSignificant = 0x1p-27f;

struct ExactLds {
    unsigned long long key[kExactCap];  // fkey(x) << 32 | ~index: descending = (value desc, index asc)
    alignas(16) float term[kExactCap];
    float norm;
    uint32_t n, len;
};

// order-preserving key of a non-NaN float (larger float -> larger key)
__device__ __forceinline__ uint32_t fkey(float f) {
    const uint32_t b = __float_as_uint(f + 0.0f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

__device__ __forceinline__ float logit_at(const SampleArgs& a, size_t row, uint32_t i) {
    return load_as_f32(a.logits, a.dt, row * a.vocab + i);
}

// block reductions (every thread gets the result)
__device__ float block_max(float v, SampleLds& s) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) s.redf[threadIdx.x >> 6] = v;
    __syncthreads();
    float m = s.redf[0];
    for (int w = 1; w < kST / 64; ++w) m = fmaxf(m, s.redf[w]);
    return m;
}

__device__ uint32_t block_or(uint32_t v, SampleLds& s) {
    __syncthreads();
    if (threadIdx.x == 0) s.flag = 0;
    __syncthreads();
    if (v) atomicOr(&s.flag, 1u);
    __syncthreads();
    return s.flag;
}

__device__ uint32_t block_min_u32(uint32_t v, SampleLds& s) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = min(v, (uint32_t)__shfl_xor((int)v, o, 64));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) s.redi[threadIdx.x >> 6] = v;
    __syncthreads();
    uint32_t m = s.redi[0];
    for (int w = 1; w < kST / 64; ++w) m = min(m, s.redi[w]);
    return m;
}

__device__ unsigned long long block_sum_u64(unsigned long long v, SampleLds& s) {
    __syncthreads();
    if (threadIdx.x == 0) s.acc64[0] = 0;
    __syncthreads();
    atomicAdd(&s.acc64[0], v);
    __syncthreads();
    return s.acc64[0];
}

__device__ __forceinline__ float fkey_value(uint32_t k) {
    return (k & 0x80000000u) ? __uint_as_float(k & 0x7fffffffu) : __uint_as_float(~k);
}

// Bitonic sort of N <= E * kST keys (a power of two of at least 64) in
// descending order, E consecutive keys per thread in registers: exchanges within a thread and within a wave need no
// barrier, so only the distances of 64 E and more go through LDS (10 of the 78
// steps at 4096 keys; with every step in LDS the sort took about 50 us of them).
template <int E>
__device__ void sort_block(unsigned long long* key, uint32_t N) {
    const uint32_t tid = threadIdx.x;
    unsigned long long v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = key[tid * E + e];
    for (uint32_t k = 2; k <= N; k <<= 1)
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
            if (j < (uint32_t)E) {
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    // j is 1 or 2 here; the partner is e ^ j
                    if ((e & j) == 0) {
                        const int o = j == 1 ? e + 1 : e + 2;
                        if (o < E) {
                            const unsigned long long a = v[e], b = v[o];
                            const bool down = ((tid * E + e) & k) == 0;
                            v[e] = down ? max(a, b) : min(a, b);
                            v[o] = down ? min(a, b) : max(a, b);
                        }
                    }
                }
                continue;
            }
            unsigned long long other[E];
            if (j < 64u * E) {
#pragma unroll
                for (int e = 0; e < E; ++e)
                    other[e] = (unsigned long long)__shfl_xor((long long)v[e], (int)(j / E), 64);
            } else {
                __syncthreads();
#pragma unroll
                for (int e = 0; e < E; ++e) key[tid * E + e] = v[e];
                __syncthreads();
#pragma unroll
                for (int e = 0; e < E; ++e) other[e] = key[(tid * E + e) ^ j];
            }
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const uint32_t i = tid * E + e;
                const bool larger = ((i & k) == 0) == ((i & j) == 0);
                v[e] = larger ? max(v[e], other[e]) : min(v[e], other[e]);
            }
        }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < E; ++e) key[tid * E + e] = v[e];
    __syncthreads();
}

// Sort the first n <= kExactCap keys of ex.key in descending order.
__device__ void sort_keys(ExactLds& ex, uint32_t n) {
    uint32_t N = 64;
    while (N < n) N <<= 1;
    static_assert(kExactCap == 4 * kST, "four keys per thread");
    for (uint32_t r = n + threadIdx.x; r < N; r += kST) ex.key[r] = 0;  // below every real key
    __syncthreads();
    if (N <= kST) sort_block<1>(ex.key, N);
    else if (N == 2 * kST) sort_block<2>(ex.key, N);
    else sort_block<4>(ex.key, N);
}

// sum += term[0] + term[1] + .., one after the other in f32, in whole blocks of
// 16 terms read ahead, until n terms are in (terms past the last are zeros).
// after(sum before the block, its first term) returns false to stop. Waiting
// for LDS at each term took 14 ns a term, most of a top-p row's time.
template <class After>
__device__ __forceinline__ void sequential_sum(const ExactLds& ex, float& sum, uint32_t n, After after) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    const f32x4* t = (const f32x4*)ex.term;
    f32x4 cur[4], next[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) cur[q] = t[q];
    for (uint32_t r0 = 0; r0 < n; r0 += 16) {
        const uint32_t r1 = min(r0 + 16, (uint32_t)kExactCap - 16) / 4;
#pragma unroll
        for (int q = 0; q < 4; ++q) next[q] = t[r1 + q];
        const float before = sum;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) sum += cur[q][e];
        if (!after(before, r0)) return;
#pragma unroll
        for (int q = 0; q < 4; ++q) cur[q] = next[q];
    }
}

// Length of the top-p prefix of the C sorted significant terms (below).
// Only a prefix shorter than `limit` is looked for (the caller takes the smaller of the two).
__device__ uint32_t exact_prefix_sorted(const SampleArgs& a, float F, uint32_t C, uint32_t V, uint32_t limit,
                                        ExactLds& ex) {
    const uint32_t tid = threadIdx.x;
    for (uint32_t r = tid; r < kExactCap; r += kST)
        ex.term[r] = r < C ? expf(fkey_value((uint32_t)(ex.key[r] >> 32)) - F) : 0.0f;
    __syncthreads();
    if (tid < 64) {  // one wave, every lane the same sum
        float norm = 0.0f;
        sequential_sum(ex, norm, C, [](float, uint32_t) { return true; });
        if (tid == 0) ex.norm = norm;
    }
    __syncthreads();
    const float norm = ex.norm;
    for (uint32_t r = tid; r < C; r += kST) ex.term[r] = ex.term[r] / norm;
    __syncthreads();
    if (tid < 64) {
        const uint32_t n = min(C, limit);
        float mass = 0.0f;
        uint32_t len = V;
        // the mass never falls, so a block's last value tells whether the prefix ends in it
        sequential_sum(ex, mass, n, [&](float before, uint32_t r0) {
            if (mass < a.top_p) return true;
            for (uint32_t r = r0; r < n && before < a.top_p; ++r) {
                before += ex.term[r];
                len = r + 1;
            }
            if (before < a.top_p) len = V;  // reached by terms past n only
            return false;
        });
        if (tid == 0) ex.len = len;
    }
    __syncthreads();
    return ex.len;
}

// Length of the top-p prefix as unified_sampling.rs:85-97 computes it: the
// norm is the f32 sum of exp(x - max) over the logits sorted by value desc
// (index asc), the mass adds exp(x - max) / norm in that order, and the prefix
// ends before the first logit at which the mass has reached p. C is the count
// of significant terms (see the caller); returns V when the mass never
// reaches p.
template <class ValueFn>
__device__ uint32_t exact_top_p_prefix(const SampleArgs& a, ValueFn value, float F, uint32_t C, uint32_t V,
                                       ExactLds& ex) {
    const uint32_t tid = threadIdx.x;
    __syncthreads();
    if (tid == 0) ex.n = 0;
    __syncthreads();
    for (uint32_t i = tid; i < V; i += kST) {
        const float x = value(i);
        if (expf(x - F) >= kSignificant)
            ex.key[atomicAdd(&ex.n, 1u)] = ((unsigned long long)fkey(x) << 32) | (0xffffffffu - i);
    }
    sort_keys(ex, C);
    return exact_prefix_sorted(a, F, C, V, V, ex);
}

// The row form: the whole workgroup (kST threads) samples one row.
__device__ void sample_row(const SampleArgs& a, size_t row, SampleLds& s, ExactLds& ex) {
    const uint32_t tid = threadIdx.x, V = a.vocab, words = (V + 31u) / 32u;
    const uint32_t* bm = a.bitmask ? a.bitmask + row * words : nullptr;
    const bool masked_row = bm != nullptr;
    const auto masked = [&](uint32_t i) { return masked_row && ((bm[i / 32] >> (i % 32)) & 1u) == 0; };

    // ---- pass A: finiteness; masked max and the temperature's overflow check
    const float recip = a.has_temperature ? 1.0f / a.temperature : 1.0f;
    uint32_t bad = 0, over = 0;
    float m0 = -INFINITY;
    for (uint32_t i = tid; i < V; i += kST) {
        float x = logit_at(a, row, i);
        if (!__builtin_isfinite(x)) bad = 1;
        if (masked(i)) x = -INFINITY;
        m0 = fmaxf(m0, x);
        if (__builtin_isfinite(x) && !__builtin_isfinite(x * recip)) over = 1;
    }
    if (block_or(bad, s)) {
        if (tid == 0) a.out[row] = 0xffffffffu;
        return;
    }
    const bool center = a.has_temperature && block_or(over, s);
    const float shift = center ? block_max(m0, s) : 0.0f;
    const auto value = [&](uint32_t i) {
        float x = masked(i) ? -INFINITY : logit_at(a, row, i);
        if (a.has_temperature) {
            if (center) x -= shift;
            x *= recip;
        }
        return x;
    };

    // ---- pass B: maximum and its lowest index
    float fmx = -INFINITY;
    for (uint32_t i = tid; i < V; i += kST) fmx = fmaxf(fmx, value(i));
    const float F = block_max(fmx, s);
    if (!a.seeds) {
        uint32_t best = 0xffffffffu;
        for (uint32_t i = tid; i < V; i += kST)
            if (value(i) == F) best = min(best, i);
        best = block_min_u32(best, s);
        if (tid == 0) a.out[row] = __builtin_isfinite(F) ? best : 0xffffffffu;
        return;
    }

    // ---- kept prefix length L (in sorted order)
    uint32_t L = V;
    if (a.has_top_k) L = min(L, a.top_k);
    if (a.has_min_p) {
        const float thr = F + logf(a.min_p);
        unsigned long long c = 0;
        for (uint32_t i = tid; i < V; i += kST) c += value(i) >= thr ? 1u : 0u;
        L = min(L, (uint32_t)block_sum_u64(c, s));
    }
    if (a.has_top_p && L > 1) {
        // Terms exp(x - max) below 2^-27 cannot move the reference's sequential
        // f32 sums: the norm is at least 1 (the maximum's own term), and a
        // running mass m is at least 1 / norm, so such a term (or its quotient
        // by the norm) is below half an ulp of the running value and every
        // later one is smaller still. When the terms at or above 2^-27 fit in
        // LDS, they are sorted (value desc, index asc) and both sums run in the
        // reference's order on one thread, which gives its prefix exactly.
        uint32_t cnt = 0;
        for (uint32_t i = tid; i < V; i += kST) cnt += expf(value(i) - F) >= kSignificant ? 1u : 0u;
        const uint32_t C = (uint32_t)block_sum_u64(cnt, s);
        if (C <= (uint32_t)kExactCap) {
            L = min(L, exact_top_p_prefix(a, value, F, C, V, ex));
        } else {
            const double kFix = 1099511627776.0;  // 2^40
            const auto term = [&](float x) { return (unsigned long long)((double)expf(x - F) * kFix); };
            unsigned long long z = 0;
            for (uint32_t i = tid; i < V; i += kST) z += term(value(i));
            const unsigned long long norm = block_sum_u64(z, s);
            const unsigned long long target = (unsigned long long)ceil((double)a.top_p * (double)norm);
            // radix descent: prefix of the key bits fixed so far, and the mass of
            // every logit above the current bucket
            uint32_t prefix = 0, pmask = 0;
            unsigned long long above = 0;
            bool found = false;
            for (int shiftb = 24; shiftb >= 0; shiftb -= 8) {
                __syncthreads();
                if (tid < 256) s.hist[tid] = 0;
                __syncthreads();
                for (uint32_t i = tid; i < V; i += kST) {
                    const float x = value(i);
                    const uint32_t k = fkey(x);
                    if ((k & pmask) == prefix) atomicAdd(&s.hist[(k >> shiftb) & 255u], term(x));
                }
                __syncthreads();
                if (tid == 0) {
                    uint32_t d = 256;
                    unsigned long long acc = above;
                    for (int b = 255; b >= 0; --b) {
                        if (acc + s.hist[b] >= target) {
                            d = (uint32_t)b;
                            break;
                        }
                        acc += s.hist[b];
                    }
                    s.scal[0] = d;
                    s.acc64[1] = acc;
                }
                __syncthreads();
                const uint32_t d = s.scal[0];
                if (d == 256) break;  // the whole row's mass stays below p: every logit is kept
                above = s.acc64[1];
                prefix |= d << shiftb;
                pmask |= 255u << shiftb;
                found = shiftb == 0;
            }
            if (found) {
                // logits with key == prefix all carry the same term t; the prefix
                // ends at the first of them whose addition reaches the target
                const float xk = (prefix & 0x80000000u) ? __uint_as_float(prefix & 0x7fffffffu) : __uint_as_float(~prefix);
                const unsigned long long t = term(xk);
                unsigned long long greater = 0;
                for (uint32_t i = tid; i < V; i += kST) greater += fkey(value(i)) > prefix ? 1u : 0u;
                greater = block_sum_u64(greater, s);
                const unsigned long long need = t ? (target - above + t - 1) / t : 1ull;  // ties up to the crossing one
                L = min(L, (uint32_t)min<unsigned long long>(greater + need, V));
            }
        }
    }
    L = max(L, 1u);

    // ---- the kept set: the L largest keys (ties by lower index), by radix select
    uint32_t kprefix = 0, kmask = 0, rank = L;  // rank: 1-based position wanted within the current bucket
    for (int shiftb = 24; shiftb >= 0; shiftb -= 8) {
        __syncthreads();
        if (tid < 256) s.hist[tid] = 0;
        __syncthreads();
        for (uint32_t i = tid; i < V; i += kST) {
            const uint32_t k = fkey(value(i));
            if ((k & kmask) == kprefix) atomicAdd(&s.hist[(k >> shiftb) & 255u], 1ull);
        }
        __syncthreads();
        if (tid == 0) {
            uint32_t r = rank, d = 0;
            for (int b = 255; b >= 0; --b) {
                if (s.hist[b] >= r) {
                    d = (uint32_t)b;
                    break;
                }
                r -= (uint32_t)s.hist[b];
            }
            s.scal[0] = d;
            s.scal[1] = r;
        }
        __syncthreads();
        kprefix |= s.scal[0] << shiftb;
        kmask |= 255u << shiftb;
        rank = s.scal[1];
    }
    // among logits with key == kprefix, the first `rank` by index are kept:
    // the rank-th smallest index, by radix select over the index bits
    uint32_t iprefix = 0, imask = 0;
    for (int shiftb = 24; shiftb >= 0; shiftb -= 8) {
        __syncthreads();
        if (tid < 256) s.hist[tid] = 0;
        __syncthreads();
        for (uint32_t i = tid; i < V; i += kST)
            if (fkey(value(i)) == kprefix && (i & imask) == iprefix) atomicAdd(&s.hist[(i >> shiftb) & 255u], 1ull);
        __syncthreads();
        if (tid == 0) {
            uint32_t r = rank, d = 0;
            for (uint32_t b = 0; b < 256; ++b) {
                if (s.hist[b] >= r) {
                    d = b;
                    break;
                }
                r -= (uint32_t)s.hist[b];
            }
            s.scal[0] = d;
            s.scal[1] = r;
        }
        __syncthreads();
        iprefix |= s.scal[0] << shiftb;
        imask |= 255u << shiftb;
        rank = s.scal[1];
    }

    // ---- scores of the kept logits with noise, argmax (lowest index on ties)
    const uint64_t seed = a.seeds[row];
    float best = -INFINITY;
    uint32_t bi = 0xffffffffu;
    for (uint32_t i = tid; i < V; i += kST) {
        const float x = value(i);
        const uint32_t k = fkey(x);
        const bool kept = k > kprefix || (k == kprefix && i <= iprefix);
        const float sc = (kept ? x : -INFINITY) + gumbel(seed, i, V);
        if (sc > best) {  // strided ascending: the first maximum of this thread has the lowest index
            best = sc;
            bi = i;
        }
    }
    const float gb = block_max(best, s);
    uint32_t cand = best == gb ? bi : 0xffffffffu;
    cand = block_min_u32(cand, s);
    if (tid == 0) a.out[row] = __builtin_isfinite(gb) ? cand : 0xffffffffu;
}

__global__ __launch_bounds__(kST) QMM_TWO_PER_CU void unified_sampling(SampleArgs a) {
    __shared__ SampleLds s;
    __shared__ ExactLds ex;
    sample_row(a, blockIdx.x, s, ex);
}

// ---- Split form. One workgroup reads a 151936-word row of f32 logits at the
// rate of one CU, and the row form reads it up to 16 times: 784 us for four
// rows with temperature, top-k and top-p. Here the passes over the row are
// spread over its 4096-logit pieces and only three or four remain
// (151936 words, four rows, temperature, top-k and top-p: 786 -> 26 us):
//   1. split_claim: the row takes one of kSlots scratch slots (its number is
//      kept in the row's output word until the token replaces it) and clears it;
//   2. split_max: finiteness and the masked maximum with its index;
//   3. split_hist: counts, fixed-point masses and the norm over kBins bins of
//      (max - x), whose order is the order of the logits;
//   4. split_gather: finds the bin in which the kept prefix ends and collects
//      the logits down to it;
//   5. split_select (one workgroup per row): sorts them, finds the prefix's end
//      exactly (in the row form's arithmetic: the sequential f32 sums when at
//      most kExactCap terms are significant, else the 2^-40 fixed-point
//      masses), scores the kept logits and ends the row;
//   6. split_score, only if more than kExactCap logits may be kept: scores
//      every logit of the row at or above the prefix's end;
//   7. split_end (one workgroup per row): ends greedy and scored rows.
// Greedy rows run 1, 2, 7; rows without filters 1, 2, 6, 7. The launches order
// the stages: a counter with which a row's last workgroup takes over the next
// stage needs a device-scope fence per workgroup, and those took 40 us a
// stage. Rows that this cannot take (no free slot, an overflowing
// temperature, no finite logit, a bin of more than kExactCap logits) run the
// row form in 5 or 7. A slot belongs to its row from the claim to the stage
// that ends the row, whatever streams, threads or graph replays are in flight.
// Which calls take it: sample_split (dispatch_rules.h).
constexpr uint32_t kPiece = 4096;
constexpr int kPer = kPiece / kST;       // logits per thread
constexpr uint32_t kBins = 256;
constexpr float kBinsPerUnit = 8.0f;     // bin of max - x; the last one takes everything past 31.9
constexpr uint32_t kSlots = 256;         // rows in flight (and per launch sequence)
constexpr uint32_t kSlotTag = 0xF0000000u, kNoSlot = 0xE0000000u;

enum : uint32_t { FLAG_BAD = 1, FLAG_OVERFLOW = 2 };  // a logit is not finite; the temperature overflows a finite one

struct SplitSlot {
    uint32_t flags;
    uint32_t significant, above_min_p;  // logits with a term of at least 2^-27; at or above max + ln(min_p)
    uint32_t candidates;
    unsigned long long best;       // largest fkey(value) << 32 | ~index
    unsigned long long norm;       // sum of the fixed-point terms
    unsigned long long threshold;  // split_score: the last kept (fkey, ~index)
    unsigned long long score;      // split_score: largest fkey(score) << 32 | ~index
    uint32_t hist_n[kBins];
    unsigned long long hist_m[kBins];
};

static __device__ SplitSlot split_slots[kSlots];
static __device__ unsigned long long split_cand[kSlots][kExactCap];
static __device__ uint32_t split_busy[kSlots / 32];

__global__ __launch_bounds__(256) void split_claim(uint32_t* out) {
    __shared__ uint32_t slot;
    if (threadIdx.x == 0) {
        uint32_t got = kNoSlot;
        for (uint32_t t = 0; t < kSlots; ++t) {  // at most one try per slot
            const uint32_t i = (blockIdx.x + t) % kSlots, bit = 1u << (i % 32);
            if (!(atomicOr(&split_busy[i / 32], bit) & bit)) {
                got = i;
                break;
            }
        }
        __threadfence();  // the slot's last owner is done with it
        slot = got;
        out[blockIdx.x] = got == kNoSlot ? kNoSlot : kSlotTag | got;
    }
    __syncthreads();
    if (slot == kNoSlot) return;
    uint32_t* w = (uint32_t*)&split_slots[slot];
    for (uint32_t i = threadIdx.x; i < sizeof(SplitSlot) / 4; i += 256) w[i] = 0;
}

// The row's slot, or null when it has none (its output word then holds kNoSlot) or has ended.
__device__ __forceinline__ SplitSlot* row_slot(const SampleArgs& a, size_t row) {
    const uint32_t w = a.out[row];
    return (w & 0xF0000000u) == kSlotTag && (w & 0x0FFFFFFFu) < kSlots ? &split_slots[w & 0x0FFFFFFFu] : nullptr;
}

// Whether the split form goes on with the row after split_max; F: its maximum.
__device__ __forceinline__ bool row_open(const SplitSlot* sl, float& F) {
    F = fkey_value((uint32_t)(sl->best >> 32));
    return sl->flags == 0 && __builtin_isfinite(F);
}

// The row's token; its slot is given back.
__device__ void finish_row(const SampleArgs& a, size_t row, SplitSlot* sl, uint32_t token) {
    __syncthreads();
    if (threadIdx.x == 0) {
        a.out[row] = token;
        const uint32_t i = (uint32_t)(sl - split_slots);
        __threadfence();
        atomicAnd(&split_busy[i / 32], ~(1u << (i % 32)));
    }
}

__device__ __forceinline__ uint32_t best_token(unsigned long long best) {
    return __builtin_isfinite(fkey_value((uint32_t)(best >> 32))) ? 0xffffffffu - (uint32_t)best : 0xffffffffu;
}

__device__ unsigned long long block_max_u64(unsigned long long v, unsigned long long* red) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = max(v, (unsigned long long)__shfl_xor((long long)v, o, 64));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    v = red[0];
    for (int w = 1; w < kST / 64; ++w) v = max(v, red[w]);
    return v;
}

// Raw logits of this thread's part of a piece (loaded before the first use) and their mask bits.
struct Piece {
    float x[kPer];
    uint32_t live;  // bit j: logit j is in the row
    uint32_t keep;  // bit j: not masked
    __device__ __forceinline__ Piece(const SampleArgs& a, size_t row) : live(0), keep(0) {
        const uint32_t i0 = blockIdx.x * kPiece + threadIdx.x;
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const uint32_t i = i0 + j * kST;
            const bool in = i < a.vocab;
            x[j] = load_as_f32(a.logits, a.dt, row * a.vocab + (in ? i : 0));
            uint32_t bits = 0xffffffffu;
            if (a.bitmask) bits = a.bitmask[row * ((a.vocab + 31u) / 32u) + (in ? i : 0) / 32];
            live |= (in ? 1u : 0u) << j;
            keep |= (in ? (bits >> (i % 32)) & 1u : 0u) << j;
        }
    }
    __device__ __forceinline__ uint32_t index(int j) const { return blockIdx.x * kPiece + threadIdx.x + j * kST; }
    // the row form's value(i) of a row whose temperature does not overflow
    __device__ __forceinline__ float value(const SampleArgs& a, float recip, int j) const {
        const float v = (keep >> j) & 1u ? x[j] : -INFINITY;
        return a.has_temperature ? v * recip : v;
    }
};

__global__ __launch_bounds__(kST) void split_max(SampleArgs a) {
    __shared__ unsigned long long red[kST / 64];
    __shared__ uint32_t flags;
    const size_t row = blockIdx.y;
    SplitSlot* sl = row_slot(a, row);
    if (!sl) return;
    const float recip = a.has_temperature ? 1.0f / a.temperature : 1.0f;
    const Piece p(a, row);
    if (threadIdx.x == 0) flags = 0;
    uint32_t f = 0;
    unsigned long long best = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        if (!((p.live >> j) & 1u)) continue;
        if (!__builtin_isfinite(p.x[j])) f |= FLAG_BAD;
        const float m = (p.keep >> j) & 1u ? p.x[j] : -INFINITY;
        if (__builtin_isfinite(m) && !__builtin_isfinite(m * recip)) f |= FLAG_OVERFLOW;
        best = max(best, ((unsigned long long)fkey(p.value(a, recip, j)) << 32) | (0xffffffffu - p.index(j)));
    }
    best = block_max_u64(best, red);
    if (f) atomicOr(&flags, f);
    __syncthreads();
    if (threadIdx.x == 0) {
        if (flags) atomicOr(&sl->flags, flags);
        atomicMax(&sl->best, best);
    }
}

__device__ __forceinline__ uint32_t bin_of(float F, float x) {
    return (uint32_t)fminf((F - x) * kBinsPerUnit, (float)(kBins - 1));  // F - x >= 0, +inf for masked logits
}
__device__ __forceinline__ unsigned long long mass_of(float F, float x) {
    return (unsigned long long)((double)expf(x - F) * 1099511627776.0);  // 2^40
}

// Where the kept prefix ends, from the row's histogram.
enum : uint32_t { PLAN_ROW, PLAN_EXACT, PLAN_BINS, PLAN_ONE_BIN, PLAN_ALL };
struct SplitPlan {
    uint32_t kind;   // row form; the significant terms; the bins down to `bin`; `bin` alone; every logit is kept
    uint32_t bin;
    uint32_t limit;  // prefix length by top-k and min-p
    uint32_t top_p;  // the fixed-point top-p prefix may end in the bin
    uint32_t base_n;  // logits above the collected ones, and their mass
    unsigned long long base_m, target;
};

__device__ __forceinline__ unsigned long long wave_scan(unsigned long long v) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned long long u = (unsigned long long)__shfl_up((long long)v, o, 64);
        if ((threadIdx.x & 63) >= (uint32_t)o) v += u;
    }
    return v;
}

// Called by the whole workgroup; wave 0 scans the bins, four per lane. score:
// a split_score launch follows, which makes one bin enough to collect.
__device__ void split_plan(const SampleArgs& a, const SplitSlot* sl, bool score, SplitPlan& plan) {
    static_assert(kBins == 256, "four bins per lane");
    if (threadIdx.x < 64) {
        const uint32_t lane = threadIdx.x, V = a.vocab;
        uint32_t L = V;
        if (a.has_top_k) L = min(L, a.top_k);
        if (a.has_min_p) L = min(L, sl->above_min_p);
        L = max(L, 1u);
        const bool top_p = a.has_top_p && L > 1;
        const bool exact = top_p && sl->significant <= (uint32_t)kExactCap;
        const unsigned long long target =
            top_p ? (unsigned long long)ceil((double)a.top_p * (double)sl->norm) : 0xffffffffffffffffull;
        uint32_t n[4];
        unsigned long long m[4], ns = 0, ms = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            n[j] = sl->hist_n[4 * lane + j];
            m[j] = sl->hist_m[4 * lane + j];
            ns += n[j];
            ms += m[j];
        }
        unsigned long long cn = wave_scan(ns) - ns, cm = wave_scan(ms) - ms;  // above the lane's bins
        // the first bin at which the count reaches L (L < V) or the mass the target
        uint32_t hit = 4;
        bool by_mass = false;
        unsigned long long an = 0, am = 0;  // above that bin
        uint32_t in = 0;                    // inside it
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const bool mass = top_p && cm + m[j] >= target;
            if (hit == 4 && (mass || (L < V && cn + n[j] >= L))) {
                hit = j;
                by_mass = mass;
                an = cn;
                am = cm;
                in = n[j];
            }
            cn += n[j];
            cm += m[j];
        }
        const unsigned long long lanes = __ballot(hit < 4);
        if (lane == (lanes ? (uint32_t)__ffsll((long long)lanes) - 1 : 0u)) {
            plan.limit = L;
            plan.bin = 4 * lane + hit;
            plan.top_p = by_mass ? 1u : 0u;
            plan.base_n = 0;
            plan.base_m = 0;
            plan.target = target;
            if (exact) {
                plan.kind = PLAN_EXACT;
            } else if (!lanes) {
                plan.kind = PLAN_ALL;
            } else if (an + in <= (unsigned long long)(score ? kST : kExactCap)) {
                plan.kind = PLAN_BINS;
            } else if (in <= (uint32_t)kExactCap) {
                plan.kind = PLAN_ONE_BIN;
                plan.base_n = (uint32_t)an;
                plan.base_m = am;
            } else {
                plan.kind = PLAN_ROW;
            }
        }
    }
    __syncthreads();
}

__global__ __launch_bounds__(kST) void split_hist(SampleArgs a) {
    __shared__ uint32_t hn[kBins];
    __shared__ unsigned long long hm[kBins];
    __shared__ unsigned long long tot[3];
    const size_t row = blockIdx.y;
    SplitSlot* sl = row_slot(a, row);
    float F;
    if (!sl || !row_open(sl, F)) return;
    const uint32_t tid = threadIdx.x;
    const float recip = a.has_temperature ? 1.0f / a.temperature : 1.0f;
    const Piece p(a, row);
    if (tid < kBins) {
        hn[tid] = 0;
        hm[tid] = 0;
    }
    if (tid < 3) tot[tid] = 0;
    __syncthreads();
    const float thr = a.has_min_p ? F + logf(a.min_p) : 0.0f;
    uint32_t sig = 0, abv = 0;
    unsigned long long norm = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        if (!((p.live >> j) & 1u)) continue;
        const float x = p.value(a, recip, j);
        const uint32_t b = bin_of(F, x);
        const unsigned long long t = mass_of(F, x);
        if (expf(x - F) >= kSignificant) ++sig;
        if (x >= thr) ++abv;
        norm += t;
        atomicAdd(&hn[b], 1u);
        if (t) atomicAdd(&hm[b], t);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        sig += (uint32_t)__shfl_xor((int)sig, o, 64);
        abv += (uint32_t)__shfl_xor((int)abv, o, 64);
        norm += (unsigned long long)__shfl_xor((long long)norm, o, 64);
    }
    if ((tid & 63) == 0) {
        atomicAdd(&tot[0], norm);
        atomicAdd(&tot[1], (unsigned long long)sig);
        atomicAdd(&tot[2], (unsigned long long)abv);
    }
    __syncthreads();
    if (tid < kBins) {
        if (hn[tid]) atomicAdd(&sl->hist_n[tid], hn[tid]);
        if (hm[tid]) atomicAdd(&sl->hist_m[tid], hm[tid]);
    }
    if (tid == 0) {
        atomicAdd(&sl->norm, tot[0]);
        atomicAdd(&sl->significant, (uint32_t)tot[1]);
        atomicAdd(&sl->above_min_p, (uint32_t)tot[2]);
    }
}

__global__ __launch_bounds__(kST) void split_gather(SampleArgs a, uint32_t score) {
    __shared__ SplitPlan plan;
    __shared__ uint32_t count, base;
    const size_t row = blockIdx.y;
    const uint32_t tid = threadIdx.x;
    SplitSlot* sl = row_slot(a, row);
    float F;
    if (!sl || !row_open(sl, F)) return;
    const Piece p(a, row);
    if (tid == 0) count = 0;
    split_plan(a, sl, score != 0, plan);
    const uint32_t kind = plan.kind, bin = plan.bin;
    if (kind == PLAN_ROW || kind == PLAN_ALL) return;
    unsigned long long* cand = split_cand[sl - split_slots];
    const float recip = a.has_temperature ? 1.0f / a.temperature : 1.0f;
    uint32_t at[kPer], in = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        if (!((p.live >> j) & 1u)) continue;
        const float x = p.value(a, recip, j);
        const uint32_t b = bin_of(F, x);
        const bool c = kind == PLAN_EXACT ? expf(x - F) >= kSignificant : kind == PLAN_BINS ? b <= bin : b == bin;
        if (c) {
            at[j] = atomicAdd(&count, 1u);
            in |= 1u << j;
        }
    }
    __syncthreads();
    if (tid == 0 && count) base = atomicAdd(&sl->candidates, count);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kPer; ++j)
        if ((in >> j) & 1u) {
            const uint32_t o = base + at[j];
            if (o < (uint32_t)kExactCap)  // the histogram has counted at most kExactCap
                cand[o] = ((unsigned long long)fkey(p.value(a, recip, j)) << 32) | (0xffffffffu - p.index(j));
        }
}

// The prefix's length among the n sorted candidates of a fixed-point top-p
// row: one past the first at which the mass reaches the target (wave 0).
__device__ uint32_t fixed_prefix(const SplitPlan& plan, const ExactLds& ex, float F, uint32_t n, SampleLds& s) {
    if (threadIdx.x < 64) {
        unsigned long long acc = plan.base_m;
        uint32_t at = n;
        for (uint32_t r0 = 0; r0 < n && at == n; r0 += 64) {
            const uint32_t r = r0 + threadIdx.x;
            const unsigned long long t =
                wave_scan(r < n ? mass_of(F, fkey_value((uint32_t)(ex.key[r] >> 32))) : 0ull);
            const unsigned long long hit = __ballot(r < n && acc + t >= plan.target);
            if (hit) at = r0 + (uint32_t)__ffsll((long long)hit);
            acc += (unsigned long long)__shfl((long long)t, 63, 64);
        }
        if (threadIdx.x == 0) s.scal[0] = at;
    }
    __syncthreads();
    return s.scal[0];
}

// score: a split_score launch follows.
__global__ __launch_bounds__(kST) void split_select(SampleArgs a, uint32_t score) {
    __shared__ SampleLds s;
    __shared__ ExactLds ex;
    __shared__ SplitPlan plan;
    __shared__ unsigned long long red[kST / 64];
    const size_t row = blockIdx.x;
    const uint32_t tid = threadIdx.x, V = a.vocab;
    SplitSlot* sl = row_slot(a, row);
    float F;
    if (!sl || !row_open(sl, F)) {
        sample_row(a, row, s, ex);
        if (sl) finish_row(a, row, sl, a.out[row]);
        return;
    }
    split_plan(a, sl, score != 0, plan);
    uint32_t kind = plan.kind;
    uint32_t n = 0, kept = 0;  // candidates; those kept
    if (kind == PLAN_EXACT || kind == PLAN_BINS || kind == PLAN_ONE_BIN) {
        const unsigned long long* cand = split_cand[sl - split_slots];
        n = min(sl->candidates, (uint32_t)kExactCap);
        for (uint32_t r = tid; r < n; r += kST) ex.key[r] = cand[r];
        sort_keys(ex, n);
        uint32_t L = plan.limit;
        if (kind == PLAN_EXACT)
            L = min(L, exact_prefix_sorted(a, F, n, V, L, ex));
        else if (plan.top_p)
            L = min(L, plan.base_n + fixed_prefix(plan, ex, F, n, s));
        L = max(L, 1u);
        kept = L - plan.base_n;  // base_n < L: the prefix ends among the candidates
        // past the significant terms: the whole row, or (rare) some count of it
        if (kind == PLAN_EXACT && kept > n) kind = L >= V ? PLAN_ALL : PLAN_ROW;
    }
    if (kind == PLAN_ROW || ((kind == PLAN_ALL || kind == PLAN_ONE_BIN) && !score)) {
        sample_row(a, row, s, ex);
        finish_row(a, row, sl, a.out[row]);
        return;
    }
    if (kind == PLAN_ALL || kind == PLAN_ONE_BIN) {
        if (tid == 0) sl->threshold = kind == PLAN_ALL ? 0 : ex.key[kept - 1];
        return;
    }
    const uint64_t seed = a.seeds[row];
    unsigned long long best = 0;
    for (uint32_t r = tid; r < kept; r += kST) {
        const unsigned long long k = ex.key[r];
        const float sc = fkey_value((uint32_t)(k >> 32)) + gumbel(seed, 0xffffffffu - (uint32_t)k, V);
        best = max(best, ((unsigned long long)fkey(sc) << 32) | (uint32_t)k);
    }
    best = block_max_u64(best, red);
    finish_row(a, row, sl, best_token(best));
}

__global__ __launch_bounds__(kST) void split_score(SampleArgs a) {
    __shared__ unsigned long long red[kST / 64];
    const size_t row = blockIdx.y;
    SplitSlot* sl = row_slot(a, row);
    float F;
    if (!sl || !row_open(sl, F)) return;
    const float recip = a.has_temperature ? 1.0f / a.temperature : 1.0f;
    const unsigned long long threshold = sl->threshold;
    const uint64_t seed = a.seeds[row];
    const Piece p(a, row);
    unsigned long long best = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        if (!((p.live >> j) & 1u)) continue;
        const float x = p.value(a, recip, j);
        const uint32_t i = p.index(j);
        if ((((unsigned long long)fkey(x) << 32) | (0xffffffffu - i)) < threshold) continue;
        best = max(best, ((unsigned long long)fkey(x + gumbel(seed, i, a.vocab)) << 32) | (0xffffffffu - i));
    }
    best = block_max_u64(best, red);
    if (threadIdx.x == 0) atomicMax(&sl->score, best);
}

__global__ __launch_bounds__(kST) void split_end(SampleArgs a) {
    __shared__ SampleLds s;
    __shared__ ExactLds ex;
    const size_t row = blockIdx.x;
    SplitSlot* sl = row_slot(a, row);
    if (!sl) {
        if (a.out[row] == kNoSlot) sample_row(a, row, s, ex);  // else split_select has ended the row
        return;
    }
    float F;
    if (!row_open(sl, F)) {
        sample_row(a, row, s, ex);
        finish_row(a, row, sl, a.out[row]);
        return;
    }
    finish_row(a, row, sl, best_token(a.seeds ? sl->score : sl->best));
}

stark_qmm_status launch_split(SampleArgs a, uint32_t batch, hipStream_t stream) {
    const uint32_t words = (a.vocab + 31u) / 32u;
    const bool filters = a.has_top_k || a.has_top_p || a.has_min_p;
    // split_select ends every row of at most as many kept logits as it has threads (with more, a row whose
    // bins hold over kExactCap would fall to the row form: top-k 4096 of 8192, 1.4 times its time)
    const bool few = a.has_top_k && a.top_k <= (uint32_t)kST;
    for (uint32_t r0 = 0; r0 < batch; r0 += kSlots) {
        const uint32_t rows = std::min(kSlots, batch - r0);
        SampleArgs b = a;
        b.logits = (const uint8_t*)a.logits + (size_t)r0 * a.vocab * (a.dt == STARK_QMM_F32 ? 4 : 2);
        b.out = a.out + r0;
        b.seeds = a.seeds ? a.seeds + r0 : nullptr;
        b.bitmask = a.bitmask ? a.bitmask + (size_t)r0 * words : nullptr;
        const dim3 grid((a.vocab + kPiece - 1) / kPiece, rows);
        hipLaunchKernelGGL(split_claim, dim3(rows), dim3(256), 0, stream, b.out);
        hipLaunchKernelGGL(split_max, grid, dim3(kST), 0, stream, b);
        if (a.seeds && filters) {
            hipLaunchKernelGGL(split_hist, grid, dim3(kST), 0, stream, b);
            hipLaunchKernelGGL(split_gather, grid, dim3(kST), 0, stream, b, few ? 0u : 1u);
            hipLaunchKernelGGL(split_select, dim3(rows), dim3(kST), 0, stream, b, few ? 0u : 1u);
        }
        if (a.seeds && !(filters && few)) hipLaunchKernelGGL(split_score, grid, dim3(kST), 0, stream, b);
        if (!(a.seeds && filters && few)) hipLaunchKernelGGL(split_end, dim3(rows), dim3(kST), 0, stream, b);
        QMM_HIP_CHECK(hipGetLastError());
    }
    return STARK_QMM_OK;
}

}  // namespace
}  // namespace qmm

using namespace qmm;

extern "C" {

stark_qmm_status stark_qmm_unified_sampling(const stark_qmm_sampling_args* args, void* stream) {
    if (!args) return STARK_QMM_INVALID_ARGUMENT;
    if (args->struct_size != sizeof(stark_qmm_sampling_args)) return STARK_QMM_ABI_MISMATCH;
    const stark_qmm_sampling_args& x = *args;
    if (x.data_type != STARK_QMM_F32 && x.data_type != STARK_QMM_BF16) return STARK_QMM_UNSUPPORTED_DATA_TYPE;
    // SamplingMethod::validate (src/encodable_block/sampling/mod.rs:73-101)
    if (x.vocab_size == 0 || !x.logits || !x.output) return STARK_QMM_INVALID_ARGUMENT;
    if (x.has_temperature &&
        (!std::isfinite(x.temperature) || x.temperature <= 0.0f || !std::isfinite(1.0f / x.temperature)))
        return STARK_QMM_INVALID_ARGUMENT;
    if (x.has_top_k && (x.top_k == 0 || x.top_k > x.vocab_size)) return STARK_QMM_INVALID_ARGUMENT;
    if (x.has_top_p && (!std::isfinite(x.top_p) || x.top_p <= 0.0f || x.top_p > 1.0f)) return STARK_QMM_INVALID_ARGUMENT;
    if (x.has_min_p && (!std::isfinite(x.min_p) || x.min_p < 0.0f || x.min_p > 1.0f)) return STARK_QMM_INVALID_ARGUMENT;
    if (x.batch_size == 0) return STARK_QMM_OK;
    SampleArgs a{};
    a.logits = x.logits;
    a.out = x.output;
    a.seeds = x.seeds;
    a.bitmask = x.bitmask;
    a.vocab = x.vocab_size;
    a.dt = x.data_type;
    a.has_temperature = x.has_temperature;
    a.temperature = x.temperature;
    a.has_top_k = x.has_top_k && x.top_k < x.vocab_size;  // as many as there are: nothing is filtered
    a.top_k = x.top_k;
    a.has_top_p = x.has_top_p;
    a.top_p = x.top_p;
    a.has_min_p = x.has_min_p;
    a.min_p = x.min_p;
    const bool filters = a.has_top_k || a.has_top_p || a.has_min_p;
    if (sample_split(x.vocab_size, x.batch_size, x.seeds != nullptr, filters) && x.vocab_size < kNoSlot)
        return launch_split(a, x.batch_size, (hipStream_t)stream);
    hipLaunchKernelGGL(unified_sampling, dim3(x.batch_size), dim3(kST), 0, (hipStream_t)stream, a);
    QMM_HIP_CHECK(hipGetLastError());
    return STARK_QMM_OK;
}

}  // extern "C"
