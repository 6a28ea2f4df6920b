// Products with int8 activations (A8W4, A8W8) on the int8 matrix cores, weight
// group 64 and activation groups of 64 or 128: the weights stream from global
// memory straight into the B operand and only the activations go through LDS.
//
// Per 64-value group  acc += s_a * (s * C + sum q_a * bias_term), C = sum q_a q_w
// exact in one v_mfma_i32_16x16x64_i8. More than 16 rows: as qgemm_a8, the terms
// (s_a * s) * C and, with a chunk's two groups in one v_mfma_f32_16x16x4_f32,
// (s_a * sum q_a) * bias_term; 8-bit codes enter as q - 128, with 128 s added to
// the bias term. Up to 16 rows (they ran on qmv_a8, whose 64 partial sums a row
// round less than eight waves' in that form, 0.7-0.9e-7 from the 64-bit product
// against 1.2-1.9e-7): 4-bit codes are centred too (as 16 (q - 8), from the same
// two masks; the bias term is then small), a group's two terms are added before
// they join the sum, and the chunk's two groups have a sum each: 0.6-0.9e-7.
//
// A lane loads 16 bytes of its weight row. For 4-bit codes these are 32 values
// and v_permlane32_swap sorts the words so that all four lane groups of an
// MFMA hold codes of one group; the nibbles split into bytes in the
// grouped-by-nibble order of the activation codes (sequential ones are
// permuted as they are staged). The activations need no conversion: 16-byte
// pieces are copied into LDS ([piece in MFMA order][row]), their group sums
// taken with v_dot4 on the way.
//
// A workgroup of eight waves is KW waves along K (each takes the 128-value
// chunks of K in turn, and the sums meet in LDS) times 8 / KW along N, 32
// columns each, for up to 16 MT rows. Few rows need all waves along K, since
// there are few columns to spread over the chip; many rows need few, since
// every workgroup copies its rows' activations. What bounds it: at few rows the
// weights (one row, N 24576, K 4096: 3.7 TB/s); at many the scaling, three
// vector operations per output and group (conversion, product of the scales,
// fma) against 16 cycles of matrix work per 16 x 16 x 64.
// Measured, us before and now (before: qmv_a8 up to 16 rows, qgemm_a8's 128 x 128
// tiles above; 4-bit, replays of a graph over copies of the weights):
//   rows                    1          16         64          256         512
//   N 24576, K  4096   27.4 17.9  93.8 17.6   86.4 36.8  100.3 94.6  134.8 (GEMM)
//   N  4096, K 12288   15.9 15.2  58.0 16.1  232.2 25.4  230.1 56.0  230.3 93.7
//   N  7424, K  1920    7.1  5.5  23.8  5.5   47.0 10.2   40.2 22.6   41.0 35.4
// (in the int8 MLP of 512 rows, between other kernels, the second one takes 108.7.)
#include "qmm_common.h"
#include "code_layout.h"

namespace qmm {
namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 8, kThreads = 64 * kWaves;

template <int MT, int KW>
struct A8Lds {
    static constexpr int R = 16 * MT, RP = R + 1;  // a row's staging stores fall on distinct banks
    static constexpr int kPieces = 8 * KW;         // 16-byte pieces of a row's pass
    static constexpr int kCols = 32 * (kWaves / KW);
    union {
        u32x4 xa[2][kPieces * RP];          // activation codes, [piece in MFMA order][row]
        float red[KW > 1 ? KW * R * kCols : 1];  // the K waves' sums, [wave][row][column]
    };
    alignas(16) float sa[2][2 * KW][R];  // activation scale per group and row
    alignas(16) float ur[2][2 * KW][R];  // sum of the group's codes; more than 16 rows: times the scale
    uint32_t pl[2][kThreads];            // raw scale | bias << 16, [group][column]
};

template <int BITS, int MT, int KW, bool BF>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4))) void qmv_a8_dense(
    A8Batch batch) {
    (void)batch;
    using L = A8Lds<MT, KW>;
    __shared__ L lds;
    constexpr int R = L::R, RP = L::RP, WL = BITS / 4, XI = R * L::kPieces / kThreads;  // pieces per thread
    constexpr uint32_t kPass = 128 * KW, kGroups = 2 * KW, kCols = L::kCols;
    static_assert(XI >= 1, "every thread stages a piece");
    const A8Batch* kb = (const A8Batch*)__builtin_amdgcn_kernarg_segment_ptr();
    uint32_t oi = 0;
    while (oi + 1 < kb->count && blockIdx.x >= kb->op[oi + 1].block_begin) ++oi;
    const AffineOp& op = kb->op[oi];
    const A8Operand& ao = kb->a[oi];
    const uint32_t M = op.m, N = op.n, K = op.k, G = K / 64;
    // column tiles of a row block are neighbours: those of one column tile share an XCD when their number is a
    // multiple of 8
    const uint32_t ct = (N + kCols - 1) / kCols, t0 = blockIdx.x - op.block_begin;
    const uint32_t n0 = t0 % ct * kCols, m0 = t0 / ct * R;
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t col = lane & 15, kq = lane >> 4, kw = wave % KW, nw = wave / KW;
    const uint32_t passes = (K + kPass - 1) / kPass;
    const size_t row_bytes = (size_t)K * BITS / 8;
    const bool biased = op.corr_kind == STARK_QMM_CORRECTION_BIASES, sg = (op.flags & FLAG_SIGNED) != 0;
    constexpr bool kFew = MT == 1;            // at most 16 rows
    constexpr bool kCentred = kFew || BITS == 8;  // codes enter less 2^(BITS - 1), 4-bit ones times 16
    const uint32_t flip = BITS == 4 ? (sg != kCentred ? 0x88888888u : 0u) : (sg ? 0u : 0x80808080u);
    // activation codes are staged in the order the weights' bytes come in
    const bool permute = BITS == 4 ? ao.grouped == 0 : ao.grouped != 0;

    const uint8_t* cp[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) cp[t] = op.codes + (size_t)min(n0 + 32 * nw + 16 * t + col, N - 1) * row_bytes;
    const uint32_t pg = op.os == 1 ? tid / kCols : tid % kGroups;
    const uint32_t pc = op.os == 1 ? tid % kCols : tid / kGroups;
    const size_t po = (size_t)min(n0 + pc, N - 1) * op.os;
    const uint16_t* scales = (const uint16_t*)op.scales;
    const uint16_t* corr = biased ? (const uint16_t*)op.corr : scales;

    // staging: piece tid % kPieces of rows tid / kPieces + (512 / kPieces) i; rows past M repeat the last
    const uint32_t piece = tid % L::kPieces, srow = tid / L::kPieces;
    constexpr uint32_t rstep = kThreads / L::kPieces;
    const uint32_t j = piece & 3;
    const uint32_t pos = (piece & ~3u) + (BITS == 4 ? (j >> 1) | ((j & 1) << 1) : j);
    const uint32_t lag = 31 - __builtin_clz(ao.group), GA = K >> lag;

    u32x4 wv[2][2][WL];  // [set][tile][16-byte load]
    u32x4 xv[XI];
    float sv[XI];
    uint32_t ps, pb;
    const auto load_xp = [&](uint32_t p) {
        const uint32_t k = p * kPass + piece * 16, kc = k < K ? k : 0;
#pragma unroll
        for (int i = 0; i < XI; ++i) {
            const size_t r = min(m0 + srow + rstep * i, M - 1);
            xv[i] = *(const u32x4*)(ao.codes + r * K + kc);
            sv[i] = ao.scales[r * GA + (kc >> lag)];
        }
        const size_t o = po + (size_t)min(p * kGroups + pg, G - 1) * op.gs;
        ps = scales[o];
        pb = corr[o];
    };
    const auto load_w = [&](uint32_t p, u32x4 (&w)[2][WL]) {
        const uint32_t k = p * kPass + kw * 128;
#pragma unroll
        for (int h = 0; h < WL; ++h) {
            const uint32_t o = code_offset<BITS>(k, h, kq, K);
            w[0][h] = *(const u32x4*)(cp[0] + o);
            w[1][h] = *(const u32x4*)(cp[1] + o);
        }
    };
    const auto stage = [&](uint32_t p, int buf) {
        const bool in = p * kPass + piece * 16 < K;
#pragma unroll
        for (int i = 0; i < XI; ++i) {
            u32x4 x = xv[i];
            if (!in) x = u32x4{0, 0, 0, 0};
            if (permute) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint32_t a = x[2 * h], b = x[2 * h + 1];
                    x[2 * h] = __builtin_amdgcn_perm(b, a, BITS == 4 ? 0x06040200u : 0x05010400u);
                    x[2 * h + 1] = __builtin_amdgcn_perm(b, a, BITS == 4 ? 0x07050301u : 0x07030602u);
                }
            }
            const uint32_t r = srow + rstep * i;
            lds.xa[buf][pos * RP + r] = x;
            int sum = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) sum = __builtin_amdgcn_sdot4((int)x[q], 0x01010101, sum, false);
            sum += (int)dpp_u32<DPP_XOR1>((uint32_t)sum);
            sum += (int)dpp_u32<DPP_XOR2>((uint32_t)sum);
            if (j == 0) {
                lds.sa[buf][piece >> 2][r] = sv[i];
                lds.ur[buf][piece >> 2][r] = kFew ? (float)sum : sv[i] * (float)sum;
            }
        }
        lds.pl[buf][pg * kCols + pc] = ps | (pb << 16);
    };

    f32x4 acc[MT][2], odd[2];  // odd (at most 16 rows): the sums of the chunks' second groups
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m][0] = acc[m][1] = f32x4{0, 0, 0, 0};
    odd[0] = odd[1] = f32x4{0, 0, 0, 0};
    const auto compute = [&](int buf, u32x4 (&w)[2][WL], uint32_t ng) {
        if (ng == 0) return;
        const uint32_t* pl = &lds.pl[buf][2 * kw * kCols + 32 * nw + col];
        u32x4 b[2][2];  // [tile][group] B operands
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            if (BITS == 4) {
                const auto s0 = __builtin_amdgcn_permlane32_swap(w[t][0][0], w[t][0][2], false, false);
                const auto s1 = __builtin_amdgcn_permlane32_swap(w[t][0][1], w[t][0][3], false, false);
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    const uint32_t a = s0[g] ^ flip, c = s1[g] ^ flip;
                    if (kFew) b[t][g] = u32x4{(a << 4) & 0xF0F0F0F0u, a & 0xF0F0F0F0u, (c << 4) & 0xF0F0F0F0u, c & 0xF0F0F0F0u};
                    else b[t][g] = u32x4{a & 0x0F0F0F0Fu, (a >> 4) & 0x0F0F0F0Fu, c & 0x0F0F0F0Fu, (c >> 4) & 0x0F0F0F0Fu};
                }
            } else {
#pragma unroll
                for (int g = 0; g < 2; ++g)
#pragma unroll
                    for (int q = 0; q < 4; ++q) b[t][g][q] = w[t][g % WL][q] ^ flip;
            }
        }
        if constexpr (kFew) {
            constexpr float unit = BITS == 4 ? 0.0625f : 1.0f, mid = (float)(1 << (BITS - 1));
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                if ((uint32_t)g >= ng) break;
                const i32x4 a = __builtin_bit_cast(i32x4, lds.xa[buf][(8 * kw + 4 * g + kq) * RP + col]);
                const f32x4 sa = *(const f32x4*)&lds.sa[buf][2 * kw + g][4 * kq];
                const f32x4 us = *(const f32x4*)&lds.ur[buf][2 * kw + g][4 * kq];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const uint32_t q = pl[g * kCols + 16 * t];
                    const float s = BF ? __uint_as_float(q << 16) : f16_bits_to_f32(q & 0xffffu);
                    const float bi = BF ? __uint_as_float(q & 0xffff0000u) : f16_bits_to_f32(q >> 16);
                    const float bt = biased ? fmaf(mid, s, bi) : 0.0f, sc = unit * s;
                    const i32x4 c = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, __builtin_bit_cast(i32x4, b[t][g]),
                                                                         i32x4{0, 0, 0, 0}, 0, 0, 0);
                    f32x4& to = g == 0 ? acc[0][t] : odd[t];
#pragma unroll
                    for (int e = 0; e < 4; ++e) to[e] = fmaf(sa[e], fmaf(sc, (float)c[e], bt * us[e]), to[e]);
                    asm volatile("" : "+v"(to));
                }
            }
            return;
        }
        // (group by group: with both groups' products in flight the register
        // budget of two workgroups per CU spills, 24 -> 31 us at 32 rows)
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            if ((uint32_t)g >= ng) break;
            float sc[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const uint32_t q = pl[g * kCols + 16 * t];
                sc[t] = BF ? __uint_as_float(q << 16) : f16_bits_to_f32(q & 0xffffu);
            }
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const i32x4 a = __builtin_bit_cast(i32x4, lds.xa[buf][(8 * kw + 4 * g + kq) * RP + 16 * m + col]);
                const f32x4 sa = *(const f32x4*)&lds.sa[buf][2 * kw + g][16 * m + 4 * kq];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const i32x4 c = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, __builtin_bit_cast(i32x4, b[t][g]),
                                                                         i32x4{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[m][t][e] = fmaf(sa[e] * sc[t], (float)c[e], acc[m][t][e]);
                    // keeps the scaling here: moved past the staging and the barrier, it would hold every block's sums
                    asm volatile("" : "+v"(acc[m][t]));
                }
            }
        }
        // the bias terms of the chunk's groups (k entries 0 and 1 of a rank-4 product)
        const bool on = kq < ng;
        const uint32_t gq = kq & 1;
        float bt[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const uint32_t q = pl[gq * kCols + 16 * t];
            const float s = BF ? __uint_as_float(q << 16) : f16_bits_to_f32(q & 0xffffu);
            const float bi = BF ? __uint_as_float(q & 0xffff0000u) : f16_bits_to_f32(q >> 16);
            const float v = (biased ? bi : -(float)(1 << (BITS - 1)) * s) + (BITS == 8 ? 128.0f * s : 0.0f);
            bt[t] = on ? v : 0.0f;
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const float u = on ? lds.ur[buf][2 * kw + gq][16 * m + col] : 0.0f;
#pragma unroll
            for (int t = 0; t < 2; ++t) acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(u, bt[t], acc[m][t], 0, 0, 0);
        }
    };
    const auto groups = [&](uint32_t p) -> uint32_t {
        const uint32_t g = p * kGroups + 2 * kw;
        return g + 2 <= G ? 2u : g < G ? 1u : 0u;
    };

    // Pass p computes from LDS buffer p % 2 and code set p % 2; the prefetches
    // past the last pass are clamped to it (their buffers are not computed).
    const uint32_t last = passes - 1;
    load_xp(0);
    load_w(0, wv[0]);
    stage(0, 0);
    load_xp(min(1u, last));
    load_w(min(1u, last), wv[1]);
    lds_barrier();
    uint32_t p = 0;
    for (; p + 2 <= last; p += 2) {
        compute(0, wv[0], 2);
        stage(p + 1, 1);
        load_xp(p + 2);
        load_w(p + 2, wv[0]);
        lds_barrier();
        compute(1, wv[1], 2);
        stage(p + 2, 0);
        load_xp(min(p + 3, last));
        load_w(min(p + 3, last), wv[1]);
        lds_barrier();
    }
    compute(0, wv[0], p == last ? groups(p) : 2u);
    if (p < last) {
        stage(p + 1, 1);
        lds_barrier();
        compute(1, wv[1], groups(p + 1));
    }

    const auto store = [&](uint32_t r, uint32_t n, float v) {
        if (m0 + r >= M || n >= N) return;
        const size_t o = (size_t)(m0 + r) * N + n;
        v *= op.ab_scale;
        if (op.flags & FLAG_ACCUMULATE) v += load_as_f32(op.d, op.d_dt, o);
        if (op.bias) v += load_as_f32(op.bias, op.w_dt, n);
        if (op.flags & FLAG_SOFT_CAP) v = op.soft_cap * tanhf(v / op.soft_cap);
        store_from_f32(op.d, op.d_dt, o, v);
    };
    if constexpr (KW == 1) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    store(16 * m + 4 * kq + e, n0 + 32 * nw + 16 * t + col, acc[m][t][e]);
    } else {
        if (kFew) {
            acc[0][0] += odd[0];
            acc[0][1] += odd[1];
        }
        lds_barrier();  // the activations are read: their LDS takes the sums
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    lds.red[(kw * R + 16 * m + 4 * kq + e) * kCols + 32 * nw + 16 * t + col] = acc[m][t][e];
        lds_barrier();
        const uint32_t rows = min((uint32_t)R, M - m0);
        for (uint32_t q = tid; q < rows * kCols; q += kThreads) {
            float v = lds.red[q] + lds.red[R * kCols + q];
            if constexpr (KW >= 4) v += lds.red[2 * R * kCols + q] + lds.red[3 * R * kCols + q];
            if constexpr (KW == 8)
                v += (lds.red[4 * R * kCols + q] + lds.red[5 * R * kCols + q]) +
                     (lds.red[6 * R * kCols + q] + lds.red[7 * R * kCols + q]);
            store(q / kCols, n0 + q % kCols, v);
        }
    }
}

template <int MT, int KW>
void launch_shape(const A8Batch& b, int bits, uint32_t tiles, hipStream_t stream) {
    const bool bf = b.op[0].w_dt == STARK_QMM_BF16;
    const dim3 grid(tiles);
    if (bits == 4 && bf) hipLaunchKernelGGL((qmv_a8_dense<4, MT, KW, true>), grid, dim3(kThreads), 0, stream, b);
    else if (bits == 4) hipLaunchKernelGGL((qmv_a8_dense<4, MT, KW, false>), grid, dim3(kThreads), 0, stream, b);
    else if (bf) hipLaunchKernelGGL((qmv_a8_dense<8, MT, KW, true>), grid, dim3(kThreads), 0, stream, b);
    else hipLaunchKernelGGL((qmv_a8_dense<8, MT, KW, false>), grid, dim3(kThreads), 0, stream, b);
}

}  // namespace

bool a8_dense_eligible(const AffineOp& o, const A8Operand& a, int bits) {
    return (bits == 4 || bits == 8) && !o.gather && o.m >= 1 && o.n >= 1 && o.group_size == 64 && a.group >= 64 &&
           o.k != 0 && o.k % 64 == 0 && o.k % a.group == 0 && o.corr_kind != STARK_QMM_CORRECTION_ZERO_POINTS &&
           (o.w_dt == STARK_QMM_BF16 || o.w_dt == STARK_QMM_F16) &&
           (((uintptr_t)o.codes | (uintptr_t)a.codes) & 15) == 0 && ((uintptr_t)a.scales & 3) == 0 &&
           (((uintptr_t)o.scales | (uintptr_t)o.corr) & 1) == 0;
}

// ops: all a8_dense_eligible for `bits`, of one plane type. few: products that the GEMM does not take.
stark_qmm_status launch_a8_dense(const AffineOp* ops, const A8Operand* as, uint32_t count, int bits, bool few,
                                 hipStream_t stream) {
    if (count == 0) return STARK_QMM_OK;
    if (count > (uint32_t)kMaxBatchOps) return STARK_QMM_UNSUPPORTED;
    int dev = 0, cus = 0;
    QMM_HIP_CHECK(hipGetDevice(&dev));
    QMM_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const int best = a8_shape(ops, count, few, (uint32_t)cus);
    A8Batch b{};
    uint64_t tiles = 0;
    for (uint32_t i = 0; i < count; ++i) {
        b.op[i] = ops[i];
        b.a[i] = as[i];
        b.op[i].block_begin = (uint32_t)tiles;
        tiles += a8_shape_tiles(kA8Shapes[best], ops[i]);
        if (tiles > 0x7fffffffu) return STARK_QMM_UNSUPPORTED;
    }
    b.count = count;
    switch (best) {
    case 0: launch_shape<1, 8>(b, bits, (uint32_t)tiles, stream); break;
    case 1: launch_shape<2, 8>(b, bits, (uint32_t)tiles, stream); break;
    case 2: launch_shape<2, 4>(b, bits, (uint32_t)tiles, stream); break;
    case 3: launch_shape<2, 2>(b, bits, (uint32_t)tiles, stream); break;
    case 4: launch_shape<4, 2>(b, bits, (uint32_t)tiles, stream); break;
    default: launch_shape<4, 1>(b, bits, (uint32_t)tiles, stream); break;
    }
    QMM_HIP_CHECK(hipGetLastError());
    return STARK_QMM_OK;
}

}  // namespace qmm
