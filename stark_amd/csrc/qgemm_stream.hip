// Prompt products of 17 to 128 rows, group 64: D = X * W^T with every weight
// rounded once to bf16(s * q + bias_term), the weights of qgemm_mfma, and f32
// sums. qgemm_mfma walks K in 64-value steps of tiles 64 columns wide, so a
// product of few rows costs its serial K loop on few workgroups.
//
// A workgroup is four waves along K times two along N. A lane loads the 16 codes
// of one 64-value group that its B operands take (8 or 16 bytes, straight to
// registers), dequantises them there and uses them for all of the workgroup's
// rows (16 MT, at most 64); only the activations go through LDS, copied as they
// are, [8-value piece in MFMA order][row], double-buffered. The waves' sums meet
// in LDS at the end. K splits in the same way in every shape, so a sum is the
// same in each of them.
// Where the registers allow (PIPE), the operands of the next pass are
// dequantised beside the matrix products of this one.
//
// What bounds it: the phases of a 256-value pass (dequantisation, LDS reads,
// matrix products, staging), about 0.6 us a pass at 32 rows and 1.0 at 64 on one
// workgroup, whatever the prefetch distance: two passes of activations and four
// of codes in flight measured the same. 128-row workgroups (one per CU), eight
// waves along K, and 128 columns a workgroup were slower at nearly all sizes.
//
// us a layer (seven products, 4-bit), before -> now, hidden / intermediate:
//   rows   1024/2816    1984/2560    2560/6912    4096/12288   8192/28672
//     17   28.3 -> 10.2 29.1 -> 10.6 68.3 -> 22.7 61.2 -> 54   211 -> 172
//     32   29.6 -> 10.2 30.5 -> 11.3 70.3 -> 23.1 62.9 -> 57   218 -> 185
//     64   32.8 -> 13.5 35.9 -> 15.2 82.1 -> 32.2 84.5 -> 72   340 -> 240
//    100   22.9 -> 13.8 22.4 -> 21.8 53.5 -> 44   104 -> 100   335 (GEMM)
//    128   21.0 -> 14.2 20.6 (GEMM)  52.2 -> 46   109 -> 105   352 (GEMM)
// 8-bit: 2560/6912 58 -> 26 (17 rows), 61 -> 39 (64), 69 -> 52 (128);
// 4096/12288 101 -> 63, 105 -> 79, 120 -> 117.
#include "qmm_common.h"

namespace qmm {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int KW = 4, kWaves = 8, kThreads = 64 * kWaves;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t st_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)bytes, 0x00020000);
}

// Byte B of u as a float.
template <int B>
__device__ __forceinline__ float byte_f32(uint32_t u) {
    float f;
    if (B == 0) asm("v_cvt_f32_ubyte0 %0, %1" : "=v"(f) : "v"(u));
    else if (B == 1) asm("v_cvt_f32_ubyte1 %0, %1" : "=v"(f) : "v"(u));
    else if (B == 2) asm("v_cvt_f32_ubyte2 %0, %1" : "=v"(f) : "v"(u));
    else asm("v_cvt_f32_ubyte3 %0, %1" : "=v"(f) : "v"(u));
    return f;
}
__device__ __forceinline__ uint32_t pack(float a, float b) {
    const bf16x2 p = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(uint32_t, p);
}

template <int MT, int NT>
struct StreamLds {
    static constexpr int R = 16 * MT, RP = R + 1;  // a row's staging stores fall on distinct banks
    static constexpr int kPieces = 8 * KW;         // 8-value pieces of a row's pass
    static constexpr int kCols = 16 * NT * (kWaves / KW);
    union {
        u32x4 xa[2][kPieces * RP];               // activations, [piece in MFMA order][row]
        float red[KW * R * kCols];  // the K waves' sums, [wave][row][column]
    };
};

template <int BITS, int MT, int NT, bool BF>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4))) void qgemm_stream(AffineBatch batch) {
    (void)batch;
    using L = StreamLds<MT, NT>;
    __shared__ L lds;
    constexpr int R = L::R, RP = L::RP, XI = R * L::kPieces / kThreads;  // pieces per thread
    constexpr bool PIPE = MT * NT < 8;  // what 128 registers hold
    constexpr uint32_t kPass = 64 * KW, kCols = L::kCols;
    static_assert(XI >= 1, "every thread stages a piece");
    const AffineBatch* kb = (const AffineBatch*)__builtin_amdgcn_kernarg_segment_ptr();
    uint32_t oi = 0;
    while (oi + 1 < kb->count && blockIdx.x >= kb->op[oi + 1].block_begin) ++oi;
    const AffineOp& op = kb->op[oi];
    const uint32_t M = op.m, N = op.n, K = op.k, G = K / 64;
    const uint32_t ct = (N + kCols - 1) / kCols, t0 = blockIdx.x - op.block_begin;
    const uint32_t n0 = t0 % ct * kCols, m0 = t0 / ct * R;
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t col = lane & 15, kq = lane >> 4, kw = wave % KW, nw = wave / KW;
    const uint32_t passes = (G + KW - 1) / KW;
    const uint32_t row_bytes = K / 8 * BITS;
    const bool biased = op.corr_kind == STARK_QMM_CORRECTION_BIASES;
    const uint32_t flip = op.flags & FLAG_SIGNED ? (BITS == 4 ? 0x88888888u : 0x80808080u) : 0u;

    uint32_t co[NT];  // byte offsets of a lane's codes of group 0
#pragma unroll
    for (int t = 0; t < NT; ++t)
        co[t] = min(n0 + 16 * (NT * nw + t) + col, N - 1) * row_bytes + 2 * BITS * kq;
    uint32_t po[NT];  // byte offsets of its columns' scales in group 0
#pragma unroll
    for (int t = 0; t < NT; ++t) po[t] = 2 * min(n0 + 16 * (NT * nw + t) + col, N - 1) * op.os;
    const uint8_t* scales = (const uint8_t*)op.scales;
    const uint8_t* corr = biased ? (const uint8_t*)op.corr : scales;
    const uint32_t x_bytes = 2 * M * K;

    // staging: piece tid % kPieces of rows tid / kPieces + (512 / kPieces) i; rows past M repeat the last
    const uint32_t piece = tid % L::kPieces, srow = tid / L::kPieces;
    constexpr uint32_t rstep = kThreads / L::kPieces;
    // the lane of k quarter kq takes piece 2 kq + j for the group's j-th MFMA
    const uint32_t pos = (piece & ~7u) + 4 * (piece & 1) + ((piece & 7) >> 1);
    const uint8_t* xp = (const uint8_t*)op.x;
    uint32_t xo[XI];  // byte offsets in pass 0
#pragma unroll
    for (int i = 0; i < XI; ++i) xo[i] = 2 * (min(m0 + srow + rstep * i, M - 1) * K + 8 * piece);

    u32x4 xv[XI];
    struct Codes {
        u32x4 c[NT];  // 4-bit: the first two words
        uint32_t s[NT], b[NT];
    } wv[2];
    // What lies past K in the last pass is another row's, or zero past the end
    // of the operand: its groups are not computed.
    const auto load_x = [&](uint32_t p) {
        const uint32_t ox = 2 * kPass * p;
        const __amdgpu_buffer_rsrc_t rx = st_rsrc(xp + ox, x_bytes - ox);
#pragma unroll
        for (int i = 0; i < XI; ++i) xv[i] = __builtin_amdgcn_raw_buffer_load_b128(rx, xo[i], 0, 0);
    };
    const auto load_w = [&](uint32_t p, Codes& w) {
        const uint32_t g = min(p * KW + kw, G - 1);  // past K: not computed
        const uint8_t* base = op.codes + g * (8 * BITS);
        const uint32_t og = 2 * g * op.gs;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            w.s[t] = *(const uint16_t*)(scales + og + po[t]);
            w.b[t] = *(const uint16_t*)(corr + og + po[t]);
            if (BITS == 4) {
                const u32x2 v = *(const u32x2*)(base + co[t]);
                w.c[t] = u32x4{v[0], v[1], 0, 0};
            } else {
                w.c[t] = *(const u32x4*)(base + co[t]);
            }
        }
    };
    const auto stage = [&](int buf) {
#pragma unroll
        for (int i = 0; i < XI; ++i) lds.xa[buf][pos * RP + srow + rstep * i] = xv[i];
    };

    struct Operands {
        bf16x8 v[NT][2];
    } bo[PIPE ? 2 : 1];
    const auto dequant = [&](const Codes& w, Operands& o) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const float s = BF ? __uint_as_float(w.s[t] << 16) : f16_bits_to_f32(w.s[t]);
            const float bi = BF ? __uint_as_float(w.b[t] << 16) : f16_bits_to_f32(w.b[t]);
            const float bt = biased ? bi : -s * (float)(1 << (BITS - 1));
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                u32x4 r;
                if (BITS == 4) {
                    const uint32_t u = w.c[t][j] ^ flip, lo = u & 0x0F0F0F0Fu, hi = (u >> 4) & 0x0F0F0F0Fu;
                    r[0] = pack(fmaf(byte_f32<0>(lo), s, bt), fmaf(byte_f32<0>(hi), s, bt));
                    r[1] = pack(fmaf(byte_f32<1>(lo), s, bt), fmaf(byte_f32<1>(hi), s, bt));
                    r[2] = pack(fmaf(byte_f32<2>(lo), s, bt), fmaf(byte_f32<2>(hi), s, bt));
                    r[3] = pack(fmaf(byte_f32<3>(lo), s, bt), fmaf(byte_f32<3>(hi), s, bt));
                } else {
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const uint32_t u = w.c[t][2 * j + h] ^ flip;
                        r[2 * h] = pack(fmaf(byte_f32<0>(u), s, bt), fmaf(byte_f32<1>(u), s, bt));
                        r[2 * h + 1] = pack(fmaf(byte_f32<2>(u), s, bt), fmaf(byte_f32<3>(u), s, bt));
                    }
                }
                o.v[t][j] = __builtin_bit_cast(bf16x8, r);
            }
        }
    };
    f32x4 acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[m][t] = f32x4{0, 0, 0, 0};
    const auto compute = [&](int buf, const Operands& b) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const u32x4* a = &lds.xa[buf][(8 * kw + kq) * RP + 16 * m + col];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const bf16x8 av = __builtin_bit_cast(bf16x8, a[4 * j * RP]);
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, b.v[t][j], acc[m][t], 0, 0, 0);
            }
        }
    };

    // Pass q multiplies LDS buffer q % 2; prefetches past the last pass are
    // clamped to it (what they bring is not computed). PIPE: the operands of pass
    // q + 1 are dequantised beside the products of pass q.
    const uint32_t last = passes - 1;
    load_x(0);
    load_w(0, wv[0]);
    load_w(min(1u, last), wv[1]);
    stage(0);
    load_x(min(1u, last));
    if (PIPE) {
        dequant(wv[0], bo[0]);
        load_w(min(2u, last), wv[0]);
    }
    lds_barrier();
    uint32_t p = 0;
    for (; p + 2 <= last; p += 2) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            constexpr int ahead = PIPE ? 1 : 0;
            stage(i ^ 1);
            load_x(min(p + i + 2, last));
            dequant(wv[i ^ ahead], bo[(i ^ 1) & ahead]);
            compute(i, bo[i & ahead]);
            load_w(min(p + i + 2 + ahead, last), wv[i ^ ahead]);
            lds_barrier();
        }
    }
    // one or two passes are left; the last may hold fewer groups than waves
    if (!PIPE) dequant(wv[0], bo[0]);
    if (p < last) {
        stage(1);
        if (PIPE) dequant(wv[1], bo[1]);
        compute(0, bo[0]);
        lds_barrier();
        if (!PIPE) dequant(wv[1], bo[0]);
        if (last * KW + kw < G) compute(1, bo[PIPE]);
    } else if (last * KW + kw < G) {
        compute(0, bo[0]);
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
    lds_barrier();  // the activations are read: their LDS takes the sums
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                lds.red[(kw * R + 16 * m + 4 * kq + e) * kCols + 16 * (NT * nw + t) + col] = acc[m][t][e];
    lds_barrier();
    const uint32_t rows = min((uint32_t)R, M - m0);
    for (uint32_t q = tid; q < rows * kCols; q += kThreads) {
        const float v = (lds.red[q] + lds.red[R * kCols + q]) + (lds.red[2 * R * kCols + q] + lds.red[3 * R * kCols + q]);
        store(q / kCols, n0 + q % kCols, v);
    }
}

template <int MT, int NT>
stark_qmm_status launch_shape(AffineBatch& b, int bits, hipStream_t stream) {
    constexpr uint32_t cols = StreamLds<MT, NT>::kCols;
    uint64_t total = 0;
    for (uint32_t i = 0; i < b.count; ++i) {
        b.op[i].block_begin = (uint32_t)total;
        total += (uint64_t)((b.op[i].n + cols - 1) / cols) * ((b.op[i].m + 16 * MT - 1) / (16 * MT));
        if (total > 0x7fffffffu) return STARK_QMM_UNSUPPORTED;
    }
    const bool bf = b.op[0].w_dt == STARK_QMM_BF16;
    const dim3 grid((uint32_t)total);
    if (bits == 4 && bf) hipLaunchKernelGGL((qgemm_stream<4, MT, NT, true>), grid, dim3(kThreads), 0, stream, b);
    else if (bits == 4) hipLaunchKernelGGL((qgemm_stream<4, MT, NT, false>), grid, dim3(kThreads), 0, stream, b);
    else if (bf) hipLaunchKernelGGL((qgemm_stream<8, MT, NT, true>), grid, dim3(kThreads), 0, stream, b);
    else hipLaunchKernelGGL((qgemm_stream<8, MT, NT, false>), grid, dim3(kThreads), 0, stream, b);
    QMM_HIP_CHECK(hipGetLastError());
    return STARK_QMM_OK;
}

}  // namespace

bool gemm_stream_eligible(const AffineOp& o, int bits) {
    if (o.m <= 16 || o.m > 128 || o.group_size != 64 || o.k == 0 || o.k % 64 || o.n == 0 || o.gather) return false;
    if ((bits != 4 && bits != 8) || o.x_dt != STARK_QMM_BF16) return false;
    if (!(o.w_dt == STARK_QMM_BF16 || o.w_dt == STARK_QMM_F16)) return false;
    if (!(o.corr_kind == STARK_QMM_CORRECTION_BIASES || o.corr_kind == STARK_QMM_CORRECTION_SYMMETRIC)) return false;
    if (((uintptr_t)o.codes | (uintptr_t)o.x) & 15) return false;
    // 32-bit byte offsets of the planes
    if (2 * ((uint64_t)o.n * o.os + (uint64_t)(o.k / 64) * o.gs) >= (1ull << 31)) return false;
    // Weights are rounded to bf16 here, so nothing may come from the kernels
    // that keep them in f32: besides the GEMM's own products (whose bound on the
    // codes has 128 rows to spare) only 4-bit ones of up to 64 rows and whole
    // 512-value steps, which have had bf16 weights up to 2 GiB of codes.
    return gemm_eligible(o, bits) ||
           (bits == 4 && o.m <= 64 && o.n >= 16 && o.k % 512 == 0 && (uint64_t)o.n * o.k / 2 < (1ull << 31) &&
            (uint64_t)64 * o.k * 2 < (1ull << 31));
}

bool gemm_stream_pays(const AffineOp* ops, uint32_t count, int bits) {
    std::vector<AffineOp> tall;
    for (uint32_t i = 0; i < count; ++i)
        if (ops[i].m > 64) tall.push_back(ops[i]);
    int dev = 0, cus = 0;
    if (tall.empty() || hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return tall.empty();
    return stream_takes(tall.data(), (uint32_t)tall.size(), bits, (uint32_t)cus);
}

// ops: all gemm_stream_eligible for `bits`, of one plane type; longest K first.
// Row blocks of equal size, at most 64 rows each; 32 or 64 columns a workgroup (stream_wide).
stark_qmm_status launch_gemm_stream(const AffineOp* ops, uint32_t count, int bits, hipStream_t stream) {
    if (count == 0) return STARK_QMM_OK;
    if (count > (uint32_t)kMaxBatchOps) return STARK_QMM_UNSUPPORTED;
    AffineBatch b{};
    std::copy(ops, ops + count, b.op);
    std::stable_sort(b.op, b.op + count, [](const AffineOp& x, const AffineOp& y) { return x.k > y.k; });
    b.count = count;
    const uint32_t mt = stream_blocks(ops, count);
    int dev = 0, cus = 0;
    QMM_HIP_CHECK(hipGetDevice(&dev));
    QMM_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const bool wide = stream_wide(ops, count, (uint32_t)cus);
    if (mt == 2) return wide ? launch_shape<2, 2>(b, bits, stream) : launch_shape<2, 1>(b, bits, stream);
    if (mt == 3) return wide ? launch_shape<3, 2>(b, bits, stream) : launch_shape<3, 1>(b, bits, stream);
    return wide ? launch_shape<4, 2>(b, bits, stream) : launch_shape<4, 1>(b, bits, stream);
}

}  // namespace qmm
