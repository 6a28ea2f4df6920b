// Products of 1 to 16 activation rows on the matrix cores, group 64, 4- or
// 8-bit, any K that is a multiple of 64 and any N and plane layout.
//
// The arithmetic is that of mfma_tile.h (codes as raw bf16 bit patterns,
// activations as x * 2^E with a per-group exponent, group sums scaled in f32),
// the dense form: all 16 A rows of an MFMA are activation rows, one group per
// accumulator. The codes go from global memory straight into the B operand (a
// lane loads 16 bytes of its row; for 4-bit codes v_permlane32_swap sorts the
// words so that every MFMA holds codes of one group), so there is no LDS pass
// for them and no row, plane or K alignment past 16-byte code rows.
//
// A workgroup of eight waves owns 32 weight rows; its waves take the 128-value
// chunks of K in turn (together they read whole lines of the rows) and their
// sums meet in LDS. A pass is eight chunks: its activations are converted once
// into LDS in MFMA order, double-buffered; a pass's activation and plane loads
// are issued before its codes, so staging the next pass leaves the code loads
// in flight.
//
// Activation row r sits in MFMA row 4 (r % 4) + r / 4, so that up to 4 (8) rows
// occupy one (two) of a lane's four accumulator entries and only those are
// scaled (EM = 1, 2, 4 entries).
#include "qmm_common.h"
#include "code_layout.h"

namespace qmm {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 8, kThreads = 64 * kWaves;
constexpr uint32_t kChunk = 128, kPass = kWaves * kChunk, kCols = 32;

struct GroupX {
    int e;      // 133 - E
    float sum;  // sum of x
};

template <int EM>
struct DenseLds {
    static constexpr int R = 4 * EM;  // activation rows staged
    static constexpr int RP = R + 1;  // a row's staging stores fall on distinct banks
    union {
        u32x4 xa[2][kPass / 8 * RP];  // activations x * 2^E, [8-value piece in MFMA order][row]
        float red[kWaves * R * kCols];  // the waves' sums, [wave][row][column]
    };
    GroupX xg[2][kPass / 64][R];
    uint32_t pl[2][kThreads];  // raw scale | bias << 16, [group][column]
};

template <int BITS, int EM, bool BIASED, bool BF>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(EM == 1 ? 5 : 4))) void qmv_dense(
    AffineBatch batch) {
    (void)batch;
    __shared__ DenseLds<EM> lds;
    constexpr int R = DenseLds<EM>::R, RP = DenseLds<EM>::RP, WL = BITS / 4;
    const AffineBatch* kb = (const AffineBatch*)__builtin_amdgcn_kernarg_segment_ptr();
    uint32_t oi = 0;
    while (oi + 1 < kb->count && blockIdx.x >= kb->op[oi + 1].block_begin) ++oi;
    const AffineOp& op = kb->op[oi];
    // blocks b and b + 8, on one XCD, take neighbouring tiles (which share the lines of group-output planes)
    const uint32_t b = blockIdx.x - op.block_begin;
    const uint32_t n0 = ((b & ~15u) + 2 * (b & 7) + ((b >> 3) & 1)) * kCols;
    const uint32_t M = op.m, N = op.n, K = op.k, G = K / 64;
    if (n0 >= N) return;
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t col = lane & 15, kq = lane >> 4;
    const uint32_t passes = (K + kPass - 1) / kPass;
    const size_t row_bytes = (size_t)K * BITS / 8;
    const uint32_t flip = op.flags & FLAG_SIGNED ? (BITS == 4 ? 0x88888888u : 0x80808080u) : 0u;

    // this lane's two weight rows (rows past N read the last one and are not stored)
    const uint8_t* cp[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) cp[t] = op.codes + (size_t)min(n0 + 16 * t + col, N - 1) * row_bytes;
    // plane entry of this thread: consecutive lanes take consecutive rows of
    // group-output planes, else consecutive groups of a row
    const uint32_t pg = op.os == 1 ? tid / kCols : tid % (kPass / 64);
    const uint32_t pc = op.os == 1 ? tid % kCols : tid / (kPass / 64);
    const size_t po = (size_t)min(n0 + pc, N - 1) * op.os;
    const uint16_t* scales = (const uint16_t*)op.scales;
    const uint16_t* corr = BIASED ? (const uint16_t*)op.corr : scales;

    // staging: 8-value piece tid % 128 of rows tid / 128 + 4 i
    const uint32_t piece = tid % (kPass / 8), srow = tid / (kPass / 8);
    constexpr uint32_t rstep = kThreads / (kPass / 8);

    u32x4 wv[2][2][WL];  // [set][tile][16-byte load]
    u32x4 xv[EM];
    uint32_t ps, pb;
    const auto load_xp = [&](uint32_t p) {
        const uint32_t k = p * kPass + piece * 8;
#pragma unroll
        for (int i = 0; i < EM; ++i) {
            const uint32_t r = srow + rstep * i;
            const bool ok = r < M && k < K;
            xv[i] = *(const u32x4*)((const uint16_t*)op.x + (ok ? (size_t)r * K + k : 0));
        }
        const size_t o = po + (size_t)min(p * (kPass / 64) + pg, G - 1) * op.gs;
        ps = scales[o];
        pb = corr[o];
    };
    const auto load_w = [&](uint32_t p, u32x4 (&w)[2][WL]) {
        const uint32_t k = p * kPass + wave * kChunk;
#pragma unroll
        for (int h = 0; h < WL; ++h) {
            const uint32_t o = code_offset<BITS>(k, h, kq, K);
            // cached: two waves read the halves of a line (with the
            // nontemporal hint 4-bit rows ran 5% and rows of no whole
            // number of lines up to 20% slower)
            w[0][h] = *(const u32x4*)(cp[0] + o);
            w[1][h] = *(const u32x4*)(cp[1] + o);
        }
    };
    const auto stage = [&](uint32_t p, int buf) {
        const uint32_t k = p * kPass + piece * 8;
#pragma unroll
        for (int i = 0; i < EM; ++i) {
            const uint32_t r = srow + rstep * i;
            if (r >= M) continue;  // whole groups of lanes leave together
            u32x4 t = xv[i];
            if (k >= K) t = u32x4{0, 0, 0, 0};
            const int E = group_shift(group_max<8>(bf16x8_exp_max(t)));
            const float se = pow2i(E), so = BITS == 4 ? pow2i(E - 4) : se;
            float f[8];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                f[2 * e] = __uint_as_float(t[e] << 16) * se;
                f[2 * e + 1] = __uint_as_float(t[e] & 0xffff0000u) * so;
            }
            // 4-bit pairs (x0,x4)(x1,x5)(x2,x6)(x3,x7); 8-bit pairs (x0,x2)(x1,x3)(x4,x6)(x5,x7)
            constexpr int p1 = BITS == 4 ? 4 : 2, p3 = BITS == 4 ? 5 : 3, p4 = BITS == 4 ? 2 : 4, p6 = BITS == 4 ? 3 : 5;
            u32x4 q;
            q[0] = permb(__float_as_uint(f[p1]), __float_as_uint(f[0]), 0x07060302u);
            q[1] = permb(__float_as_uint(f[p3]), __float_as_uint(f[1]), 0x07060302u);
            q[2] = permb(__float_as_uint(f[6]), __float_as_uint(f[p4]), 0x07060302u);
            q[3] = permb(__float_as_uint(f[7]), __float_as_uint(f[p6]), 0x07060302u);
            lds.xa[buf][piece_pos<BITS>(piece) * RP + r] = q;
            float sm = 0.0f;
#pragma unroll
            for (int e = 0; e < 4; ++e) sm = dot2_bf16(t[e], 0x3F803F80u, sm);
            sm = group_sum<8>(sm);
            if ((piece & 7) == 0) lds.xg[buf][piece >> 3][r] = GroupX{133 - E, sm};
        }
        lds.pl[buf][pg * kCols + pc] = ps | (pb << 16);
    };

    // The f32 error comes from the running sums' roundings, two a group (K 12288,
    // 4-bit, 12 rows: 1.62e-7 of the result, 8-bit 1.61e-7): two sums (1.38e-7,
    // within 0.5% of the time), or, for 8-bit rows 9 to 16, whose second sums
    // spill (+7%), one that takes a group's two terms joined (1.35e-7, +1%; joined
    // everywhere: +1% everywhere).
    constexpr int SUMS = BITS == 8 && EM == 4 ? 1 : 2;
    float acc[SUMS][2][EM];  // [group of a chunk][tile][entry]
#pragma unroll
    for (int g = 0; g < SUMS; ++g)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int e = 0; e < EM; ++e) acc[g][t][e] = 0.0f;
    // this lane's A row: MFMA row col = 4 (r % 4) + r / 4; entries past EM repeat a row and are not read
    const uint32_t arow = (col >> 2) + ((col & 3) < (uint32_t)EM ? 4 * (col & 3) : 0);
    const auto compute = [&](int buf, u32x4 (&w)[2][WL], uint32_t ng) {
        // code words of group g's MFMA j, tile t
        uint32_t u[2][2][2][WL];  // [tile][group][MFMA]
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                if (BITS == 4) {
                    const auto s = __builtin_amdgcn_permlane32_swap(w[t][0][2 * j], w[t][0][2 * j + 1], false, false);
                    u[t][0][j][0] = s[0];
                    u[t][1][j][0] = s[1];
                } else {
#pragma unroll
                    for (int h = 0; h < 2; ++h)
#pragma unroll
                        for (int q = 0; q < WL; ++q)
                            u[t][h][j][q] = w[t][h % WL][2 * j + q];
                }
            }
        if (flip) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
#pragma unroll
                        for (int q = 0; q < WL; ++q) u[t][h][j][q] ^= flip;
        }
        const uint32_t* pl = &lds.pl[buf][2 * wave * kCols + col];
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            if ((uint32_t)g >= ng) break;
            const u32x4* a = &lds.xa[buf][(16 * wave + 8 * g + kq) * RP + arow];
            const bf16x8 a0 = __builtin_bit_cast(bf16x8, a[0]), a1 = __builtin_bit_cast(bf16x8, a[4 * RP]);
            GroupX xg[EM];
#pragma unroll
            for (int e = 0; e < EM; ++e) xg[e] = lds.xg[buf][2 * wave + g][kq + 4 * e];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                bf16x8 b[2];
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    u32x4 q;
                    if (BITS == 4) {
                        const uint32_t x = u[t][g][j][0], y = x >> 8;
                        q = u32x4{x & 0x000F000Fu, x & 0x00F000F0u, y & 0x000F000Fu, y & 0x00F000F0u};
                    } else {
                        const uint32_t x = u[t][g][j][0], y = u[t][g][j][WL - 1];
                        q = u32x4{x & 0x00FF00FFu, (x >> 8) & 0x00FF00FFu, y & 0x00FF00FFu, (y >> 8) & 0x00FF00FFu};
                    }
                    b[j] = __builtin_bit_cast(bf16x8, q);
                }
                f32x4 c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b[0], f32x4{0, 0, 0, 0}, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b[1], c, 0, 0, 0);
                const uint32_t p = pl[g * kCols + 16 * t];
                const float sc = BF ? __uint_as_float(p << 16) : f16_bits_to_f32(p & 0xffffu);
                const float bi = !BIASED ? -(float)(1 << (BITS - 1)) * sc
                                 : BF    ? __uint_as_float(p & 0xffff0000u)
                                         : f16_bits_to_f32(p >> 16);
#pragma unroll
                for (int e = 0; e < EM; ++e) {
                    float& s = acc[g % SUMS][t][e];
                    const float d = ldexp_f32(c[e], xg[e].e);
                    s = SUMS == 2 ? fmaf(sc, d, fmaf(bi, xg[e].sum, s)) : s + fmaf(sc, d, bi * xg[e].sum);
                }
            }
            // keeps the scaling here: moved past the staging and the barrier, it would hold every group's sums live
#pragma unroll
            for (int e = 0; e < EM; ++e) asm volatile("" : "+v"(acc[g % SUMS][0][e]), "+v"(acc[g % SUMS][1][e]));
        }
    };
    // groups of this wave's chunk in a pass
    const auto groups = [&](uint32_t p) -> uint32_t {
        const uint32_t g = p * (kPass / 64) + 2 * wave;
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
    lds_barrier();  // the activations are read: their LDS takes the sums
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < EM; ++e) {
            const uint32_t r = kq + 4 * e;
            lds.red[(wave * R + r) * kCols + 16 * t + col] = SUMS == 2 ? acc[0][t][e] + acc[1][t][e] : acc[0][t][e];
        }
    lds_barrier();
    for (uint32_t q = tid; q < M * kCols; q += kThreads) {
        const uint32_t r = q / kCols, c = q % kCols, n = n0 + c;
        if (n >= N) continue;
        const float* s = &lds.red[r * kCols + c];
        constexpr uint32_t st = R * kCols;
        float v = ((s[0] + s[st]) + (s[2 * st] + s[3 * st])) + ((s[4 * st] + s[5 * st]) + (s[6 * st] + s[7 * st]));
        v *= op.ab_scale;
        const size_t o = (size_t)r * N + n;
        if (op.flags & FLAG_ACCUMULATE) v += load_as_f32(op.d, op.d_dt, o);
        if (op.bias) v += load_as_f32(op.bias, op.w_dt, n);
        if (op.flags & FLAG_SOFT_CAP) v = op.soft_cap * tanhf(v / op.soft_cap);
        store_from_f32(op.d, op.d_dt, o, v);
    }
}

template <int BITS, bool BIASED, bool BF>
void launch_em(const AffineBatch& b, int em, hipStream_t stream) {
    const dim3 grid(b.total);
    if (em == 1) hipLaunchKernelGGL((qmv_dense<BITS, 1, BIASED, BF>), grid, dim3(kThreads), 0, stream, b);
    else if (em == 2) hipLaunchKernelGGL((qmv_dense<BITS, 2, BIASED, BF>), grid, dim3(kThreads), 0, stream, b);
    else hipLaunchKernelGGL((qmv_dense<BITS, 4, BIASED, BF>), grid, dim3(kThreads), 0, stream, b);
}

}  // namespace

bool dense_eligible(const AffineOp& o, int bits) {
    return (bits == 4 || bits == 8) && o.x_dt == STARK_QMM_BF16 && !o.gather && o.m >= 1 && o.m <= 16 &&
           (o.corr_kind == STARK_QMM_CORRECTION_BIASES || o.corr_kind == STARK_QMM_CORRECTION_SYMMETRIC) &&
           (o.w_dt == STARK_QMM_BF16 || o.w_dt == STARK_QMM_F16) && o.group_size == 64 && o.k != 0 && o.k % 64 == 0 &&
           o.n != 0 && (((uintptr_t)o.codes | (uintptr_t)o.x) & 15) == 0 &&
           (((uintptr_t)o.scales | (uintptr_t)o.corr) & 1) == 0;
}

// Measured against the other matrix-core kernels over four layers of
// projections (hidden / intermediate sizes 1024 to 4096 / 2560 to 12288, us):
//  - planes those cannot read (rows of no whole 8 groups): one row, hidden 1024:
//    59 -> 28; 8-bit, hidden 2560 / 6912: 185 -> 93;
//  - 4-bit, 3 to 8 rows: always faster (hidden 4096 / 12288: 123 -> 101, 126 ->
//    120, 135 -> 128 at 3, 5, 8 rows; 2048 / 6144: 70 -> 49 at 5); 9 to 16 rows:
//    faster unless qmv_small_m gets long runs (small_m_long);
//  - 8-bit: faster from 9 rows, and from 5 unless the tiles come out badly
//    (w8_rows5_mfma; hidden 4096 / 11008: 199 -> 178 at 6 rows, 295 -> 214 at 16;
//    155 -> 168 at 3);
//  - one or two rows: few_rows_rule (4-bit passes with an idle share: hidden 2560
//    / 6912, 32%: 60 -> 56; 3584 / 9728, 11%: 77 -> 79, 88 -> 85; 2048 / 6144,
//    none: 39 -> 44, 40 -> 45; 8-bit, 1024-value passes, hidden 4096 / 11008:
//    147 -> 161; qmv_stream, K % 4096 == 0: 85 -> 95).
DenseRule::DenseRule(const AffineOp* ops, uint32_t count, int b)
    : bits(b), few_rows{false, false}, many_rows(true), mid_rows(true) {
    const auto readable = [&](const AffineOp& o) { return mfma_eligible(o, bits); };
    const auto cus = [] {
        int dev = 0, n = 0;
        return hipGetDevice(&dev) == hipSuccess &&
                       hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess
                   ? (uint32_t)n
                   : 256u;
    };
    if (count == 1 && ops[0].m <= 2) {  // the call that is all launch: no copies, nothing asked of the device
        if (dense_eligible(ops[0], bits)) few_rows = few_rows_rule(ops, 1, bits, 0u, readable);
        return;
    }
    // the products of each rule: the call's own array where they all fall under one
    const auto rule_of = [&](const AffineOp& o) {
        if (!dense_eligible(o, bits)) return 0;
        if (o.m <= 2) return 1;
        if (o.m > 8) return bits == 4 ? 2 : 0;
        return o.m > 4 && bits == 8 ? 3 : 0;
    };
    uint32_t n[4] = {};
    for (uint32_t i = 0; i < count; ++i) ++n[rule_of(ops[i])];
    std::vector<AffineOp> part;
    const auto products = [&](int rule) {
        if (n[rule] == count) return ops;
        part.clear();
        part.reserve(n[rule]);
        for (uint32_t i = 0; i < count; ++i)
            if (rule_of(ops[i]) == rule) part.push_back(ops[i]);
        return (const AffineOp*)part.data();
    };
    if (n[1]) few_rows = few_rows_rule(products(1), n[1], bits, cus(), readable);
    if (n[2]) {
        const AffineOp* many = products(2);
        if (small_m_eligible(many, n[2])) many_rows = !small_m_long(many, n[2], cus());
    }
    if (n[3]) {
        const AffineOp* mid = products(3);
        if (std::all_of(mid, mid + n[3], readable)) mid_rows = !w8_rows5_mfma(mid, n[3], cus());
    }
}

bool DenseRule::takes(const AffineOp& o) const {
    if (!dense_eligible(o, bits)) return false;
    if (!mfma_eligible(o, bits)) return true;
    if (o.m <= 2) return few_rows.idle || few_rows.drag;
    if (bits == 8) return o.m > 8 || (o.m > 4 && mid_rows);
    return o.m <= 8 || many_rows || !small_m_eligible(&o, 1);
}

// ops: all dense_eligible for `bits`, of one entry count (rows), correction and plane type.
static stark_qmm_status launch_dense_class(const AffineOp* ops, uint32_t count, int bits, hipStream_t stream) {
    AffineBatch b{};
    std::vector<AffineOp> v(ops, ops + count);
    std::stable_sort(v.begin(), v.end(), [](const AffineOp& x, const AffineOp& y) { return x.k > y.k; });
    uint64_t total = 0;
    uint32_t m = 0;
    for (uint32_t i = 0; i < count; ++i) {
        b.op[i] = v[i];
        b.op[i].block_begin = (uint32_t)total;
        total += ((uint64_t)v[i].n + 16 * kCols - 1) / (16 * kCols) * 16;  // whole groups of 16 tiles
        m = std::max(m, v[i].m);
    }
    if (total > 0x7fffffffu) return STARK_QMM_UNSUPPORTED;
    b.count = count;
    b.total = (uint32_t)total;
    const int em = m <= 4 ? 1 : m <= 8 ? 2 : 4;
    const bool bi = v[0].corr_kind == STARK_QMM_CORRECTION_BIASES, bf = v[0].w_dt == STARK_QMM_BF16;
    if (bits == 4) {
        if (bi) bf ? launch_em<4, true, true>(b, em, stream) : launch_em<4, true, false>(b, em, stream);
        else bf ? launch_em<4, false, true>(b, em, stream) : launch_em<4, false, false>(b, em, stream);
    } else {
        if (bi) bf ? launch_em<8, true, true>(b, em, stream) : launch_em<8, true, false>(b, em, stream);
        else bf ? launch_em<8, false, true>(b, em, stream) : launch_em<8, false, false>(b, em, stream);
    }
    QMM_HIP_CHECK(hipGetLastError());
    return STARK_QMM_OK;
}

stark_qmm_status launch_affine_dense(const AffineOp* ops, uint32_t count, int bits, hipStream_t stream) {
    std::vector<AffineOp> cls[3][2][2];
    for (uint32_t i = 0; i < count; ++i)
        cls[ops[i].m <= 4 ? 0 : ops[i].m <= 8 ? 1 : 2][ops[i].corr_kind == STARK_QMM_CORRECTION_BIASES]
           [ops[i].w_dt == STARK_QMM_BF16].push_back(ops[i]);
    for (auto& a : cls)
        for (auto& c : a)
            for (auto& v : c)
                for (size_t s = 0; s < v.size(); s += kMaxBatchOps) {
                    const uint32_t n = (uint32_t)std::min<size_t>(kMaxBatchOps, v.size() - s);
                    const stark_qmm_status st = launch_dense_class(v.data() + s, n, bits, stream);
                    if (st != STARK_QMM_OK) return st;
                }
    return STARK_QMM_OK;
}

}  // namespace qmm
