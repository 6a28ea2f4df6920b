// Grouped expert products for prompts (more than 16 tokens), 4-bit group-64
// banks: one slot is up to 64 routes of one expert, and a workgroup computes a
// column tile of the expert's rows for all of a slot's routes, so an expert's
// weights are read once per 64 routes.
//
// The arithmetic is the routed kernels' exact form (mfma_tile.h): codes enter
// v_mfma_f32_16x16x32_bf16 as raw bf16 bit patterns, activations as x * 2^E
// with a per-group exponent, a group's sum is brought back with ldexp, scaled
// in f32 and added to the accumulator; the bias terms bias * sum(x) of four
// groups are one v_mfma_f32_16x16x4_f32 (f32 products and sums).
//
// What bounds it: at 512 tokens (32 routes an expert on average) the 340 MB of
// expert weights are 60 us of HBM and take 132: the vector work of a group (the
// exponents, the scaling of every sum) beside the loads, most of all in the up
// product, whose activations every column tile converts again. Hence:
//  - B operands come straight from global memory: a lane loads 16 bytes (32
//    codes) of its row, so an instruction reads 64 bytes of each of 16 rows,
//    and v_permlane32_swap sorts the words so that all four lane groups of an
//    MFMA hold codes of one 64-value group (no LDS pass for the codes, and all
//    16 activation rows of every MFMA are in use, where the slot form of
//    mfma_tile.h uses 8);
//  - the routes' activations are converted once per workgroup into LDS, in
//    MFMA order ([16-byte piece][row]: operand reads are contiguous), and
//    serve its eight waves' 32 rows each;
//  - chunks of 128 values, activations and planes double-buffered in LDS, the
//    codes in two register sets; a chunk's activation and plane loads are
//    issued before its codes, so staging the next chunk leaves the code loads
//    in flight.
// Measured (model 2048, hidden 768, 128 experts, top 8, router included): 512
// tokens 1978 -> 178 us, 160 with the router's later product (the products
// 1103 + 851 -> 86 + 46 us, 2.6 and 2.5 TB/s of weights). The slot form of
// mfma_tile.h (16 routes a slot, half of every MFMA empty, codes through LDS, the
// weights once per 16 routes) stays for group sizes 32 and 128 and where
// moe_grouped (dispatch_rules.h) says so.
#include "qmm_common.h"
#include "code_layout.h"

namespace qmm {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kWaves = 8, kThreads = 64 * kWaves;
constexpr int kSlot = 64;         // routes per slot
constexpr int kChunk = 128;       // k values per chunk (two groups)
constexpr int kPieces = kChunk / 8;
constexpr int kRowPad = kSlot + 1;  // a row's 16 staging stores fall on distinct banks
constexpr int kCols = 32 * kWaves;  // bank rows per workgroup

struct GroupLds {
    u32x4 xa[2][kPieces * kRowPad];  // activations x * 2^E, [piece in MFMA order][route]
    alignas(16) int xe[2][2][kSlot];    // 133 - E per group and route
    // rings of four chunks: the bias terms of two chunks are added at once
    float xs[4][2][kSlot];    // sum of x per group and route
    uint32_t pl[4][2][kCols];  // scale | bias << 16 (raw bf16) per group and bank row
    uint32_t route[kSlot];
};

// B operand (8 codes of one row) of a code word: pairs (q0, q4) (16 q1, 16 q5)
// (q2, q6) (16 q3, 16 q7), as the activations are staged.
__device__ __forceinline__ bf16x8 codes8(uint32_t u) {
    const uint32_t v = u >> 8;
    return __builtin_bit_cast(bf16x8, u32x4{u & 0x000F000Fu, u & 0x00F000F0u, v & 0x000F000Fu, v & 0x00F000F0u});
}

// One column tile of one slot with MT 16-row blocks of routes. UP: the waves'
// 16 value rows and the matching 16 gate rows, gated SiLU in the epilogue.
// Otherwise 32 output rows per wave.
template <bool UP, bool SIGNED, int MT>
__device__ __forceinline__ void group_tile(const MoeGroup& L, GroupLds& lds, uint32_t expert, uint32_t cnt, uint32_t tile) {
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t col = lane & 15, kq = lane >> 4;
    const uint32_t K = UP ? L.model : L.hidden, N = UP ? L.hidden : L.model;
    const uint32_t G = K / 64, chunks = (K + kChunk - 1) / kChunk;
    const size_t row_bytes = K / 2;
    // bank rows of the wave's two 16-row tiles; a wave past the last rows works on the first ones and stores nothing
    const uint32_t wcols = UP ? 16 : 32;
    const uint32_t n0 = tile * (wcols * kWaves) + wave * wcols;
    const bool live = n0 < N;
    const size_t bank0 = (size_t)expert * (UP ? 2 * L.hidden : L.model);
    const size_t rowA = bank0 + (live ? n0 : 0), rowB = rowA + (UP ? L.hidden : 16);
    const uint8_t* cpA = L.codes + (rowA + col) * row_bytes + code_lane_offset(kq, K);
    const uint8_t* cpB = L.codes + (rowB + col) * row_bytes + code_lane_offset(kq, K);

    // staging: 16-byte piece tid % 16 of rows tid / 16 + 32 i
    constexpr int XI = (MT + 1) / 2;
    const uint32_t piece = tid & 15, srow = tid >> 4;
    const uint16_t* xp[XI];
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        const uint32_t r = lds.route[min(srow + 32 * i, cnt - 1)];
        xp[i] = L.x + (size_t)(UP ? r / L.active : r) * K;
    }
    // planes: one (row, group) entry per thread; consecutive lanes take
    // consecutive rows of group-output planes, consecutive groups otherwise
    const uint32_t pg = L.os == 1 ? tid / kCols : tid % 2, pr = L.os == 1 ? tid % kCols : tid / 2;
    size_t po;
    {
        // column pr of the workgroup's tile: wave pr / 32, its tile A or B
        const uint32_t w = pr / 32, c = pr % 32, n = tile * (wcols * kWaves) + w * wcols;
        po = (bank0 + (n < N ? n : 0) + (c & 15) + ((c & 16) ? (UP ? L.hidden : 16) : 0)) * L.os;
    }
    const uint16_t* corr = L.corr ? L.corr : L.scales;  // a symmetric bank's bias half is not read

    u32x4 wv[2][2];  // [set][tile]
    u32x4 xv[XI];
    uint32_t ps, pb;
    // activations and planes of a chunk; pieces past K are read from the row's start and staged as zeros
    const auto load_xp = [&](uint32_t c) {
        const uint32_t k = c * kChunk + piece * 8;
#pragma unroll
        for (int i = 0; i < XI; ++i) xv[i] = *(const u32x4*)(xp[i] + (k < K ? k : 0));
        const size_t o = po + (size_t)min(2 * c + pg, G - 1) * L.gs;
        ps = L.scales[o];
        pb = corr[o];
    };
    const auto load_w = [&](uint32_t c, u32x4 (&w)[2]) {
        const size_t o = code_chunk_offset(c * kChunk, kq, K);  // codes past K are not computed
        w[0] = *(const u32x4*)(cpA + o);
        w[1] = *(const u32x4*)(cpB + o);
    };
    const auto stage = [&](uint32_t c, int buf) {
        const bool in = c * kChunk + piece * 8 < K;
#pragma unroll
        for (int i = 0; i < XI; ++i) {
            const uint32_t r = srow + 32 * i;
            if (MT == 1 && r >= 16) continue;
            u32x4 t = xv[i];
            if (!in) t = u32x4{0, 0, 0, 0};
            const int E = group_shift(group_max<8>(bf16x8_exp_max(t)));
            const float se = pow2i(E), so = pow2i(E - 4);
            float f[8];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                f[2 * e] = __uint_as_float(t[e] << 16) * se;
                f[2 * e + 1] = __uint_as_float(t[e] & 0xffff0000u) * so;
            }
            u32x4 q;
            q[0] = permb(__float_as_uint(f[4]), __float_as_uint(f[0]), 0x07060302u);
            q[1] = permb(__float_as_uint(f[5]), __float_as_uint(f[1]), 0x07060302u);
            q[2] = permb(__float_as_uint(f[6]), __float_as_uint(f[2]), 0x07060302u);
            q[3] = permb(__float_as_uint(f[7]), __float_as_uint(f[3]), 0x07060302u);
            lds.xa[buf][piece_pos<4>(piece) * kRowPad + r] = q;
            float sm = 0.0f;
#pragma unroll
            for (int e = 0; e < 4; ++e) sm = dot2_bf16(t[e], 0x3F803F80u, sm);
            sm = group_sum<8>(sm);
            if ((piece & 7) == 0) {
                lds.xe[buf][piece >> 3][r] = 133 - E;
                lds.xs[c & 3][piece >> 3][r] = sm;
            }
        }
        lds.pl[c & 3][pg][pr] = ps | (pb << 16);
    };

    f32x4 acc[MT][2];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m][0] = acc[m][1] = f32x4{0, 0, 0, 0};
    const uint32_t bmask = L.corr ? 0xffff0000u : 0u;
    // Products of chunk c's first ng groups, from LDS buffer buf and codes w.
    const auto compute = [&](uint32_t c, int buf, u32x4 (&w)[2], uint32_t ng) {
        const uint32_t* pl = &lds.pl[c & 3][0][32 * wave + col];
        // words of group 0 (half 0) and group 1 (half 1): [tile][half][MFMA]
        uint32_t u[2][2][2];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const auto p = __builtin_amdgcn_permlane32_swap(w[t][2 * j], w[t][2 * j + 1], false, false);
                u[t][0][j] = p[0] ^ (SIGNED ? 0x88888888u : 0u);
                u[t][1][j] = p[1] ^ (SIGNED ? 0x88888888u : 0u);
            }
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            if ((uint32_t)g >= ng) break;
            bf16x8 b[2][2];
            float sc[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                b[t][0] = codes8(u[t][g][0]);
                b[t][1] = codes8(u[t][g][1]);
                sc[t] = __uint_as_float(pl[g * kCols + 16 * t] << 16);
            }
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const u32x4* a = &lds.xa[buf][(8 * g + kq) * kRowPad + 16 * m + col];
                const bf16x8 a0 = __builtin_bit_cast(bf16x8, a[0]);
                const bf16x8 a1 = __builtin_bit_cast(bf16x8, a[4 * kRowPad]);
                const i32x4 xe = *(const i32x4*)&lds.xe[buf][g][16 * m + 4 * kq];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    f32x4 v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b[t][0], f32x4{0, 0, 0, 0}, 0, 0, 0);
                    v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b[t][1], v, 0, 0, 0);
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[m][t][e] = fmaf(sc[t], ldexp_f32(v[e], xe[e]), acc[m][t][e]);
                    // keeps the flush here: moved past the staging and the barrier, it would hold every block's sums live
                    asm volatile("" : "+v"(acc[m][t]));
                }
            }
        }
    };
    // Bias terms of the n <= 4 groups of chunks c and c + 1: rank-4 products in f32.
    const auto bias = [&](uint32_t c, uint32_t n) {
        const bool on = kq < n;
        const uint32_t slot = (c + (kq >> 1)) & 3;
        float bt[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const uint32_t p = lds.pl[slot][kq & 1][32 * wave + col + 16 * t];
            const uint32_t b = (p & bmask) | (__float_as_uint(-8.0f * __uint_as_float(p << 16)) & ~bmask);
            bt[t] = on ? __uint_as_float(b) : 0.0f;
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const float xs = on ? lds.xs[slot][kq & 1][16 * m + col] : 0.0f;
#pragma unroll
            for (int t = 0; t < 2; ++t)
                acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(xs, bt[t], acc[m][t], 0, 0, 0);
        }
    };

    // Chunk c computes from LDS buffer c % 2 and code set c % 2. The prefetches
    // past the last chunk are clamped to it (their buffers are not computed).
    const uint32_t last = chunks - 1, tail = G - 2 * last;  // groups of the last chunk
    load_xp(0);
    load_w(0, wv[0]);
    stage(0, 0);
    load_xp(min(1u, last));
    load_w(min(1u, last), wv[1]);
    lds_barrier();
    uint32_t c = 0;
    for (; c + 2 <= last; c += 2) {
        compute(c, 0, wv[0], 2);
        stage(c + 1, 1);
        load_xp(c + 2);
        load_w(c + 2, wv[0]);
        lds_barrier();
        compute(c + 1, 1, wv[1], 2);
        bias(c, 4);
        stage(c + 2, 0);
        load_xp(min(c + 3, last));
        load_w(min(c + 3, last), wv[1]);
        lds_barrier();
    }
    compute(c, 0, wv[0], c == last ? tail : 2);
    if (c < last) {
        stage(c + 1, 1);
        lds_barrier();
        compute(c + 1, 1, wv[1], tail);
    }
    bias(c, G - 2 * c);

    if (!live) return;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t r = 16 * m + 4 * kq + e;
            if (r >= cnt) continue;
            uint16_t* o = L.out + (size_t)lds.route[r] * N + n0 + col;
            if (UP) {
                o[0] = gated_silu(acc[m][0][e], acc[m][1][e]);
            } else {
                o[0] = f32_to_bf16_bits(acc[m][0][e]);
                o[16] = f32_to_bf16_bits(acc[m][1][e]);
            }
        }
}

template <bool UP, bool SIGNED>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4))) void moe_group(MoeGroup L) {
    __shared__ GroupLds lds;
    const uint32_t slot = blockIdx.x / L.tiles, tile = blockIdx.x % L.tiles;
    if (slot >= L.header[0]) return;
    const uint32_t expert = L.table[4 * slot], first = L.table[4 * slot + 1], cnt = L.table[4 * slot + 2];
    if (threadIdx.x < kSlot) lds.route[threadIdx.x] = L.sorted[first + min(threadIdx.x, cnt - 1)];
    __syncthreads();
    if (cnt <= 16)
        group_tile<UP, SIGNED, 1>(L, lds, expert, cnt, tile);
    else if (cnt <= 32)
        group_tile<UP, SIGNED, 2>(L, lds, expert, cnt, tile);
    else if (cnt <= 48)
        group_tile<UP, SIGNED, 3>(L, lds, expert, cnt, tile);
    else
        group_tile<UP, SIGNED, 4>(L, lds, expert, cnt, tile);
}

// Counting sort of the routes by expert and the slot records (expert, first
// entry of sorted[], count): one workgroup. An expert's routes are cut into
// slots of equal 16-row blocks, so none is left with a remainder of a few.
__global__ __launch_bounds__(1024) void moe_group_slots(const uint32_t* ids, uint32_t routes, uint32_t experts,
                                                        uint32_t* sorted, uint32_t* table, uint32_t* header) {
    __shared__ uint32_t cnt[1024], off[1024], wsum[2][16];
    const uint32_t t = threadIdx.x, lane = t & 63, wave = t >> 6;
    cnt[t] = 0;
    __syncthreads();
    for (uint32_t r = t; r < routes; r += 1024) {
        uint32_t e = ids[r];
        e = e < experts ? e : 0;  // out-of-range ids read expert 0's rows (MoeGatherRows, moe.rs:87-107)
        atomicAdd(&cnt[e], 1u);
    }
    __syncthreads();
    // exclusive scans of the route counts and the slot counts over the experts
    const uint32_t c = cnt[t], n = (c + kSlot - 1) / kSlot;
    uint32_t ic = c, in = n;
    for (uint32_t d = 1; d < 64; d <<= 1) {
        const uint32_t u = __shfl_up(ic, d, 64), v = __shfl_up(in, d, 64);
        if (lane >= d) {
            ic += u;
            in += v;
        }
    }
    if (lane == 63) {
        wsum[0][wave] = ic;
        wsum[1][wave] = in;
    }
    __syncthreads();
    uint32_t pc = 0, pn = 0;
    for (uint32_t w = 0; w < wave; ++w) {
        pc += wsum[0][w];
        pn += wsum[1][w];
    }
    const uint32_t first = pc + ic - c;
    off[t] = first;
    if (n) {
        const uint32_t step = ((c + n - 1) / n + 15) / 16 * 16;  // rows per slot, at most 64
        uint32_t* rec = table + 4 * (pn + in - n);
        for (uint32_t s = 0; s < n; ++s, rec += 4) {
            const uint32_t a = min(s * step, c);
            rec[0] = t;
            rec[1] = first + a;
            rec[2] = min(step, c - a);
        }
    }
    if (t == 1023) header[0] = pn + in;
    __syncthreads();
    for (uint32_t r = t; r < routes; r += 1024) {
        uint32_t e = ids[r];
        e = e < experts ? e : 0;
        sorted[atomicAdd(&off[e], 1u)] = r;
    }
}

}  // namespace

stark_qmm_status launch_moe_group_slots(const uint32_t* ids, uint32_t routes, uint32_t experts, uint32_t* sorted,
                                        uint32_t* table, uint32_t* header, hipStream_t stream) {
    hipLaunchKernelGGL(moe_group_slots, dim3(1), dim3(1024), 0, stream, ids, routes, experts, sorted, table, header);
    QMM_HIP_CHECK(hipGetLastError());
    return STARK_QMM_OK;
}

stark_qmm_status launch_moe_group(MoeGroup g, bool up, bool signed_codes, uint32_t routes, uint32_t experts,
                                  hipStream_t stream) {
    // every expert in use has a slot, and one more per 64 routes at most
    const uint32_t slots = std::min(routes, experts + routes / kSlot);
    const uint32_t cols = up ? 16 * kWaves : kCols;
    g.tiles = ((up ? g.hidden : g.model) + cols - 1) / cols;
    const dim3 grid(slots * g.tiles);
    if (up) {
        if (signed_codes) hipLaunchKernelGGL((moe_group<true, true>), grid, dim3(kThreads), 0, stream, g);
        else hipLaunchKernelGGL((moe_group<true, false>), grid, dim3(kThreads), 0, stream, g);
    } else {
        if (signed_codes) hipLaunchKernelGGL((moe_group<false, true>), grid, dim3(kThreads), 0, stream, g);
        else hipLaunchKernelGGL((moe_group<false, false>), grid, dim3(kThreads), 0, stream, g);
    }
    QMM_HIP_CHECK(hipGetLastError());
    return STARK_QMM_OK;
}

}  // namespace qmm
