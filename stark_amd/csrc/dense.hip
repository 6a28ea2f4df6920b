// Full-precision GEMV used for MatmulB::FullPrecision operands (e.g. the MoE
// router, a bf16 [experts, model] matrix; crates/stark-engine/src/encodable_block/mlp/qwen_moe.rs:64).
// Per output the reference multiplies and adds sequentially in f32
// (crates/stark-engine/src/backends/cpu/kernel/matmul/kernel.rs:206-218, 267); here one
// wave owns a row and reduces 64 lane-partials (sums agree to f32 rounding).
#include "qmm_common.h"

namespace qmm {

namespace {

__global__ __launch_bounds__(256) void gemv_dense_rows(DenseOp op) {
    const int lane = threadIdx.x & 63;
    const uint32_t n = blockIdx.x * 4 + (threadIdx.x >> 6);
    const uint32_t m = blockIdx.y;
    if (n >= op.n) return;
    const size_t row = op.gather ? op.gather[(size_t)m * op.n + n] : n;
    const size_t o = (size_t)m * op.n + n;
    if (row >= op.bank_rows) {
        if (lane == 0) store_from_f32(op.d, op.d_dt, o, __builtin_nanf(""));
        return;
    }
    float acc = 0.0f;
    for (uint32_t k = lane; k < op.k; k += 64) {
        const float a = load_as_f32(op.x, op.x_dt, (size_t)m * op.k + k);
        const float w = load_as_f32(op.w, op.w_dt, row * op.ld + k);
        acc = fmaf(a, w, acc);
    }
    acc = wave_sum(acc);
    if (lane == 0) {
        float v = op.ab_scale * acc;
        if (op.flags & FLAG_ACCUMULATE) v += load_as_f32(op.d, op.d_dt, o);
        if (op.bias) v += load_as_f32(op.bias, op.w_dt, n);
        if (op.flags & FLAG_SOFT_CAP) v = op.soft_cap * tanhf(v / op.soft_cap);
        store_from_f32(op.d, op.d_dt, o, v);
    }
}

// The wave sums of V values (a power of two up to 64), each in the order of
// wave_sum: while several values are left, the halves of the wave exchange, so
// that a lane adds for one of two values. Returns the sum of value
// lane / (64 / V).
template <int V, int OFF = 32>
__device__ __forceinline__ float wave_sums(float (&v)[V], int lane) {
    if constexpr (V == 1) {
        float t = v[0];
#pragma unroll
        for (int off = OFF; off >= 1; off >>= 1) t += __shfl_xor(t, off, 64);
        return t;
    } else {
        float h[V / 2];
#pragma unroll
        for (int j = 0; j < V / 2; ++j) {
            const uint32_t a = __float_as_uint(v[j]), b = __float_as_uint(v[j + V / 2]);
            if constexpr (OFF == 32) {
                const auto p = __builtin_amdgcn_permlane32_swap(a, b, false, false);
                h[j] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
            } else if constexpr (OFF == 16) {
                const auto p = __builtin_amdgcn_permlane16_swap(a, b, false, false);
                h[j] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
            } else {
                const bool up = lane & OFF;
                h[j] = (up ? v[j + V / 2] : v[j]) + __shfl_xor(up ? v[j] : v[j + V / 2], OFF, 64);
            }
        }
        return wave_sums<V / 2, OFF / 2>(h, lane);
    }
}

// bf16 x and w, no gather, 16-byte aligned rows: one workgroup for R weight rows
// and MT activation rows; its four waves split K (8 values per lane per load)
// and meet in LDS. Rows past the last repeat it, so that all loads of a step are
// issued before the first is waited for. The order of a sum depends on neither
// R nor MT. What bounded it were the wave sums, six exchanges through LDS for
// each output and wave; wave_sums takes 10 for 8 outputs and 32 for 32, most of
// them lane swaps. A router of 128 rows, K = 2048, at 1, 8, 64, 512 and 2048
// rows: 3.8, 4.5, 5.8, 23.1, 79 -> 2.4, 2.7, 3.7, 7.5, 22.7 us; 30000 rows,
// K = 1024, 8 rows: 66.9 -> 15.2 us (4.0 TB/s). Those read one matrix over and
// over; between the other kernels of a layer the router takes 4.5 and 8.7 us at 4
// and 512 rows.
template <int MT, int R>
__global__ __launch_bounds__(256) void gemv_dense_bf16(DenseOp op) {
    __shared__ float part[4][R][MT];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t n0 = blockIdx.x * R, m0 = blockIdx.y * MT;
    const uint16_t* w = (const uint16_t*)op.w;
    const uint16_t* x = (const uint16_t*)op.x;
    float acc[R * MT];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[r * MT + t] = 0.0f;
    for (uint32_t k = (wave * 64 + lane) * 8; k < op.k; k += 2048) {
        u32x4 wv[R], xv[MT];
#pragma unroll
        for (int r = 0; r < R; ++r) wv[r] = *(const u32x4*)(w + (size_t)min(n0 + r, op.n - 1) * op.ld + k);
#pragma unroll
        for (int t = 0; t < MT; ++t) xv[t] = *(const u32x4*)(x + (size_t)min(m0 + t, op.m - 1) * op.k + k);
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[r * MT + t] = dot2_bf16(wv[r][e], xv[t][e], acc[r * MT + t]);
    }
    constexpr int V = R * MT;
    const float sum = wave_sums<V>(acc, lane);
    if (lane % (64 / V) == 0) (&part[wave][0][0])[lane / (64 / V)] = sum;
    __syncthreads();
    const uint32_t r = threadIdx.x / MT, t = threadIdx.x % MT;
    if (r < (uint32_t)R && n0 + r < op.n && m0 + t < op.m) {
        const float total = (part[0][r][t] + part[1][r][t]) + (part[2][r][t] + part[3][r][t]);
        const size_t o = (size_t)(m0 + t) * op.n + n0 + r;
        float v = op.ab_scale * total;
        if (op.flags & FLAG_ACCUMULATE) v += load_as_f32(op.d, op.d_dt, o);
        if (op.bias) v += load_as_f32(op.bias, op.w_dt, n0 + r);
        if (op.flags & FLAG_SOFT_CAP) v = op.soft_cap * tanhf(v / op.soft_cap);
        store_from_f32(op.d, op.d_dt, o, v);
    }
}

// B stored [K, ld] (b_transpose = false): thread per output.
__global__ __launch_bounds__(256) void gemv_dense_cols(DenseOp op) {
    const uint32_t n = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t m = blockIdx.y;
    if (n >= op.n) return;
    const size_t col = op.gather ? op.gather[(size_t)m * op.n + n] : n;
    const size_t o = (size_t)m * op.n + n;
    if (col >= op.bank_rows) {
        store_from_f32(op.d, op.d_dt, o, __builtin_nanf(""));
        return;
    }
    float acc = 0.0f;
    for (uint32_t k = 0; k < op.k; ++k)
        acc = fmaf(load_as_f32(op.x, op.x_dt, (size_t)m * op.k + k), load_as_f32(op.w, op.w_dt, k * op.ld + col), acc);
    float v = op.ab_scale * acc;
    if (op.flags & FLAG_ACCUMULATE) v += load_as_f32(op.d, op.d_dt, o);
    if (op.bias) v += load_as_f32(op.bias, op.w_dt, n);
    if (op.flags & FLAG_SOFT_CAP) v = op.soft_cap * tanhf(v / op.soft_cap);
    store_from_f32(op.d, op.d_dt, o, v);
}

}  // namespace

stark_qmm_status launch_dense_gemv(const DenseOp& op, hipStream_t stream) {
    if (op.n == 0 || op.m == 0) return STARK_QMM_OK;
    const bool fast = op.transpose && op.w_dt == STARK_QMM_BF16 && op.x_dt == STARK_QMM_BF16 && !op.gather &&
                      op.k % 8 == 0 && op.ld % 8 == 0 && (((uintptr_t)op.w | (uintptr_t)op.x) & 15) == 0;
    if (fast) {
        // four weight rows a workgroup once those give every CU two (128 rows,
        // K = 2048, one against four: 64 activation rows 3.72 and 3.45 us, 32
        // rows 3.13 and 3.31)
        const uint32_t mb = (op.m + 7) / 8;
        int dev = 0, cus = 0;
        QMM_HIP_CHECK(hipGetDevice(&dev));
        QMM_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        const bool four = (uint64_t)((op.n + 3) / 4) * mb >= 2 * (uint64_t)cus;
        if (op.m == 1) hipLaunchKernelGGL((gemv_dense_bf16<1, 1>), dim3(op.n), dim3(256), 0, stream, op);
        else if (op.m <= 4) hipLaunchKernelGGL((gemv_dense_bf16<4, 1>), dim3(op.n), dim3(256), 0, stream, op);
        else if (four) hipLaunchKernelGGL((gemv_dense_bf16<8, 4>), dim3((op.n + 3) / 4, mb), dim3(256), 0, stream, op);
        else hipLaunchKernelGGL((gemv_dense_bf16<8, 1>), dim3(op.n, mb), dim3(256), 0, stream, op);
    } else if (op.transpose) {
        hipLaunchKernelGGL(gemv_dense_rows, dim3((op.n + 3) / 4, op.m), dim3(256), 0, stream, op);
    } else {
        hipLaunchKernelGGL(gemv_dense_cols, dim3((op.n + 255) / 256, op.m), dim3(256), 0, stream, op);
    }
    QMM_HIP_CHECK(hipGetLastError());
    return STARK_QMM_OK;
}

}  // namespace qmm
