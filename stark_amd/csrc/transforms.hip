// Activation transforms around the quantized products, on gfx950:
//  - ActivationTransform (crates/stark-engine/src/backends/cpu/kernel/activation_transform/activation_transform.rs:48-156):
//    input RHT (x * factors, then the 32-point Walsh-Hadamard transform),
//    output RHT (transform, then * factors, optional bias), and symmetric int8
//    quantization of the input-RHT result (scale per 32/64/128 values, codes
//    in sequential or grouped-by-nibble order, optional int32 group sums);
//  - GatedActMul (crates/stark-engine/src/backends/cpu/kernel/gated_act_mul/gated_act_mul.rs:17-152):
//    value * activation(gate) in the storage type, optional clipping and SiLU
//    alpha, optional RHT and int8 quantization;
//  - the output-RHT D-op of the products (kernel.rs:287-300), which runs the
//    output transform in place on d and adds the bias after it.
// A thread owns 8 consecutive values of a row, so every load and store of a
// wave covers whole lines; four consecutive lanes hold a 32-value stripe and 4,
// 8 or 16 a scale group. The butterfly runs in the reference's order (pairs
// (l, l|s) for s = 1, 2, .., 16; distances 8 and 16 through DPP), then the
// scale 1/sqrt(32) as the reference computes it, so every float matches the
// CPU restatement. What bounds it is memory for the plain transforms (512 x
// 4096 bf16 quantized: 58 -> 5 us; one thread per scale group read and wrote
// strided lines) and the division and expf of each value for the gated ones
// (512 x 12288 bf16 SiLU, quantized: 169 -> 18 us).
#include "qmm_common.h"

// The reference evaluates `a * b + c` as a rounded product and a rounded sum;
// no contraction into fma here, so the floats match the CPU restatement.
#pragma clang fp contract(off)

namespace qmm {
namespace {

constexpr int kBlock = 32;  // HADAMARD_TRANSFORM_BLOCK_SIZE (gpu_types/hadamard_order.rs:1)

__device__ __forceinline__ float ld(const void* p, uint32_t dt, size_t i) { return load_as_f32(p, dt, i); }
__device__ __forceinline__ void st(void* p, uint32_t dt, size_t i, float v) { store_from_f32(p, dt, i, v); }
__device__ __forceinline__ float rnd(uint32_t dt, float v) {
    return dt == STARK_QMM_BF16 ? bf16_bits_to_f32(f32_to_bf16_bits(v)) : v;
}

constexpr int kVec = 8;  // values per thread

// 8 f32 or bf16 values at element i (vec: 16-byte aligned there).
__device__ __forceinline__ void ld8(const void* p, uint32_t dt, size_t i, bool vec, float (&v)[kVec]) {
    if (!vec) {
#pragma unroll
        for (int e = 0; e < kVec; ++e) v[e] = ld(p, dt, i + e);
    } else if (dt == STARK_QMM_F32) {
        const u32x4 a = *(const u32x4*)((const float*)p + i), b = *(const u32x4*)((const float*)p + i + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = __uint_as_float(a[e]);
            v[4 + e] = __uint_as_float(b[e]);
        }
    } else {
        const u32x4 a = *(const u32x4*)((const uint16_t*)p + i);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[2 * e] = __uint_as_float(a[e] << 16);
            v[2 * e + 1] = __uint_as_float(a[e] & 0xffff0000u);
        }
    }
}

// The same of a bias, which has the plane type of its product and so may be f16 too.
__device__ __forceinline__ void bias8(const void* p, uint32_t dt, size_t i, bool vec, float (&v)[kVec]) {
    ld8(p, dt, i, vec && dt != STARK_QMM_F16, v);
}

__device__ __forceinline__ void st8(void* p, uint32_t dt, size_t i, bool vec, const float (&v)[kVec]) {
    if (!vec) {
#pragma unroll
        for (int e = 0; e < kVec; ++e) st(p, dt, i + e, v[e]);
    } else if (dt == STARK_QMM_F32) {
        u32x4 a, b;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            a[e] = __float_as_uint(v[e]);
            b[e] = __float_as_uint(v[4 + e]);
        }
        *(u32x4*)((float*)p + i) = a;
        *(u32x4*)((float*)p + i + 4) = b;
    } else {
        u32x4 a;
#pragma unroll
        for (int e = 0; e < 4; ++e) a[e] = f32_to_bf16_bits(v[2 * e]) | ((uint32_t)f32_to_bf16_bits(v[2 * e + 1]) << 16);
        *(u32x4*)((uint16_t*)p + i) = a;
    }
}

// RHT signs of 8 values (vec: 16-byte aligned there).
__device__ __forceinline__ void signs8(const int32_t* f, size_t i, bool vec, float (&v)[kVec]) {
    if (vec) {
        const u32x4 a = *(const u32x4*)(f + i), b = *(const u32x4*)(f + i + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = (float)(int32_t)a[e];
            v[4 + e] = (float)(int32_t)b[e];
        }
    } else {
#pragma unroll
        for (int e = 0; e < kVec; ++e) v[e] = (float)f[i + e];
    }
}

// activation_transform/mod.rs:28-43 over the 32 values of four consecutive
// lanes (q: this lane's place among them).
__device__ __forceinline__ void hadamard32(float (&v)[kVec], uint32_t q) {
#pragma unroll
    for (int s = 1; s < kVec; s <<= 1)
#pragma unroll
        for (int l = 0; l < kVec; ++l)
            if ((l & s) == 0) {
                const float a = v[l], b = v[l | s];
                v[l] = a + b;
                v[l | s] = a - b;
            }
#pragma unroll
    for (int l = 0; l < kVec; ++l) {
        const float o = dpp_f32<DPP_XOR1>(v[l]);  // distance 8
        v[l] = (q & 1) ? o - v[l] : v[l] + o;
    }
#pragma unroll
    for (int l = 0; l < kVec; ++l) {
        const float o = dpp_f32<DPP_XOR2>(v[l]);  // distance 16
        v[l] = (q & 2) ? o - v[l] : v[l] + o;
    }
    const float scale = 1.0f / __fsqrt_rn((float)kBlock);
#pragma unroll
    for (int l = 0; l < kVec; ++l) v[l] *= scale;
}

// Sum over 4, 8 or 16 consecutive lanes.
__device__ __forceinline__ int32_t lanes_sum(int32_t v, uint32_t lanes) {
    v += (int32_t)dpp_u32<DPP_XOR1>((uint32_t)v);
    v += (int32_t)dpp_u32<DPP_XOR2>((uint32_t)v);
    const int32_t v8 = v + (int32_t)dpp_u32<DPP_HALF_MIRROR>((uint32_t)v);
    const int32_t v16 = v8 + (int32_t)dpp_u32<DPP_MIRROR>((uint32_t)v8);
    return lanes == 4 ? v : lanes == 8 ? v8 : v16;
}

// mod.rs:9-26 on one scale group of LANES consecutive lanes (this lane: values
// k .. k + 7 of the row); writes codes (layout order, Int8CodeLayout::index,
// matmul_a.rs:31-46), the scale and the group sums.
template <int LANES>
__device__ __forceinline__ void quantize_group(const float (&t)[kVec], uint32_t k, bool grouped, uint32_t sum_group,
                                               bool vec, int8_t* q, float* scales, int32_t* sums) {
    float m = 0.0f;  // the largest |t| that is a number
#pragma unroll
    for (int i = 0; i < kVec; ++i) m = fmaxf(m, fabsf(t[i]));
    m = __uint_as_float(group_max<LANES>(__float_as_uint(m)));
    const float divisor = (isfinite(m) && m > 0.0f) ? m / 127.0f : 1.0f;
    const uint32_t lane = (k / kVec) % LANES;
    if (lane == 0) scales[k / (kVec * LANES)] = divisor;
    int8_t c[kVec];
    int32_t sum = 0;
#pragma unroll
    for (int i = 0; i < kVec; ++i) {
        const float r = roundf(t[i] / divisor);
        c[i] = isnan(r) ? (int8_t)0 : (int8_t)fminf(fmaxf(r, -127.0f), 127.0f);
        sum += c[i];
    }
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    u32x2 w = {0, 0};
#pragma unroll
    for (int i = 0; i < kVec; ++i) {
        // grouped by nibble: values (0, 2, 4, 6) then (1, 3, 5, 7)
        const uint32_t b = (uint32_t)(uint8_t)c[i];
        const int g = (i & 1) * 4 + i / 2;
        w[g / 4] |= (grouped ? b : 0u) << (8 * (g % 4));
        w[i / 4] |= (grouped ? 0u : b) << (8 * (i % 4));
    }
    if (vec) {
        *(u32x2*)(q + k) = w;
    } else {
#pragma unroll
        for (int i = 0; i < kVec; ++i) q[k + i] = (int8_t)(w[i / 4] >> (8 * (i % 4)));
    }
    if (sums) {
        const int32_t total = lanes_sum(sum, sum_group / kVec);
        if (k % sum_group == 0) sums[k / sum_group] = total;
    }
}

struct TransformArgs {
    const void* input;     // T, or NULL (in place: read fp_out)
    void* fp_out;          // T
    const void* bias;      // BiasT or NULL
    int8_t* q_out;
    float* scales_out;
    int32_t* sums_out;
    const int32_t* factors;
    uint32_t batch, count, op, grouped, scale_group, sum_group, t_dt, bias_dt;
    uint32_t vec_in, vec_out;  // operands read / results written are aligned for 16-byte (codes 8-byte) access
};

// ActivationTransform: thread = 8 values; LANES lanes per scale group (4 for the FP ops).
template <int LANES>
__global__ __launch_bounds__(256) void activation_transform(TransformArgs a) {
    const uint32_t per_row = a.count / kVec;
    const uint32_t item = blockIdx.x * 256 + threadIdx.x;
    if (item >= a.batch * per_row) return;
    const uint32_t row = item / per_row, k = item % per_row * kVec;
    const size_t ro = (size_t)row * a.count;
    const void* src = a.input ? a.input : a.fp_out;
    const bool input_rht = a.op != 1;
    float v[kVec], f[kVec];
    ld8(src, a.t_dt, ro + k, a.vec_in, v);
    signs8(a.factors, k, a.vec_in, f);
    if (input_rht) {
#pragma unroll
        for (int e = 0; e < kVec; ++e) v[e] *= f[e];
    }
    hadamard32(v, item);
    if (!input_rht) {
#pragma unroll
        for (int e = 0; e < kVec; ++e) v[e] *= f[e];
    }
    if (a.op >= 2) {  // Quantize / QuantizeWithGroupSums
        quantize_group<LANES>(v, k, a.grouped != 0, a.sum_group, a.vec_out, a.q_out + ro,
                              a.scales_out + (size_t)row * (a.count / a.scale_group),
                              a.op == 3 ? a.sums_out + (size_t)row * (a.count / a.sum_group) : nullptr);
        return;
    }
    if (a.bias) {
        float b[kVec];
        bias8(a.bias, a.bias_dt, k, a.vec_in, b);
#pragma unroll
        for (int e = 0; e < kVec; ++e) v[e] = rnd(a.t_dt, v[e]) + b[e];
    }
    st8(a.fp_out, a.t_dt, ro + k, a.vec_out, v);
}

// ActivationType::activate (gpu_types/activation_type.rs:19-111) on a value
// stored in dt; every bf16 operation of the materialized forms rounds.
__device__ __forceinline__ float activate(uint32_t type, float x, uint32_t dt, bool has_alpha, float alpha) {
    constexpr float K0 = 0.044715f, K1 = 0.7978846f;
    switch (type) {
    case STARK_QMM_ACT_SILU: {
        const float al = has_alpha ? alpha : 1.0f;
        return rnd(dt, x / (1.0f + expf(-al * x)));
    }
    case STARK_QMM_ACT_SILU_MATERIALIZED_SIGMOID: {
        const float e = rnd(dt, expf(fabsf(x)));
        const float lower = rnd(dt, 1.0f / rnd(dt, 1.0f + e));
        const float sig = x < 0.0f ? lower : rnd(dt, 1.0f - lower);
        return rnd(dt, x * sig);
    }
    case STARK_QMM_ACT_GELU_APPROX: {
        const float arg = K1 * (x + K0 * x * x * x);
        return rnd(dt, 0.5f * x * (1.0f + tanhf(arg)));
    }
    case STARK_QMM_ACT_GELU_MATERIALIZED_POLYNOMIAL: {
        const float cubic = rnd(dt, x * x * x);
        const float term = rnd(dt, rnd(dt, K0) * cubic);
        const float inner = rnd(dt, x + term);
        const float arg = rnd(dt, rnd(dt, K1) * inner);
        const float act = rnd(dt, tanhf(arg));
        return rnd(dt, rnd(dt, 0.5f * x) * rnd(dt, 1.0f + act));
    }
    case STARK_QMM_ACT_GELU_EXACT: return rnd(dt, 0.5f * x * (1.0f + erff(x * 0.70710677f)));
    case STARK_QMM_ACT_SOFTPLUS: return x > 20.0f ? x : rnd(dt, logf(1.0f + expf(x)));
    default: return x;  // identity
    }
}

__device__ __forceinline__ float clamp_f(float x, float lo, float hi) { return x < lo ? lo : (x > hi ? hi : x); }

struct GatedArgs {
    const void* act;
    const void* value;     // separate value operand, or NULL (interleaved)
    void* fp_out;
    int8_t* q_out;
    float* scales_out;
    int32_t* sums_out;
    const int32_t* factors;  // RHT signs or NULL
    uint32_t gated_dim, batch, value_offset, value_row_stride, act_type, has_alpha;
    float alpha, gate_min, gate_max, value_min, value_max;
    uint32_t clip_gate, clip_value, op, grouped, scale_group, sum_group, t_dt;
    uint32_t vec_in, vec_out;  // as TransformArgs
};

__device__ __forceinline__ float gated_one(const GatedArgs& a, float value, float gate) {
    if (a.clip_gate) gate = rnd(a.t_dt, clamp_f(gate, a.gate_min, a.gate_max));
    const bool alpha = a.has_alpha && a.act_type == STARK_QMM_ACT_SILU;
    const float activated = activate(a.act_type, gate, a.t_dt, alpha, a.alpha);
    if (a.clip_value) value = rnd(a.t_dt, clamp_f(value, a.value_min, a.value_max));
    return rnd(a.t_dt, value * activated);
}

// First elements of row `batch` of the gate and value operands.
__device__ __forceinline__ void gated_rows(const GatedArgs& a, size_t batch, const void*& value, size_t& gi, size_t& vi) {
    value = a.value ? a.value : a.act;
    gi = a.value ? batch * a.gated_dim : batch * 2 * a.gated_dim + a.gated_dim;
    vi = a.value ? batch * a.value_row_stride + a.value_offset : batch * 2 * a.gated_dim;
}

// GatedActMul: thread = 8 values; LANES lanes per scale group when quantizing.
template <int LANES>
__global__ __launch_bounds__(256) void gated_act_mul(GatedArgs a) {
    const uint32_t per_row = a.gated_dim / kVec;
    const uint32_t item = blockIdx.x * 256 + threadIdx.x;
    if (item >= a.batch * per_row) return;
    const size_t batch = item / per_row;
    const uint32_t k = item % per_row * kVec;
    const void* value;
    size_t gi, vi;
    gated_rows(a, batch, value, gi, vi);
    float v[kVec], g[kVec];
    ld8(value, a.t_dt, vi + k, a.vec_in, v);
    ld8(a.act, a.t_dt, gi + k, a.vec_in, g);
#pragma unroll
    for (int e = 0; e < kVec; ++e) v[e] = gated_one(a, v[e], g[e]);
    if (a.factors) {
        signs8(a.factors, k, a.vec_in, g);
#pragma unroll
        for (int e = 0; e < kVec; ++e) v[e] *= g[e];
        hadamard32(v, item);
    }
    if (a.op != 0) {
        quantize_group<LANES>(v, k, a.grouped != 0, a.sum_group, a.vec_out, a.q_out + batch * a.gated_dim,
                              a.scales_out + batch * (a.gated_dim / a.scale_group),
                              a.op == 2 ? a.sums_out + batch * (a.gated_dim / a.sum_group) : nullptr);
        return;
    }
    st8(a.fp_out, a.t_dt, batch * a.gated_dim + k, a.vec_out, v);
}

// Few values, or rows of no whole number of 8 (no RHT): thread = one value.
__global__ __launch_bounds__(256) void gated_act_mul_one(GatedArgs a) {
    const uint32_t item = blockIdx.x * 256 + threadIdx.x;
    if (item >= a.batch * a.gated_dim) return;
    const size_t batch = item / a.gated_dim;
    const uint32_t k = item % a.gated_dim;
    const void* value;
    size_t gi, vi;
    gated_rows(a, batch, value, gi, vi);
    st(a.fp_out, a.t_dt, batch * a.gated_dim + k, gated_one(a, ld(value, a.t_dt, vi + k), ld(a.act, a.t_dt, gi + k)));
}

// sg: scale group of the quantizing ops, else 32; items: threads.
template <template <int> class K, class Args>
stark_qmm_status launch_by_group(uint32_t sg, uint32_t items, const Args& a, hipStream_t stream) {
    if (items == 0) return STARK_QMM_OK;
    const dim3 grid((items + 255) / 256);
    switch (sg) {
    case 32: hipLaunchKernelGGL(K<4>::fn(), grid, dim3(256), 0, stream, a); break;
    case 64: hipLaunchKernelGGL(K<8>::fn(), grid, dim3(256), 0, stream, a); break;
    case 128: hipLaunchKernelGGL(K<16>::fn(), grid, dim3(256), 0, stream, a); break;
    default: return STARK_QMM_INVALID_ARGUMENT;
    }
    QMM_HIP_CHECK(hipGetLastError());
    return STARK_QMM_OK;
}

template <int LANES>
struct AT {
    static auto fn() { return activation_transform<LANES>; }
};
template <int LANES>
struct GA {
    static auto fn() { return gated_act_mul<LANES>; }
};

bool aligned(const void* p, size_t n) { return ((uintptr_t)p & (n - 1)) == 0; }

// Rows of `width` values: whole rows per launch, so that the items of one stay 32-bit.
uint32_t rows_per_launch(uint32_t width) { return std::max(1u, 0x7fffffffu / std::max(1u, width)); }

stark_qmm_status run_transform(TransformArgs a, uint32_t sg, hipStream_t stream) {
    a.vec_in = aligned(a.input ? a.input : a.fp_out, 16) && aligned(a.factors, 16) && aligned(a.bias, 16);
    a.vec_out = a.op >= 2 ? aligned(a.q_out, 8) : aligned(a.fp_out, 16);
    const uint32_t rows = a.batch, step = rows_per_launch(a.count);
    const size_t esz = a.t_dt == STARK_QMM_F32 ? 4 : 2;
    for (uint32_t r = 0; r < rows; r += step) {
        TransformArgs b = a;
        b.batch = std::min(step, rows - r);
        const size_t e = (size_t)r * a.count;
        if (a.input) b.input = (const uint8_t*)a.input + e * esz;
        if (a.fp_out) b.fp_out = (uint8_t*)a.fp_out + e * esz;
        if (a.q_out) b.q_out = a.q_out + e;
        if (a.scales_out) b.scales_out = a.scales_out + e / a.scale_group;
        if (a.sums_out && a.sum_group) b.sums_out = a.sums_out + e / a.sum_group;
        const stark_qmm_status s = launch_by_group<AT>(sg, b.batch * (a.count / kVec), b, stream);
        if (s != STARK_QMM_OK) return s;
        if (rows - r <= step) break;
    }
    return STARK_QMM_OK;
}

stark_qmm_status run_gated(GatedArgs a, uint32_t sg, hipStream_t stream) {
    const size_t esz = a.t_dt == STARK_QMM_F32 ? 4 : 2;
    // One value a thread where 8 a thread leave the chip waiting for the divisions
    // and exponentials of one after the other: no RHT, up to 3072 values a CU (bf16
    // SiLU of 4096-value rows: 1 row 2.8 against 4.6 us, 128 rows 4.1 and 4.9, 192 rows
    // 5.0 and 5.1, 256 rows 6.1 and 5.1), and rows of no whole 8 values.
    int dev = 0, cus = 0;
    QMM_HIP_CHECK(hipGetDevice(&dev));
    QMM_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const bool rows8 = a.gated_dim % kVec == 0 &&
                       (a.factors || (uint64_t)a.batch * a.gated_dim > 3072ull * (uint64_t)cus);
    a.vec_in = aligned(a.act, 16) && aligned(a.factors, 16) &&
               (!a.value || (aligned((const uint8_t*)a.value + (size_t)a.value_offset * esz, 16) &&
                             a.value_row_stride * esz % 16 == 0));
    a.vec_out = a.op != 0 ? aligned(a.q_out, 8) : aligned(a.fp_out, 16);
    const uint32_t rows = a.batch, step = rows_per_launch(a.gated_dim);
    for (uint32_t r = 0; r < rows; r += step) {
        GatedArgs b = a;
        b.batch = std::min(step, rows - r);
        const size_t e = (size_t)r * a.gated_dim;
        b.act = (const uint8_t*)a.act + e * esz * (a.value ? 1 : 2);
        if (a.value) b.value = (const uint8_t*)a.value + (size_t)r * a.value_row_stride * esz;
        if (a.fp_out) b.fp_out = (uint8_t*)a.fp_out + e * esz;
        if (a.q_out) b.q_out = a.q_out + e;
        if (a.scales_out) b.scales_out = a.scales_out + e / a.scale_group;
        if (a.sums_out && a.sum_group) b.sums_out = a.sums_out + e / a.sum_group;
        if (rows8) {
            const stark_qmm_status s = launch_by_group<GA>(sg, b.batch * (a.gated_dim / kVec), b, stream);
            if (s != STARK_QMM_OK) return s;
        } else {
            const uint32_t items = b.batch * a.gated_dim;
            if (items) hipLaunchKernelGGL(gated_act_mul_one, dim3((items + 255) / 256), dim3(256), 0, stream, b);
            QMM_HIP_CHECK(hipGetLastError());
        }
        if (rows - r <= step) break;
    }
    return STARK_QMM_OK;
}

bool float_dt(uint32_t dt) { return dt == STARK_QMM_F32 || dt == STARK_QMM_BF16; }

}  // namespace

stark_qmm_status launch_output_rht(void* d, uint32_t d_dt, const void* bias, uint32_t bias_dt,
                                   const int32_t* factors, uint32_t rows, uint32_t n, hipStream_t stream) {
    TransformArgs a{};
    a.fp_out = d;
    a.bias = bias;
    a.factors = factors;
    a.batch = rows;
    a.count = n;
    a.op = STARK_QMM_TRANSFORM_OUTPUT_RHT;
    a.t_dt = d_dt;
    a.bias_dt = bias_dt;
    a.scale_group = kBlock;
    return run_transform(a, kBlock, stream);
}

}  // namespace qmm

using namespace qmm;

extern "C" {

stark_qmm_status stark_qmm_activation_transform(const stark_qmm_activation_transform_args* args, void* stream) {
    if (!args || args->struct_size != sizeof(stark_qmm_activation_transform_args)) return STARK_QMM_ABI_MISMATCH;
    const stark_qmm_activation_transform_args& x = *args;
    if (x.op > STARK_QMM_TRANSFORM_QUANTIZE_WITH_GROUP_SUMS || !float_dt(x.data_type) ||
        (x.bias && !float_dt(x.bias_data_type)))
        return STARK_QMM_UNSUPPORTED_DATA_TYPE;
    if (!x.rht_factors || x.element_count % kBlock) return STARK_QMM_INVALID_ARGUMENT;
    const bool quantize = x.op >= STARK_QMM_TRANSFORM_QUANTIZE;
    uint32_t sg = kBlock;
    if (quantize) {
        // ActivationQuantization::new (activation_transform.rs:27-42)
        sg = x.scale_group_size;
        if (!(sg == 32 || sg == 64 || sg == 128) || x.element_count % sg || !x.q_out || !x.scales_out)
            return STARK_QMM_INVALID_ARGUMENT;
        if (x.op == STARK_QMM_TRANSFORM_QUANTIZE_WITH_GROUP_SUMS &&
            (!(x.sum_group_size == 32 || x.sum_group_size == 64 || x.sum_group_size == 128) ||
             x.sum_group_size > sg || !x.group_sums_out))
            return STARK_QMM_INVALID_ARGUMENT;
    } else if (!x.output) {
        return STARK_QMM_INVALID_ARGUMENT;
    }
    TransformArgs a{};
    a.input = x.in_place ? nullptr : x.input;
    if (!x.in_place && !x.input) return STARK_QMM_INVALID_ARGUMENT;
    a.fp_out = x.output;
    a.bias = x.bias;
    a.q_out = x.q_out;
    a.scales_out = x.scales_out;
    a.sums_out = x.group_sums_out;
    a.factors = x.rht_factors;
    a.batch = x.batch_size;
    a.count = x.element_count;
    a.op = x.op;
    a.grouped = x.grouped_by_nibble;
    a.scale_group = sg;
    a.sum_group = x.sum_group_size;
    a.t_dt = x.data_type;
    a.bias_dt = x.bias_data_type;
    return run_transform(a, sg, (hipStream_t)stream);
}

stark_qmm_status stark_qmm_gated_act_mul(const stark_qmm_gated_act_mul_args* args, void* stream) {
    if (!args || args->struct_size != sizeof(stark_qmm_gated_act_mul_args)) return STARK_QMM_ABI_MISMATCH;
    const stark_qmm_gated_act_mul_args& x = *args;
    if (!float_dt(x.data_type)) return STARK_QMM_UNSUPPORTED_DATA_TYPE;
    if (x.act_type > STARK_QMM_ACT_GELU_MATERIALIZED_POLYNOMIAL || x.op > STARK_QMM_GATED_QUANTIZE_WITH_GROUP_SUMS ||
        !x.act_operand)
        return STARK_QMM_INVALID_ARGUMENT;
    if (!x.interleaved && !x.value_operand) return STARK_QMM_INVALID_ARGUMENT;
    // gated_act_mul.rs:46-51
    const bool quantize = x.op != STARK_QMM_GATED_FULL_PRECISION;
    if (quantize && !x.hadamard_factors) return STARK_QMM_INVALID_ARGUMENT;  // quantized gate activation requires RHT
    if (x.hadamard_factors && x.gated_dim % kBlock) return STARK_QMM_INVALID_ARGUMENT;
    uint32_t sg = kBlock;
    if (quantize) {
        sg = x.scale_group_size;
        if (!(sg == 32 || sg == 64 || sg == 128) || x.gated_dim % sg || !x.q_out || !x.scales_out)
            return STARK_QMM_INVALID_ARGUMENT;
        if (x.op == STARK_QMM_GATED_QUANTIZE_WITH_GROUP_SUMS &&
            (!(x.sum_group_size == 32 || x.sum_group_size == 64 || x.sum_group_size == 128) ||
             x.sum_group_size > sg || !x.group_sums_out))
            return STARK_QMM_INVALID_ARGUMENT;
    } else if (!x.fp_out) {
        return STARK_QMM_INVALID_ARGUMENT;
    }
    GatedArgs a{};
    a.act = x.act_operand;
    a.value = x.interleaved ? nullptr : x.value_operand;
    a.fp_out = x.fp_out;
    a.q_out = x.q_out;
    a.scales_out = x.scales_out;
    a.sums_out = x.group_sums_out;
    a.factors = x.hadamard_factors;
    a.gated_dim = x.gated_dim;
    a.batch = x.batch_dim;
    a.value_offset = x.value_offset;
    a.value_row_stride = x.value_row_stride;
    a.act_type = x.act_type;
    a.has_alpha = x.has_activation_alpha;
    a.alpha = x.activation_alpha;
    a.clip_gate = x.clip_gate;
    a.gate_min = x.gate_clip_min;
    a.gate_max = x.gate_clip_max;
    a.clip_value = x.clip_value;
    a.value_min = x.value_clip_min;
    a.value_max = x.value_clip_max;
    a.op = x.op;
    a.grouped = x.grouped_by_nibble;
    a.scale_group = sg;
    a.sum_group = x.sum_group_size;
    a.t_dt = x.data_type;
    return run_gated(a, sg, (hipStream_t)stream);
}

}  // extern "C"
