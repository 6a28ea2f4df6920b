// Rules by which a launch picks its kernel or its shape from the sizes of its
// products: plain C++, so that a CPU test can ask which one a size gets. Op is
// any type with the rows m, columns n and depth k of a product.
#pragma once
#include <algorithm>
#include <cstdint>

namespace qmm {

// ---- Int8 activations, weight-streaming kernel (qmv_a8_dense.hip).

// Shapes (16-row blocks, waves along K of eight), two workgroups per CU each,
// and the measured time of one pass of 128 kw values with the second workgroup
// of each CU (full) and without (half), in us; a round also pays about 4 us of
// first loads and last sums.
struct A8Shape {
    int mt, kw;
    double full, half;
};
inline constexpr A8Shape kA8Shapes[] = {{1, 8, 1.5, 1.0}, {2, 8, 2.3, 1.65}, {2, 4, 2.1, 1.25}, {2, 2, 2.0, 1.1},
                                        {4, 2, 3.1, 1.8}, {4, 1, 2.5, 1.65}};
inline constexpr int kA8ShapeCount = sizeof(kA8Shapes) / sizeof(kA8Shapes[0]);

template <class Op>
uint64_t a8_shape_tiles(const A8Shape& s, const Op& o) {
    const uint32_t cols = 32 * (8 / s.kw), rows = 16 * s.mt;
    return (uint64_t)((o.n + cols - 1) / cols) * ((o.m + rows - 1) / rows);
}

// Estimated time of the launch in a shape: whole rounds of two workgroups per CU, and the rest.
template <class Op>
double a8_shape_cost(const A8Shape& s, const Op* ops, uint32_t count, uint32_t cus) {
    uint64_t tiles = 0;
    double passes = 0;
    for (uint32_t i = 0; i < count; ++i) {
        const uint64_t t = a8_shape_tiles(s, ops[i]);
        tiles += t;
        passes += (double)t * ((ops[i].k + 128 * s.kw - 1) / (128 * s.kw));
    }
    passes /= std::max<uint64_t>(tiles, 1);
    const uint64_t rounds = tiles / (2 * cus), rest = tiles % (2 * cus);
    const double full = 4.0 + passes * s.full, half = 4.0 + passes * s.half;
    return rounds * full + (rest > cus ? full : rest ? half : 0.0);
}

// The shape of a launch; few: the first one, whose sums are the most exact
// (products that ran on qmv_a8 before: up to 16 rows, or past the GEMM's bounds).
template <class Op>
int a8_shape(const Op* ops, uint32_t count, bool few, uint32_t cus) {
    int best = 0;
    double cost = 0;
    for (int i = 0; i < (few ? 1 : kA8ShapeCount); ++i) {
        const double c = a8_shape_cost(kA8Shapes[i], ops, count, std::max(cus, 1u));
        if (i == 0 || c < cost) {
            best = i;
            cost = c;
        }
    }
    return best;
}

// One product of one or two rows whose columns are few: 32 a workgroup leave
// most CUs idle, where qmv_a8 gives each a wave. us, qmv_a8 and streaming:
//   4-bit, one row, K 4096: N 1024 5.5 6.7; 2304 6.4 6.8; 3072 6.8 6.8; 3584 7.2 6.9
//     K 1024: N 1024 3.2 3.6; 2304 3.9 4.1; 2560 4.5 4.3   K 512: N 512 3.4 3.4; 1536 3.6 3.5
//     K 8192: N 2048 9.1 10.2; 3072 10.2 11.1; 3584 11.3 11.3
//   4-bit, two rows, K 4096: N 1024 6.3 6.8; 1536 6.8 6.8   K 1024: slower from N 256
//   8-bit, one row, K 1024: N 1024 3.5 4.6; 3584 4.8 4.8; 4608 5.2 4.9   K 512: N 4608 4.3 4.8
//     K 2048: N 1024 4.6 5.5; 1536 5.8 5.5   K 4096: N 512 6.5 7.3; 1024 7.7 7.4   K 8192: N 256 10.5 11.4
//   8-bit, two rows, K 1024: N 2304 4.4 4.8; 2560 5.1 4.9   K 512: N 3072 4.3 4.7; 3584 4.6 4.7
inline bool a8_wave_per_row(uint32_t m, uint32_t n, uint32_t k, int bits, uint32_t cus) {
    if (m < 1 || m > 2) return false;
    if (bits == 4) {
        if (m == 2) return n <= 4 * cus && k >= 2048;
        return n <= (k >= 2048 ? 12 : k >= 1024 ? 9 : 2) * cus;
    }
    const uint64_t unit = 1024ull * cus, weights = (uint64_t)n * k;
    if (m == 2) return k <= 1024 && weights <= 9 * unit;
    return weights <= (k <= 1024 ? 14 : 8) * unit;
}

}  // namespace qmm
