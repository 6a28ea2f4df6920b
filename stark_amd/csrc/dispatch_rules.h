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

// ---- Prompt products of 17 to 128 rows, group 64: qgemm_stream, whose workgroups
// take 32 or 64 columns by one of equal row blocks (at most 64 rows), two a CU, or
// the GEMM (128 rows by 64 columns, one a CU) past 64 rows.

// 16-row blocks of a workgroup.
template <class Op>
uint32_t stream_blocks(const Op* ops, uint32_t count) {
    uint32_t m = 0;
    for (uint32_t i = 0; i < count; ++i) m = std::max(m, ops[i].m);
    const uint32_t blocks = (m + 63) / 64;
    return std::max(2u, (m + 16 * blocks - 1) / (16 * blocks));
}

// 64-column workgroups of a launch.
template <class Op>
uint64_t stream_tiles(const Op* ops, uint32_t count) {
    const uint32_t rows = 16 * stream_blocks(ops, count);
    uint64_t tiles = 0;
    for (uint32_t i = 0; i < count; ++i) tiles += (uint64_t)((ops[i].n + 63) / 64) * ((ops[i].m + rows - 1) / rows);
    return tiles;
}

// 64 columns a workgroup (each LDS read feeds two matrix products) instead of
// 32: from 1.5 workgroups a CU on (64 rows of the seven products of 4096 / 12288,
// 608: 71.9 against 77.9 us; of 2560 / 6912, 356: 37.7 against 32.2; 32 rows, N
// 20480, K 4096, 320: 29.4 and 29.2, N 28672, 448: 29.9 against 35.6), and with 33
// rows and more of one depth already where 32 columns make between one and three
// a CU (64 rows, K 4096: N 8192, 128 workgroups of 64 columns 22.8 against 16.3; N
// 10240, 160: 22.9 against 26.6; 96 rows, N 10240, 320: 28.9 against 30.4, K 2048
// 17.5 against 16.1). With few columns a workgroup the activations come from L2
// too often for 25 to 32 rows of a deep product (N 12288, K 12288: 17 rows 42.7 us,
// 32 rows 52.1, 64 columns 49.9).
template <class Op>
bool stream_wide(const Op* ops, uint32_t count, uint32_t cus) {
    const uint64_t tiles = stream_tiles(ops, count);
    if (2 * tiles > 3 * (uint64_t)cus) return true;
    uint32_t k = 0;
    for (uint32_t i = 0; i < count; ++i) {
        if (ops[i].k != ops[0].k) return false;
        k = ops[i].k;
    }
    return stream_blocks(ops, count) > 2 && 2 * tiles > cus && (tiles <= cus || k > 2048);
}

// Whether a launch's products of more than 64 rows run on qgemm_stream. One
// depth: by its 64-column workgroups a CU. The GEMM's tiles are as many as half
// of them, and full past 112 rows. us, GEMM and here, K 4096, 4-bit: 97 rows, N 8192
// (1.0) 32.4 22.5, 10240 (1.25) 32.6 30.5, 12288 (1.5) 32.7 34.3, 28672 50.9 64.1; 96
// rows, 12288 32.7 31.9, 16384 (2.0) 33.5 32.6 (8-bit, K 12288: 100.7 104.8), 20480
// (2.5) 48.6 46.4 (K 1024: 16.3 16.9), 28672 (3.5) 51.1 58.5; 128 rows, 8192 30.9 22.9, 10240 31.2 31.7
// (8-bit 35.0 32.6, K 2048 19.6 19.9), 12288 31.4 36.3. Several depths: the GEMM
// takes what its deepest product's serial K loop takes, about 7.8 ns a value of K,
// or, with tiles enough, 0.5 us for 2^20 weights, where this kernel takes 0.55:
// here from 62 values of K for 10^6 weights (97 rows, seven products: 1024 / 1024
// (176) 13.9 and 10.0, 2560 / 6912 (99) 53 and 44, 4096 / 12288 (64) 103.5 and 100,
// 4096 / 8192 (57) 73.6 and 81.5), past 112 rows with a deep product only (128 rows
// of 1536 / 1536 (118) 15.6 and 16.9, 2048 / 2048 (89) 19.3 and 21.2).
template <class Op>
bool stream_takes(const Op* ops, uint32_t count, int bits, uint32_t cus) {
    double weights = 0, k = 0;
    uint32_t m = 0;
    bool mixed = false;
    for (uint32_t i = 0; i < count; ++i) {
        weights += 1e-6 * ops[i].n * ops[i].k;
        k = std::max(k, (double)ops[i].k);
        m = std::max(m, ops[i].m);
        mixed = mixed || ops[i].k != ops[0].k;
    }
    if (mixed) return k >= 62 * weights && (m <= 112 || k >= 2816 || k >= 150 * weights);
    const double fill = (double)stream_tiles(ops, count) / cus;
    if (m <= 96) return fill <= 1.5 || (fill > 2.0 && fill <= 2.5 && k > 1024);
    if (m <= 112) return fill <= (k > 2048 ? 1.25 : 1.0);
    return fill <= (k > 512 ? 1.0 : 0.75) || (bits == 8 && fill <= 1.25 && k > 2048);
}

// ---- Sampling: whether a call takes the split form (pieces of a row on several
// workgroups, in three to seven launches) or the row form (one launch, a
// workgroup a row, two a CU). us, row and split form:
//   greedy, 1 to 48 rows: 16384 logits 11.2 to 11.9 and 14.0 to 15.2; 16385 more
//     than in the split form, 151936 nine times (one row)
//   greedy, 64 rows: 16385 alike; 96: 24000 alike; 128: 20000 1.24 times longer
//     split, 32000 0.95; 192 and 256: 24000 1.4 and 1.55, 32000 0.77 and 0.96
//   greedy, 512 rows (two rounds of scratch slots): 32000 1.54, 65536 1.12
//   sampled, up to 128 rows: shorter split at every size (256 logits, one row:
//     temperature 38 and 16, top-p 44 and 29; 4096: 49 and 17, 143 and 89)
//   sampled, 512 rows with filters: 64 logits 1.3 to 1.5 times longer split, 4096
//     1.0 to 1.1, 16384 0.8 to 1.0; temperature alone 1.0 to 0.6
inline bool sample_split(uint32_t vocab, uint32_t rows, bool sampled, bool filters) {
    if (!sampled) return vocab > (rows <= 64 ? 16384u : rows <= 256 ? 28000u : 80000u);
    return vocab > 1 && !(filters && rows > 256 && vocab <= 16384);
}

// ---- Routed experts: whether a call of group-64 banks takes the grouped products
// of a prompt (moe_group.hip), whose workgroups are 128 up rows by 64 routes of
// one expert. From 17 tokens on (us against the slot form of fewer tokens, model /
// hidden / experts / active: 17 tokens, 2048/768/128/8 77 against 156, 1024/512/
// 128/2 29 and 38, 2048/512/32/2 33 and 48, 512/512/2/2 25 and 31, 256/128/4/1 17
// and 29), but for one expert of up to 64 tokens, which is one slot on a few
// workgroups (2048/1024: 24 tokens 42.8 against 32.5, 64 64.3 and 57.6; 128 65.8 and
// 100.8), unless it is small (512/256: 21 to 32 against 29 to 36).
inline bool moe_grouped(uint32_t tokens, uint32_t experts, uint32_t model, uint32_t hidden) {
    return tokens > 16 && (experts > 1 || tokens > 64 || (uint64_t)model * hidden <= 384 * 1024);
}

// ---- Products of up to 16 rows, group 64: qmv_dense (32-column tiles, two
// workgroups per CU, 1024 values a pass) or qmv_mfma (16-column tiles, three per
// CU, in 64-column groups dealt to the XCDs). Over the products of one launch.

// Columns and 32-column tiles of a launch, and the depth that most of its weights have.
struct LaunchSize {
    uint64_t columns = 0, tiles = 0;
    uint32_t k = 0;
    bool mixed = false;  // products of different depths
    bool even = true;    // qmv_mfma's groups come out even over the eight XCDs: a multiple of 512 columns in all
};
template <class Op>
LaunchSize launch_size(const Op* ops, uint32_t count) {
    LaunchSize z;
    double most = -1;
    for (uint32_t i = 0; i < count; ++i) {
        z.columns += ops[i].n;
        z.tiles += (ops[i].n + 31) / 32;
        z.mixed = z.mixed || ops[i].k != ops[0].k;
        z.even = z.even && ops[i].n % 64 == 0;
        double weights = 0;
        for (uint32_t j = 0; j < count; ++j) weights += ops[j].k == ops[i].k ? (double)ops[j].n * ops[j].k : 0.0;
        if (weights > most) {
            most = weights;
            z.k = ops[i].k;
        }
    }
    z.even = z.even && z.columns % 512 == 0;
    return z;
}

// One or two rows.
// idle: 4-bit, whose qmv_mfma passes of 2048 values run past K: all are dense, in
// one launch (hidden 3072 / 8192, seven products: 19.9 us with the 8192-deep one
// on its own kernel, 15.1 together, 16.3 on qmv_mfma). One depth: from 15% of the
// weights walked for nothing on (two of 6912 x 2560, 38%: 9.1 against 7.5 us;
// 9984 x 3328, 19%: 11.7 and 11.7). Products of several depths, whose tiles the
// lists of qmv_mfma even out better: from 19.5% (3072 / 8192, 20%: above;
// 1536 / 6144, 19%: 8.4 against 9.4; 3328 / 9984, 15%: 17.9 against 20.2), and not
// when its columns come out even and the dense tiles are few (1024 / 2048 to
// 4096, 42 to 46%: 4.7 to 5.8 against 5.4 to 6.6).
// drag: products beside one whose planes qmv_mfma cannot read join it: a second
// launch costs 3 to 6 us (8-bit 2560 / 6912: 23.3 against 26.5; 4-bit 2048 / 5568:
// 9.3 against 15.2), the dense kernel about 10% of their time, which is more from
// 160 MB on.
struct FewRowsRule {
    bool idle, drag;
};
template <class Op, class Readable>
FewRowsRule few_rows_rule(const Op* ops, uint32_t count, int bits, uint32_t cus, Readable readable) {
    double walked = 0, used = 0, others = 0;
    bool unreadable = false, mixed = false;
    for (uint32_t i = 0; i < count; ++i) {
        const Op& o = ops[i];
        mixed = mixed || o.k != ops[0].k;
        walked += (double)o.n * ((o.k + 2047) / 2048 * 2048);
        used += (double)o.n * o.k;
        if (!readable(o)) unreadable = true;
        else others += (double)o.n * o.k * bits / 8;
    }
    bool idle = bits == 4 && used < (mixed ? 0.805 : 0.85) * walked;
    if (idle && mixed) {
        const LaunchSize z = launch_size(ops, count);
        idle = !(z.even && 2 * z.tiles <= 3 * (uint64_t)cus);
    }
    return {idle, unreadable && others < 160e6};
}

// Whether a launch of 4-bit products of 9 to 16 rows, all of which it can take,
// stays with qmv_small_m: what that saves is the activation stage of each 32
// columns, through its runs, and those need many passes (32 columns x 1024
// values) for each of its two resident workgroups a CU (16 rows: 11.5 passes
// each on the seven products of 4096 / 12288, 154 us for four layers against
// 169; 5.9 at 3072 / 8192, 109 against 106; 2.2 at 2048 / 6144, 87 against 62).
template <class Op>
bool small_m_long(const Op* ops, uint32_t count, uint32_t cus) {
    uint64_t units = 0;
    for (uint32_t i = 0; i < count; ++i) units += (uint64_t)((ops[i].n + 31) / 32) * (ops[i].k / 1024);
    return units >= 8 * 2 * (uint64_t)cus;
}

// Whether qmv_mfma takes a launch's 8-bit products of 5 to 8 rows, all of which
// it can read. Its columns have to come out even (else some workgroup has two
// tiles where others have one: N 6912, K 4096 21.1 us against 10.1), and it is then
// the faster one where the dense tiles come out badly: between one and 1.5 a CU
// (N 12288, eight rows, K 1024 5.8 against 7.1, 2560 1.16 times, 4096 16.2 against
// 16.9, 12288 39.8 against 45.1; at two passes, K 1025 to 2048, alike), and where
// K is an odd number of passes, one above all (K 1024: N 4096 4.2 against 4.7,
// 24576 9.6 against 10.9, 8192 and 16384 alike, two of 4096 5.1 against 5.5; N
// 27648: K 3072 25.4 against 27.1, 5120 39.1 against 43.0, 4096 32.6 against 30.3,
// 7168 52.6 against 54.4). Of several depths and many tiles also without even
// columns (seven products, hidden 2304 / 6912 22.9 against 24.6, 2560 / 6912 25.1
// against 26.1, 5120 / 13824 72.2 against 75.2; 4096 / 11008 47.0 against 44.5).
template <class Op>
bool w8_rows5_mfma(const Op* ops, uint32_t count, uint32_t cus) {
    if (count == 0) return false;
    const LaunchSize z = launch_size(ops, count);
    const uint32_t passes = (z.k + 1023) / 1024;
    const bool many = z.tiles > 2 * (uint64_t)cus;
    if (z.mixed && many) return passes % 2 == 1 && passes <= 5;
    if (!z.even) return false;
    if (z.tiles > cus && 2 * z.tiles <= 3 * (uint64_t)cus) return passes != 2;
    if (passes == 1) return many || (16 * z.tiles >= 3 * (uint64_t)cus && (count > 1 ? 1 : 2) * z.tiles <= cus);
    return many && z.k % 2048 == 1024 && passes <= 5;
}

}  // namespace qmm
