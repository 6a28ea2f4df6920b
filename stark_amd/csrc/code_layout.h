// Where in a weight row the codes lie that a lane of the streaming kernels
// loads. Plain C++ besides the qualifiers, so the bounds are checked on the CPU.
#pragma once
#include <cstdint>

#if defined(__HIP__)
#define QMM_HOST_DEVICE __host__ __device__ inline
#else
#define QMM_HOST_DEVICE inline
#endif

namespace qmm {

// Byte offset in its row (K values of BITS bits, K % 64 == 0) of the 16 bytes
// that lane quarter kq loads for the 128-value chunk at k. 4-bit: the 32 codes
// at k + 32 kq; 8-bit: two loads h, of the 16 codes at k + 64 h + 16 kq. Past K
// the row's first bytes, which are not computed; all 16 lie in the row.
template <int BITS>
QMM_HOST_DEVICE uint32_t code_offset(uint32_t k, uint32_t h, uint32_t kq, uint32_t K) {
    static_assert(BITS == 4 || BITS == 8, "packed codes");
    const uint32_t kl = BITS == 4 ? k + 32 * kq : k + 64 * h + 16 * kq;
    return kl < K ? kl / (8 / BITS) : 0;
}

// The 4-bit offset in two parts, for a kernel that has no register for a third
// address: the lane's, added to its row once, and the chunk's. Past K the lane's
// part stays: 16 kq + 16 bytes are in every row of 128 values and more, and in
// a row of 64 (32 bytes) quarters 2 and 3 have none (left there, they read up to
// 32 bytes past the last row of the codes).
QMM_HOST_DEVICE uint32_t code_lane_offset(uint32_t kq, uint32_t K) { return 32 * kq < K ? 16 * kq : 0; }
QMM_HOST_DEVICE uint32_t code_chunk_offset(uint32_t k, uint32_t kq, uint32_t K) { return k + 32 * kq < K ? k / 2 : 0; }

// Place of 8-value piece v of a pass in MFMA order (what the loads above make of
// a row). 4-bit: within a 64-value group, piece 4 (kq & 1) + 2 j + (kq >> 1)
// belongs to lane quarter kq of the group's j-th MFMA (permlane32_swap of 16-byte
// loads); 8-bit: piece 2 kq + j.
template <int BITS>
QMM_HOST_DEVICE uint32_t piece_pos(uint32_t v) {
    const uint32_t p = v & 7;
    return (v & ~7u) + (BITS == 4 ? 4 * ((p >> 1) & 1) + ((p >> 2) | ((p & 1) << 1)) : 4 * (p & 1) + (p >> 1));
}

}  // namespace qmm
