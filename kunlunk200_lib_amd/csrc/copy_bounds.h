// Source offsets of the LDS copies of the wide prefill tiles, and the step whose
// bytes a copy takes. Plain functions of integers, so that a host program can walk
// every copy of a call (tests/copy_bounds_walk.cpp): each one must lie inside the
// matrix, or have a lane offset past the buffer's extent (zeros, no access), without
// the scalar offset being counted in the bounds check.
#pragma once

#include <cstdint>

#ifdef __HIPCC__
#define KK_HOST_DEVICE __attribute__((host)) __attribute__((device)) __attribute__((always_inline)) inline
#else
#define KK_HOST_DEVICE inline
#endif

namespace kk {

// Copies run ahead of the products: what would lie past the last step is the last
// step again (into a slot that nobody reads).
KK_HOST_DEVICE int copied_step(int step, int steps) { return step < steps ? step : steps - 1; }

// The row of its tile that weight row `r` is copied from: past the matrix (`left` rows
// from the tile's first) its last row again.
KK_HOST_DEVICE uint32_t tile_row(int r, int left) { return static_cast<uint32_t>(r < left ? r : left - 1); }

// f16_wide_gemm, 1 KiB copy `i` (below 32 KG) of a step: the weight byte of lane `lane`
// within the tile's rows. PAIR: copied rows 128 .. 255 are the up matrix's.
template <int KG, bool PAIR>
KK_HOST_DEVICE uint32_t wide_f16_weight(int i, int lane, int left, uint32_t row_bytes) {
    constexpr int kChunks = 4 * KG, kRowsPerCopy = 64 / kChunks;
    const int r = kRowsPerCopy * i + lane / kChunks, pos = lane % kChunks;
    const int swizzle = KG == 1 ? (r >> 2) & 3 : (r >> 1) & 7;
    return tile_row(PAIR ? r & 127 : r, left) * row_bytes + 16u * static_cast<uint32_t>(pos ^ swizzle);
}

// q4_wide_gemm, 1 KiB copy `i` of a super-stage (144 bytes of each of 256 rows): 36 of
// them, and four whose lanes lie past any extent. PAIR: copies 18 .. 35 are the up matrix's.
template <bool PAIR>
KK_HOST_DEVICE uint32_t wide_q4_weight(int i, int lane, int left, uint32_t row_bytes) {
    if (i >= 36) return 0x80000000u;
    const int q = (PAIR && i >= 18 ? i - 18 : i) * 64 + lane;
    return tile_row(q / 9, left) * row_bytes + 16u * static_cast<uint32_t>(q % 9);
}

} // namespace kk
