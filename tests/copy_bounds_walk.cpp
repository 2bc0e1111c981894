// Walks the weight copies of the wide prefill tiles (csrc/copy_bounds.h) over every step
// that a call of K = k issues, for tiles with `left` weight rows, and requires of each
// 16-byte lane that it lies inside those rows or has a lane offset past the buffer's
// extent: in range whether or not the bounds check counts the scalar (step) offset.
#include "copy_bounds.h"

#include <cstdio>
#include <initializer_list>

static long walked = 0, bad = 0;

static void lane_ok(const char *kernel, int k, int left, int step, uint32_t lane_off, uint32_t step_off, uint32_t extent) {
    ++walked;
    if (lane_off >= extent || uint64_t{lane_off} + step_off + 16 <= extent) return;
    if (bad++ < 5)
        std::printf("%s k=%d rows=%d copy of step %d: bytes %u + %u .. +15 of %u\n", kernel, k, left, step, lane_off,
                    step_off, extent);
}

// f16_wide_gemm: steps 0 .. 2 first, then step s + 3 in step s
template <int KG, bool PAIR>
static void f16(int k, int left) {
    const int steps = k / (32 * KG);
    const uint32_t row = 2u * k, extent = row * left;
    for (int s = 0; s < steps + 3; ++s)
        for (int i = 0; i < 32 * KG / 2; ++i)
            for (int lane = 0; lane < 64; ++lane)
                lane_ok("f16_wide_gemm", k, left, s, kk::wide_f16_weight<KG, PAIR>(i, lane, left, row),
                        static_cast<uint32_t>(kk::copied_step(s, steps)) * (64 * KG), extent);
}

// q4_wide_gemm: super-stage 0 first, then super-stage p + 1 during super-stage p
template <bool PAIR>
static void q4(int k, int left) {
    const int supers = k / 256;
    const uint32_t row = k / 32 * 18u, extent = row * left;
    for (int p = 0; p < supers + 1; ++p)
        for (int i = 0; i < 40; ++i)
            for (int lane = 0; lane < 64; ++lane)
                lane_ok("q4_wide_gemm", k, left, p, kk::wide_q4_weight<PAIR>(i, lane, left, row),
                        static_cast<uint32_t>(kk::copied_step(p, supers)) * 144, extent);
}

int main() {
    for (int k : {32, 64, 96, 320, 4096, 5600, 16384})
        for (int left : {1, 2, 33, 127, 128, 255, 256}) {
            f16<1, false>(k, left);
            if (left <= 128) f16<1, true>(k, left);
            if (k % 64 == 0) f16<2, false>(k, left);
            if (k % 64 == 0 && left <= 128) f16<2, true>(k, left);
            if (k % 256 == 0) q4<false>(k, left);
            if (k % 256 == 0 && left <= 128) q4<true>(k, left);
        }
    std::printf("%ld lanes, %ld outside\n", walked, bad);
    return bad != 0;
}
