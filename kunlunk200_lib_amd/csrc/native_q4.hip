// GEMV over the native Q4 layout (reference src/q4-layout.cpp:15-37,
// src/k200.cpp:554-617) on gfx950.
//
// Layout: for N32 tile t and K32 block b, 512 bytes at (t * blocks + b) * 512
// hold byte [pair j][lane r] = signed nibbles of row 32t + r, K 32b + 2j (low)
// and 32b + 2j + 1 (high); after the 256-byte aligned payload, 32 FP16 block
// scales per tile-block at (t * blocks + b) * 32 + r. Rows past N are zero.
//
// Arithmetic is exact up to the activation representation: each 32-value
// activation block is a 23-bit signed fixed point with a power-of-two block
// scale s_b (kk::fixed_point_digits), so sum_j q_j X_j is an exact int32 from
// 24 v_dot8_i32_i4 per row and block, and y_r += float(S) * (d_rb * s_b) in F32.
//
// native_q4_gemv (one column, two on small matrices; native_q4_mfma below takes the rest):
// one workgroup per half tile (16 rows); the two halves of a tile
// run on the same XCD (workgroup i runs on XCD i % 8), so the second reads the
// tile's cache lines from L2. The workgroup's waves take items of 16 K32
// blocks in turn. In an item, lane l owns block 16i + l/4 and rows
// 16h + 4(l%4) .. +3: it loads the 16 pair dwords of those rows (stride 32
// bytes; the 4 lanes of a block read 16 contiguous bytes per pair) and turns
// each group of four pair dwords into four row dwords of 8 consecutive K
// values with a 4 x 4 byte transpose (8 v_perm_b32). Activation loads are
// issued first, then the first weight items, then the activations are
// converted while the weights are in flight (the memory counter is in order).
// Rows are reduced over lanes, then over waves in a fixed order: results are
// bitwise reproducible.
#include "device_common.h"
#include "launch.h"

#include <algorithm>

namespace {

constexpr int kNqWaves = 8;
constexpr int kNqThreads = 64 * kNqWaves;
constexpr int kNqDepth = 2;                 // items in flight per wave
constexpr int kNqLanesPerBlock = 4;         // 4 lanes x 4 rows = one half tile
constexpr int kNqItemBlocks = 64 / kNqLanesPerBlock;
constexpr int kNqRows = 16;                 // rows per workgroup
constexpr int kNqMaxColumns = 2;            // batch columns per launch (more: native_q4_mfma)
constexpr int kNqMaxPasses = 6;             // activation staging passes (8 values per thread each)
constexpr size_t kNqLdsLimit = 64 * 1024;

size_t lds_bytes(int blocks, int columns) {
    // per column and block: 24 digit dwords and one scale; per wave and
    // column: the workgroup's row partials
    return static_cast<size_t>(columns) * blocks * (96 + 4) + static_cast<size_t>(kNqWaves) * columns * kNqRows * 4;
}

int passes_for(int blocks, int columns) { return (columns * blocks * 4 + kNqThreads - 1) / kNqThreads; }

template <int B, int PASSES>
__global__ __launch_bounds__(kNqThreads) void native_q4_gemv(const uint8_t *__restrict__ w,
                                                            const uint16_t *__restrict__ scales,
                                                            const void *__restrict__ x, int x_f16,
                                                            float *__restrict__ y, int k, int n, int tiles) {
    extern __shared__ uint4 lds4[];
    // workgroup -> (tile, half): i = 16 (t / 8) + t % 8 + 8 h keeps both halves on XCD t % 8
    const int tile = (blockIdx.x >> 4) * 8 + (blockIdx.x & 7);
    const int half = (blockIdx.x >> 3) & 1;
    if (tile >= tiles) return;                    // whole workgroup: no barrier reached yet
    const int blocks = k >> 5;
    const int items = (blocks + kNqItemBlocks - 1) / kNqItemBlocks;
    uint4 *digits = lds4;                                                                      // [B][blocks][6]
    float *block_scale = reinterpret_cast<float *>(lds4 + static_cast<size_t>(B) * blocks * 6);  // [B][blocks]
    float *partial = block_scale + B * blocks;                                                 // [waves][B][16]

    const int lane = threadIdx.x & (kk::kWave - 1);
    const int wid = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int c = lane & (kNqLanesPerBlock - 1);  // rows 16 half + 4c .. +3 of the tile
    const size_t tile_block0 = static_cast<size_t>(tile) * blocks;
    const int row_byte = kNqRows * half + 4 * c;

    // 1. activation loads: thread (b, block, q) of each pass owns values 8q .. 8q+7 of a block
    const int groups = B * blocks * 4;
    float xv[PASSES][8];
#pragma unroll
    for (int pass = 0; pass < PASSES; ++pass) {
        const int g = min(pass * kNqThreads + static_cast<int>(threadIdx.x), groups - 1);
        const int b = g / (blocks * 4);
        const size_t base = static_cast<size_t>(b) * k + static_cast<size_t>(g - b * blocks * 4) * 8;
        if (x_f16) {
            const uint16_t *xh = static_cast<const uint16_t *>(x) + base;
#pragma unroll
            for (int t = 0; t < 8; ++t) xv[pass][t] = kk::half_bits_to_float(xh[t]);
        } else {
            const float *xf = static_cast<const float *>(x) + base;
#pragma unroll
            for (int t = 0; t < 8; ++t) xv[pass][t] = xf[t];
        }
    }
    __builtin_amdgcn_sched_barrier(0);

    // 2. the first weight items
    auto load_item = [&](int s, uint32_t (&buf)[18]) {
        const int it = min(wid + kNqWaves * s, items - 1);
        const int blk = min(it * kNqItemBlocks + lane / kNqLanesPerBlock, blocks - 1);
        const uint8_t *src = w + (tile_block0 + blk) * 512 + row_byte;
#pragma unroll
        for (int p = 0; p < 16; ++p) buf[p] = *reinterpret_cast<const uint32_t *>(src + 32 * p);
        const uint2 sc = *reinterpret_cast<const uint2 *>(scales + (tile_block0 + blk) * 32 + row_byte);
        buf[16] = sc.x;
        buf[17] = sc.y;
    };
    // every wave runs the same count of items (the last ones may add zero);
    // loads beyond that count are skipped by a uniform branch
    const int iters = (items + kNqWaves - 1) / kNqWaves;
    const int iters_padded = (iters + kNqDepth - 1) / kNqDepth * kNqDepth;
    uint32_t ring[kNqDepth][18];
#pragma unroll
    for (int d = 0; d < kNqDepth; ++d) {
        if (d < iters) load_item(d, ring[d]);
        __builtin_amdgcn_sched_barrier(0);
    }

    // 3. activations -> block scale and six digit dwords per 8 values
#pragma unroll
    for (int pass = 0; pass < PASSES; ++pass) {
        const int idx = pass * kNqThreads + static_cast<int>(threadIdx.x);
        const int g = min(idx, groups - 1);
        const int b = g / (blocks * 4);
        const int rem = g - b * blocks * 4;
        float m = 0.0f, bad = 0.0f;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const float a = fabsf(xv[pass][t]);
            bad = (a <= 3.402823466e38f) ? bad : 1.0f;
            m = fmaxf(m, a);
        }
        // the four threads of a block are the lanes of one quad
        m = fmaxf(m, kk::dpp_move<0xb1>(m));
        m = fmaxf(m, kk::dpp_move<0x4e>(m));
        bad = fmaxf(bad, kk::dpp_move<0xb1>(bad));
        bad = fmaxf(bad, kk::dpp_move<0x4e>(bad));
        // 2^(e-1) <= m < 2^e; e >= -100 keeps 2^(22-e) finite
        const int e = max(__builtin_amdgcn_frexp_expf(m), -100);
        uint32_t dig[6];
        kk::fixed_point_digits(xv[pass], ldexpf(1.0f, 22 - e), dig);
        if (idx < groups) {
            uint32_t *dst = reinterpret_cast<uint32_t *>(digits) + static_cast<size_t>(b * blocks) * 24 + rem * 6;
#pragma unroll
            for (int l = 0; l < 6; ++l) dst[l] = dig[l];
            if ((rem & 3) == 0)
                block_scale[b * blocks + (rem >> 2)] = bad != 0.0f ? __builtin_nanf("") : ldexpf(1.0f, e - 22);
        }
    }
    __syncthreads();

    // 4. items: 4 rows x one K32 block per lane
    float acc[B][4];
#pragma unroll
    for (int b = 0; b < B; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[b][r] = 0.0f;

    auto compute_item = [&](int s, const uint32_t (&buf)[18]) {
        const int it = wid + kNqWaves * s;
        const int blk_raw = it * kNqItemBlocks + lane / kNqLanesPerBlock;
        const bool live = it < items && blk_raw < blocks;
        const int blk = min(min(it, items - 1) * kNqItemBlocks + lane / kNqLanesPerBlock, blocks - 1);
        float d[4];
        d[0] = kk::half_bits_to_float(buf[16] & 0xffffu);
        d[1] = kk::half_bits_to_float(buf[16] >> 16);
        d[2] = kk::half_bits_to_float(buf[17] & 0xffffu);
        d[3] = kk::half_bits_to_float(buf[17] >> 16);
        // row dwords: o[r][q] nibble t = row 4c+r, K 8q+t (4 x 4 byte transposes)
        uint32_t o[4][4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t a = buf[4 * q], bb = buf[4 * q + 1], cc = buf[4 * q + 2], dd = buf[4 * q + 3];
            const uint32_t ab_lo = __builtin_amdgcn_perm(bb, a, 0x05010400u);    // a0 b0 a1 b1
            const uint32_t ab_hi = __builtin_amdgcn_perm(bb, a, 0x07030602u);    // a2 b2 a3 b3
            const uint32_t cd_lo = __builtin_amdgcn_perm(dd, cc, 0x05010400u);
            const uint32_t cd_hi = __builtin_amdgcn_perm(dd, cc, 0x07030602u);
            o[0][q] = __builtin_amdgcn_perm(cd_lo, ab_lo, 0x05040100u);          // a0 b0 c0 d0
            o[1][q] = __builtin_amdgcn_perm(cd_lo, ab_lo, 0x07060302u);          // a1 b1 c1 d1
            o[2][q] = __builtin_amdgcn_perm(cd_hi, ab_hi, 0x05040100u);
            o[3][q] = __builtin_amdgcn_perm(cd_hi, ab_hi, 0x07060302u);
        }
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const uint4 *dsrc = digits + (static_cast<size_t>(b) * blocks + blk) * 6;
            uint32_t dg[24];
#pragma unroll
            for (int g = 0; g < 6; ++g) {
                const uint4 v4 = dsrc[g];
                dg[4 * g] = v4.x;
                dg[4 * g + 1] = v4.y;
                dg[4 * g + 2] = v4.z;
                dg[4 * g + 3] = v4.w;
            }
            const float sb = block_scale[b * blocks + blk];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                int t[6];
#pragma unroll
                for (int l = 0; l < 6; ++l) {
                    t[l] = 0;
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        t[l] = __builtin_amdgcn_sdot8(static_cast<int>(o[r][q]), static_cast<int>(dg[q * 6 + l]),
                                                      t[l], false);
                }
                int sum = t[5];
#pragma unroll
                for (int l = 4; l >= 0; --l) sum = (sum << 4) + t[l];
                acc[b][r] = fmaf(static_cast<float>(sum), live ? d[r] * sb : 0.0f, acc[b][r]);
            }
        }
    };

    for (int base = 0; base < iters_padded; base += kNqDepth) {
#pragma unroll
        for (int dpt = 0; dpt < kNqDepth; ++dpt) {
            if (base + dpt < iters) compute_item(base + dpt, ring[dpt]);   // uniform; no loads inside
            if (base + dpt + kNqDepth < iters) load_item(base + dpt + kNqDepth, ring[dpt]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // 5. rows: sum the 16 lanes of each row group (fixed xor order), then the waves
#pragma unroll
    for (int b = 0; b < B; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float v = acc[b][r];
            v += __shfl_xor(v, 4, kk::kWave);
            v += __shfl_xor(v, 8, kk::kWave);
            v += __shfl_xor(v, 16, kk::kWave);
            v += __shfl_xor(v, 32, kk::kWave);
            if (lane < kNqLanesPerBlock) partial[(wid * B + b) * kNqRows + 4 * c + r] = v;
        }
    __syncthreads();
    if (static_cast<int>(threadIdx.x) < kNqRows * B) {
        const int b = threadIdx.x / kNqRows, row = threadIdx.x % kNqRows;
        float v = 0.0f;
#pragma unroll
        for (int wv = 0; wv < kNqWaves; ++wv) v += partial[(wv * B + b) * kNqRows + row];
        const int gr = tile * 32 + kNqRows * half + row;
        if (gr < n) y[static_cast<size_t>(b) * n + gr] = v;
    }
}

template <int B, int PASSES>
hipError_t launch_columns(const uint8_t *w, const uint16_t *scales, const void *x, int x_f16, float *y, int k,
                          int n, hipStream_t stream) {
    const int tiles = (n + 31) / 32;
    const int groups = 16 * ((tiles + 7) / 8);      // 8 tiles x 2 halves per group of 16 workgroups
    const size_t lds = lds_bytes(k >> 5, B);
    hipLaunchKernelGGL((native_q4_gemv<B, PASSES>), dim3(groups), dim3(kNqThreads), lds, stream, w, scales, x,
                       x_f16, y, k, n, tiles);
    return hipGetLastError();
}

template <int B>
hipError_t launch_passes(int passes, const uint8_t *w, const uint16_t *scales, const void *x, int x_f16, float *y,
                         int k, int n, hipStream_t stream) {
    switch (passes) {
    case 1: return launch_columns<B, 1>(w, scales, x, x_f16, y, k, n, stream);
    case 2: return launch_columns<B, 2>(w, scales, x, x_f16, y, k, n, stream);
    case 3: return launch_columns<B, 3>(w, scales, x, x_f16, y, k, n, stream);
    case 4: return launch_columns<B, 4>(w, scales, x, x_f16, y, k, n, stream);
    case 5: return launch_columns<B, 5>(w, scales, x, x_f16, y, k, n, stream);
    case 6: return launch_columns<B, 6>(w, scales, x, x_f16, y, k, n, stream);
    default: return hipErrorInvalidValue;
    }
}

// ---------------------------------------------------------------------------
// native_q4_mfma: more than one column on int8 MFMA (v_mfma_i32_16x16x32_i8, one K32
// block per instruction), up to 5 columns per workgroup.
//
// The activations are the same 23-bit block fixed point, here as three signed
// base-256 digits: the digits of all columns are the 16 operand columns of one
// MFMA, so every block's digit sums are exact as above; each operand column
// accumulates in F32 with the digit's weight in the block scale, and a column's
// three sums meet at the end. (Three MFMAs per block for 16 columns, put together
// per block, need half the VALU operations per column but took 17.6 and 45 us where
// this takes 11 and 29, K4096 and K11008 x N4096 at 16 columns.)
//
// One workgroup per 32-row tile and column group, its 8 waves taking blocks in turn. Lane l reads, for
// K group g = l / 16 and row quad u = (l % 16) / 2, the dwords (4 rows of one pair) of
// pairs g + 8 (l & 1) and that + 4: 128 contiguous bytes of the tile's 512 per 32 lanes and
// instruction. One exchange with the neighbour lane and byte permutes make them rows 2c
// and 2c + 1 (c = l % 16) over the pairs g, g + 4, g + 8, g + 12; each nibble stays in the
// high half of its byte (16 q). D of row set i: register r of lane l is row
// 8 (l / 16) + 2 r + i, column l % 16.
//
// Bound by the CU: the decode, two conversions and a multiply-add per block sum and the
// three loads per block keep a CU busy for about 90 cycles per block of a tile, so 128
// tiles (N4096) leave half the chip idle. us per call before (dot products, 4 columns per pass)
// / after: K4096 x N11008 4 columns 33.8 / 25.4, 16 columns 94 / 47; K4096 x N4096 4 columns
// 22.5 / 20.6, 16 columns 53 / 26; K11008 x N4096 4 columns 48.5 / 30.5, 16 columns 151 / 44;
// about 15 of each are the launch and the wait for the result. 16 waves per workgroup
// take as long (K4096 x N11008: 27.8).
constexpr int kNmWaves = 8, kNmThreads = 64 * kNmWaves;
constexpr int kNmDepth = 4;                  // blocks in flight per wave
constexpr int kNmMaxColumns = 5;             // 15 of the 16 operand columns
constexpr int kNmChunkColumns = 512;         // activation blocks x columns of a chunk, at most
constexpr int kNmGroups = kNmChunkColumns * 4 / kNmThreads;   // groups of 8 activations per thread and chunk
constexpr int kNmStep = kNmWaves * kNmDepth;                  // blocks per chunk are a multiple of this
constexpr int kNmPart = kNmWaves * 16 * 33 * 4;               // the waves' sums
static_assert(kNmChunkColumns / kNmMaxColumns >= kNmStep, "a chunk of every column count");

// Activation blocks in LDS at a time (100 bytes per block and column, 50 KiB at most).
int nm_chunk(int blocks, int columns) {
    return std::min(kNmChunkColumns / columns / kNmStep * kNmStep, (blocks + kNmStep - 1) / kNmStep * kNmStep);
}

typedef int int4v __attribute__((ext_vector_type(4)));
typedef float float2a4 __attribute__((ext_vector_type(2), aligned(4)));

// A barrier after this wave's LDS accesses that leaves its global loads in flight
// (__syncthreads waits for those too).
__device__ __forceinline__ void nm_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);          // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <bool F16X>
__global__ __launch_bounds__(kNmThreads, 4) void native_q4_mfma(const uint8_t *__restrict__ w,
                                                            const uint16_t *__restrict__ scales,
                                                            const void *__restrict__ x, float *__restrict__ y, int k,
                                                            int n, int batch, int columns, int chunk, int column_groups,
                                                            int tiles) {
    extern __shared__ uint4 lds4[];
    // workgroup -> (tile, column group): all groups of a tile, one after the other, on XCD tile % 8
    const int unit = blockIdx.x >> 3;
    const int tile = (unit / column_groups) * 8 + (blockIdx.x & 7), c0 = unit % column_groups * columns;
    if (tile >= tiles) return;                                 // whole workgroup: no barrier reached yet
    x = static_cast<const uint8_t *>(x) + static_cast<size_t>(c0) * k * (F16X ? 2 : 4);
    y += static_cast<size_t>(c0) * n;
    columns = min(columns, batch - c0);
    const int blocks = k >> 5;
    const int jn = 3 * columns;                                // operand columns: digit * columns + column
    uint2 *digits = reinterpret_cast<uint2 *>(lds4);           // [chunk][4][jn]
    float *block_scale = reinterpret_cast<float *>(digits + static_cast<size_t>(chunk) * 4 * jn);   // [chunk][columns]
    const int lane = threadIdx.x & (kk::kWave - 1);
    const int wid = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int g = lane >> 4, c16 = lane & 15, odd = lane & 1;

    const uint8_t *wl = w + static_cast<size_t>(tile) * blocks * 512 + 32 * (g + 8 * odd) + 4 * (c16 >> 1);
    const uint16_t *sl = scales + static_cast<size_t>(tile) * blocks * 32 + 8 * g;
    uint32_t raw[kNmDepth][2];
    uint4 sc[kNmDepth];
    auto load = [&](int s, int d) {                            // block wid + 8 s; past K: the last block
        const int blk = min(wid + kNmWaves * s, blocks - 1);
        raw[d][0] = *reinterpret_cast<const uint32_t *>(wl + static_cast<size_t>(blk) * 512);
        raw[d][1] = *reinterpret_cast<const uint32_t *>(wl + static_cast<size_t>(blk) * 512 + 128);
        sc[d] = *reinterpret_cast<const uint4 *>(sl + static_cast<size_t>(blk) * 32);
    };

    float acc[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][r] = 0.0f;
    // operand column of this lane (the spare ones repeat the last), its column and digit
    const int j0 = min(c16, jn - 1), col = j0 % columns;
    const float digit_scale = j0 < columns ? 0.0625f : j0 < 2 * columns ? 16.0f : 4096.0f;   // 256^digit / 16
    // even lanes keep rows 0, 1 of the quad and hold pairs 0, 1; odd lanes rows 2, 3 and pairs 2, 3
    const uint32_t sel0 = odd ? 0x05040100u : 0x01000504u, sel1 = odd ? 0x07060302u : 0x03020706u;

    // v_perm_b32(own, received): bytes of pairs 0 .. 3 of one row
    auto compute = [&](int lb, int d) {                        // lb: block within the chunk
        const uint32_t lo = __builtin_amdgcn_perm(raw[d][1], raw[d][0], 0x05010400u);   // rows 0 and 1, this lane's two pairs
        const uint32_t hi = __builtin_amdgcn_perm(raw[d][1], raw[d][0], 0x07030602u);   // rows 2 and 3
        const uint32_t keep = odd ? hi : lo, send = odd ? lo : hi;
        const uint32_t got = __builtin_amdgcn_update_dpp(0, send, 0xb1, 0xf, 0xf, true);
        const uint32_t row[2] = {__builtin_amdgcn_perm(keep, got, sel0), __builtin_amdgcn_perm(keep, got, sel1)};
        const long b = *reinterpret_cast<const long *>(digits + (lb * 4 + g) * jn + j0);
        const float sb = block_scale[lb * columns + col] * digit_scale;
        const uint32_t sw[4] = {sc[d].x, sc[d].y, sc[d].z, sc[d].w};
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            union { uint32_t u[2]; long v; } a;
            a.u[0] = (row[i] << 4) & 0xf0f0f0f0u;
            a.u[1] = row[i] & 0xf0f0f0f0u;
            const int4v t = __builtin_amdgcn_mfma_i32_16x16x32_i8(a.v, b, int4v{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float dw = kk::half_bits_to_float(i ? sw[r] >> 16 : sw[r] & 0xffffu);
                acc[i][r] = fmaf(static_cast<float>(t[r]), dw * sb, acc[i][r]);
            }
        }
    };

    // activations of a chunk: thread = up to kNmGroups (block, column, K group) of 8 values, the
    // K group fastest, then the column: the digits' LDS writes then cover all banks (with the
    // block before the column they hit two). Blocks past K: the last one again.
    float v[kNmGroups][8];
    int place[kNmGroups];                                      // block of the chunk << 8 | column
#pragma unroll
    for (int u = 0; u < kNmGroups; ++u) {
        const int cb = (static_cast<int>(threadIdx.x) + u * kNmThreads) >> 2;
        place[u] = (cb / columns) << 8 | cb % columns;
    }
    auto load_x = [&](int base) {
#pragma unroll
        for (int u = 0; u < kNmGroups; ++u) {
            int at_place = place[u];
            asm volatile("" : "+v"(at_place));                          // keeps what follows from being hoisted into spills
            const uint32_t at = static_cast<uint32_t>(at_place & 255) * k + min(base + (at_place >> 8), blocks - 1) * 32 + 2 * (lane & 3);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if constexpr (F16X) {
                    const uint16_t *xh = static_cast<const uint16_t *>(x) + at + 8 * q;
                    v[u][2 * q] = kk::half_bits_to_float(xh[0]);
                    v[u][2 * q + 1] = kk::half_bits_to_float(xh[1]);
                } else {
                    const float2a4 f = *reinterpret_cast<const float2a4 *>(static_cast<const float *>(x) + at + 8 * q);
                    v[u][2 * q] = f.x;
                    v[u][2 * q + 1] = f.y;
                }
            }
        }
    };
    auto convert = [&](int here) {
#pragma unroll
        for (int u = 0; u < kNmGroups; ++u) {
            if (kNmThreads * u + 64 * wid >= here * columns * 4) break;   // wave-uniform
            int at_place = place[u];
            asm volatile("" : "+v"(at_place));
            const int b = at_place & 255, lb = at_place >> 8;
            float m = 0.0f, bad = 0.0f;                        // bad: NaN once a value is not finite
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                bad = fmaf(v[u][t], 0.0f, bad);
                m = fmaxf(m, fabsf(v[u][t]));
            }
            // the four threads of a block are the lanes of one quad
            m = fmaxf(m, kk::dpp_move<0xb1>(m));
            m = fmaxf(m, kk::dpp_move<0x4e>(m));
            bad += kk::dpp_move<0xb1>(bad);
            bad += kk::dpp_move<0x4e>(bad);
            // 2^(e-1) <= m < 2^e; e >= -100 keeps 2^(22-e) finite
            const int e = max(__builtin_amdgcn_frexp_expf(m), -100);
            const float to_fixed = ldexpf(1.0f, 22 - e);
            // v * 2^(22-e) rounded, + 0x808080: its bytes are the digits + 128
            uint32_t z[8];
#pragma unroll
            for (int t = 0; t < 8; ++t)
                z[t] = (__float_as_uint(fmaf(v[u][t], to_fixed, 12582912.0f)) + (0x808080u - 0x4b400000u)) ^ 0x808080u;
            uint32_t dig[3][2];                                // [digit][even / odd K], the four pairs' bytes
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint32_t p01 = __builtin_amdgcn_perm(z[2 + h], z[h], 0x05010400u);       // z0.0 z1.0 z0.1 z1.1
                const uint32_t p23 = __builtin_amdgcn_perm(z[6 + h], z[4 + h], 0x05010400u);
                dig[0][h] = __builtin_amdgcn_perm(p23, p01, 0x05040100u);
                dig[1][h] = __builtin_amdgcn_perm(p23, p01, 0x07060302u);
                dig[2][h] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(z[6 + h], z[4 + h], 0x0c0c0602u),
                                                  __builtin_amdgcn_perm(z[2 + h], z[h], 0x0c0c0602u), 0x05040100u);
            }
            if (lb < here) {
                uint2 *dst = digits + (lb * 4 + (lane & 3)) * jn + b;
#pragma unroll
                for (int l = 0; l < 3; ++l) dst[l * columns] = make_uint2(dig[l][0], dig[l][1]);
                if ((lane & 3) == 0) block_scale[lb * columns + b] = bad != 0.0f ? __builtin_nanf("") : ldexpf(1.0f, e - 22);
            }
        }
    };

    load_x(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int d = 0; d < kNmDepth; ++d) {                       // the first weights behind the first activations,
        load(d, d);                                            // in the loop's order: the waits there count loads
        __builtin_amdgcn_sched_barrier(0);
    }
    int base = 0;
    do {                                                       // (K has blocks: no test in front for the loads to sink behind)
        const int here = min(chunk, blocks - base);
        if (base) nm_barrier();
        convert(here);
        if (base + chunk < blocks) load_x(base + chunk);   // the next chunk's, behind this one's products
        nm_barrier();
        const int s0 = base / kNmWaves;                           // chunk % kNmStep == 0: the ring index stays static
        int t = 0;
        do {
#pragma unroll
            for (int d = 0; d < kNmDepth; ++d) {
                const int lb = wid + kNmWaves * (t + d);
                if (lb < here) compute(lb, d);                 // wave-uniform
                load(s0 + t + d + kNmDepth, d);
                __builtin_amdgcn_sched_barrier(0);
            }
            t += kNmDepth;
        } while (kNmWaves * t < here);
    } while ((base += chunk) < blocks);
    nm_barrier();                                           // the digits are idle
    float *part = reinterpret_cast<float *>(lds4);             // [wave][operand column][33]
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) part[(wid * 16 + c16) * 33 + 8 * g + 2 * r + i] = acc[i][r];
    nm_barrier();
    const int row = threadIdx.x & 31, b = threadIdx.x >> 5, gr = tile * 32 + row;
    if (b < columns && gr < n) {
        float v = 0.0f;                                        // the smallest digit's sum first, the waves' in pairs
#pragma unroll
        for (int l = 0; l < 3; ++l) {
            float p[kNmWaves];
#pragma unroll
            for (int wv = 0; wv < kNmWaves; ++wv) p[wv] = part[(wv * 16 + l * columns + b) * 33 + row];
            v += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
        }
        y[static_cast<size_t>(b) * n + gr] = v;
    }
}

template <bool F16X>
hipError_t launch_mfma(const uint8_t *w, const uint16_t *scales, const void *x, float *y, int k, int n, int batch,
                       hipStream_t stream) {
    // columns in equal groups: the spare operand columns cost as much as used ones
    const int groups = (batch + kNmMaxColumns - 1) / kNmMaxColumns, columns = (batch + groups - 1) / groups;
    const int column_groups = (batch + columns - 1) / columns, tiles = (n + 31) / 32;
    const int chunk = nm_chunk(k >> 5, columns);
    const size_t lds = std::max<size_t>(static_cast<size_t>(chunk) * columns * 100, kNmPart);
    // a launch holds fewer than 2^32 threads: many columns of few rows take several
    const int tile_slots = (tiles + 7) / 8 * 8, most = static_cast<int>(0xffffffffu / kNmThreads) / tile_slots;
    for (int g0 = 0; g0 < column_groups; g0 += most) {
        const int groups_here = std::min(most, column_groups - g0);
        const size_t c0 = static_cast<size_t>(g0) * columns;
        hipLaunchKernelGGL(native_q4_mfma<F16X>, dim3(static_cast<unsigned>(tile_slots) * groups_here), dim3(kNmThreads), lds,
                           stream, w, scales, static_cast<const uint8_t *>(x) + c0 * k * (F16X ? 2 : 4), y + c0 * n, k, n,
                           batch - static_cast<int>(c0), columns, chunk, groups_here, tiles);
        const hipError_t rc = hipGetLastError();
        if (rc != hipSuccess) return rc;
    }
    return hipSuccess;
}

} // namespace

extern "C" size_t kk_native_q4_payload_bytes(int k, int n) {
    const size_t rows = (static_cast<size_t>(n) + 31) & ~static_cast<size_t>(31);
    return (rows * k / 2 + 255) & ~static_cast<size_t>(255);
}

extern "C" int kk_native_q4_gemv(const void *weights, const void *x, int x_f16, float *y, int k, int n, int batch,
                                 hipStream_t stream) {
    if (!weights || !x || !y || k <= 0 || k % 32 != 0 || k > 16384 || n <= 0 || batch <= 0)
        return hipErrorInvalidValue;
    if ((reinterpret_cast<uintptr_t>(weights) & 255) != 0) return hipErrorInvalidValue;
    if ((reinterpret_cast<uintptr_t>(x) & (x_f16 ? 1 : 3)) != 0 || (reinterpret_cast<uintptr_t>(y) & 3) != 0)
        return hipErrorInvalidValue;
    const uint8_t *w = static_cast<const uint8_t *>(weights);
    const uint16_t *scales = reinterpret_cast<const uint16_t *>(w + kk_native_q4_payload_bytes(k, n));
    const int blocks = k >> 5;
    const size_t x_bytes = x_f16 ? 2 : 4;
    // One column, and two on small matrices, stay on the dot product kernel (us per call,
    // which ends with a wait of about 15: K4096 x N4096 one column 17.1 against 19.8, two
    // 19.1 / 20.0, three 20.8 / 20.6; two columns of K4096 x N11008 26.0 / 24.9 and K11008 x
    // N4096 31.0 / 28.0).
    if (batch > 2 || (batch == 2 && static_cast<size_t>(k) * n >= (size_t{32} << 20)))
        return x_f16 ? launch_mfma<true>(w, scales, x, y, k, n, batch, stream)
                     : launch_mfma<false>(w, scales, x, y, k, n, batch, stream);
    // columns per launch: LDS within the limit and activation passes within the register budget
    auto fits = [&](int cols) {
        return lds_bytes(blocks, cols) <= kNqLdsLimit && passes_for(blocks, cols) <= kNqMaxPasses;
    };
    if (!fits(1)) return hipErrorInvalidValue;
    int fit = 1;
    while (fit < kNqMaxColumns && fits(fit + 1)) ++fit;
    for (int c0 = 0; c0 < batch; c0 += fit) {
        const int cols = std::min(fit, batch - c0);
        const int passes = passes_for(blocks, cols);
        const void *xc = static_cast<const uint8_t *>(x) + static_cast<size_t>(c0) * k * x_bytes;
        float *yc = y + static_cast<size_t>(c0) * n;
        hipError_t status;
        switch (cols) {
        case 1: status = launch_passes<1>(passes, w, scales, xc, x_f16, yc, k, n, stream); break;
        default: status = launch_passes<2>(passes, w, scales, xc, x_f16, yc, k, n, stream); break;
        }
        if (status != hipSuccess) return status;
    }
    return hipSuccess;
}
