// Common Q4 ABI v1 kernels (reference src/q4-common.inc, src/q4-activation.inc,
// src/q4-pair.inc; persistent layout src/q4-common-pack.h:16-31) on gfx950.
//
// Weight layout (layout 1 "Micro32Bank", scale order 1 "KMajor"): for output
// column c and K32 block b the 16 bytes of signed nibble pairs (K 2p low,
// 2p + 1 high) of that column's block are contiguous at
// ((c/32) * (Kp/32) + b) * 512 + (c%16) * 32 + ((c%32)/16) * 16, so one 16-byte
// load gives a lane 32 K values of one column in natural order; the FP16
// scales are [b][Np] after the weights.
//
// Activations are quantized as the reference does (reference
// kernels/kunlun-common-{max,main,residual}-exact.xpu, quant-row-serial):
//   M = 1: per tensor, two int8 components: max0 = max|x| (1 if 0),
//          q0 = rnd(x * (127/max0)), r = x - q0 * (max0/127), q1 the same on r;
//   M > 1: per row, one component q = rnd(x * (127/max_row)).
// rnd rounds half away from zero and clamps to [-127, 127]. Products with the
// weights are exact integer block sums (M = 1: v_dot4_i32_i8 on weights widened
// to 16*q; M > 1: fp16 MFMA), then y = sum_b d_b * (S0 s0 + S1 s1) in F32.
#include "device_common.h"
#include "launch.h"
#include "lds_opt_in.h"

#include <algorithm>

namespace {

constexpr int kCqWaves = 8;
constexpr int kCqThreads = 64 * kCqWaves;
constexpr int kCqDepth = 4;            // GEMV items (block pairs) in flight per wave
constexpr int kQuantThreads = 1024;    // single-workgroup per-tensor quantization
constexpr int kRowThreads = 256;       // Row A8: one workgroup per row

typedef int int32x4 __attribute__((ext_vector_type(4)));

// Max of |x| bit patterns over the workgroup (NaN above Inf, as the
// reference's integer max); every thread gets the result.
template <int Threads>
__device__ uint32_t block_max_bits(uint32_t v, uint32_t *scratch) {
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) v = max(v, static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), offset, kk::kWave)));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
    __syncthreads();
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < Threads / 64; ++i) m = max(m, scratch[i]);
    return m;
}

// One row of X (k F16 or F32 values, the type a template parameter of the
// kernels: a runtime flag would put a branch around every load, and each
// load would be waited for before the next is issued) through a buffer
// resource whose extent is the row's bytes: value j outside [0, k) reads zero
// without a memory access, so the loads need no bounds branch either.
struct XRow {
    __amdgpu_buffer_rsrc_t rsrc;
    int k;
};
template <bool F16>
__device__ __forceinline__ XRow x_row(const void *x, size_t row, int k) {
    constexpr size_t kElem = F16 ? 2 : 4;
    const uint8_t *base = static_cast<const uint8_t *>(x) + row * static_cast<size_t>(k) * kElem;
    return {__builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(base), 0, static_cast<int>(k * kElem), 0x00020000),
            k};
}
template <bool F16>
__device__ __forceinline__ float x_value(const XRow &r, int j) {
    const uint32_t jj = static_cast<uint32_t>(j) < static_cast<uint32_t>(r.k) ? static_cast<uint32_t>(j) : 0x20000000u;
    if (F16) return kk::half_bits_to_float(__builtin_amdgcn_raw_buffer_load_b16(r.rsrc, static_cast<int>(2u * jj), 0, 0));
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r.rsrc, static_cast<int>(4u * jj), 0, 0));
}

__device__ __forceinline__ uint32_t pack4(int a, int b, int c, int d) {
    return (static_cast<uint32_t>(a) & 255u) | ((static_cast<uint32_t>(b) & 255u) << 8) |
           ((static_cast<uint32_t>(c) & 255u) << 16) | (static_cast<uint32_t>(d) << 24);
}

// Two-component per-tensor quantization of the values a workgroup holds
// (v[i][t] for its groups; values past k are zero): on return v holds the
// residuals' codes' inputs replaced by the codes themselves in q0/q1, and
// s[] = {max0/127, max1/127, max0, max1}. Every thread of the workgroup calls it.
template <int Threads, int Groups>
__device__ void quantize_pair(float (&v)[Groups][8], int (&q0)[Groups][8], int (&q1)[Groups][8], float (&s)[4],
                              uint32_t *scratch) {
#pragma clang fp contract(off)
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < Groups; ++i)
#pragma unroll
        for (int t = 0; t < 8; ++t) m = max(m, __float_as_uint(v[i][t]) & 0x7fffffffu);
    m = block_max_bits<Threads>(m, scratch);
    const float max0 = m ? __uint_as_float(m) : 1.0f;
    const float s0 = max0 / 127.0f, inv0 = 127.0f / max0;
    uint32_t m1 = 0;
#pragma unroll
    for (int i = 0; i < Groups; ++i)
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const float scaled = v[i][t] * inv0;
            q0[i][t] = kk::round_clamp(scaled, 127);
            const float back = static_cast<float>(q0[i][t]) * s0;
            v[i][t] = v[i][t] - back;                       // residual
            m1 = max(m1, __float_as_uint(v[i][t]) & 0x7fffffffu);
        }
    m1 = block_max_bits<Threads>(m1, scratch);
    const float max1 = m1 ? __uint_as_float(m1) : 1.0f;
    const float s1 = max1 / 127.0f, inv1 = 127.0f / max1;
#pragma unroll
    for (int i = 0; i < Groups; ++i)
#pragma unroll
        for (int t = 0; t < 8; ++t) q1[i][t] = kk::round_clamp(v[i][t] * inv1, 127);
    s[0] = s0;
    s[1] = s1;
    s[2] = max0;
    s[3] = max1;
}

// Writes group g's codes to the view (main at (g/4)*64 + (g%4)*8, residual
// 2kp further, the group's gap bytes zero).
__device__ __forceinline__ void write_view_group(int8_t *values, int kp, int g, const int (&a)[8], const int (&b)[8]) {
    const size_t at = static_cast<size_t>(g / 4) * 64 + (g % 4) * 8;
    uint32_t *main = reinterpret_cast<uint32_t *>(values + at);
    uint32_t *resid = reinterpret_cast<uint32_t *>(values + 2 * static_cast<size_t>(kp) + at);
    main[0] = pack4(a[0], a[1], a[2], a[3]);
    main[1] = pack4(a[4], a[5], a[6], a[7]);
    main[8] = 0;                          // bytes at + 32 .. + 40: the group's gap
    main[9] = 0;
    resid[0] = pack4(b[0], b[1], b[2], b[3]);
    resid[1] = pack4(b[4], b[5], b[6], b[7]);
    resid[8] = 0;
    resid[9] = 0;
}

__device__ __forceinline__ void write_view_tail(int8_t *values, int kp, float *params, const float (&s)[4]) {
    if (threadIdx.x < 256) reinterpret_cast<uint32_t *>(values + 4 * static_cast<size_t>(kp))[threadIdx.x] = 0;
    if (threadIdx.x < 16) params[threadIdx.x] = threadIdx.x < 4 ? s[threadIdx.x] : 0.0f;
}

// ---------------------------------------------------------------------------
// M = 1: two-component per-tensor quantization into the reference's view:
// main code of K j at values[(j/32)*64 + j%32], residual at values[2kp + ...],
// the other 32 bytes of each 64-byte group and values[4kp .. 4kp+1024) zero;
// params = {max0/127, max1/127, max0, max1, 0 ...} (16 floats).
// One workgroup; thread t owns groups of 8 values g = t + 1024 i.
template <bool F16>
__global__ __launch_bounds__(kQuantThreads) void common_quant_pair(const void *__restrict__ x, int x_f16, int k,
                                                                  int kp, int8_t *__restrict__ values,
                                                                  float *__restrict__ params) {
#pragma clang fp contract(off)
    __shared__ uint32_t scratch[kQuantThreads / 64];
    constexpr int kMaxGroups = 2;              // kp <= 16384 = 2 * 1024 * 8
    const int groups = kp / 8;
    float v[kMaxGroups][8];
    const XRow xr = x_row<F16>(x, 0, k);
#pragma unroll
    for (int i = 0; i < kMaxGroups; ++i) {
        const int g = threadIdx.x + kQuantThreads * i;
#pragma unroll
        for (int t = 0; t < 8; ++t) v[i][t] = x_value<F16>(xr, g < groups ? 8 * g + t : -1);
    }
    int q0[kMaxGroups][8], q1[kMaxGroups][8];
    float sc[4];
    quantize_pair<kQuantThreads, kMaxGroups>(v, q0, q1, sc, scratch);
#pragma unroll
    for (int i = 0; i < kMaxGroups; ++i) {
        const int g = threadIdx.x + kQuantThreads * i;
        if (g < groups) write_view_group(values, kp, g, q0[i], q1[i]);
    }
    write_view_tail(values, kp, params, sc);
}

// ---------------------------------------------------------------------------
// M > 1: Row A8. Workgroup r quantizes row r of X (rows >= `rows` are the
// zero padding rows: scale 1/127, codes 0) into values[(r/128) * chunk_stride +
// (r%128) * kp ..] and writes the row scale to all 16 floats of params[r*16 ..].
// The same codes also go to `frags` as the GEMM's fp16 A operands (an int8 is
// exact in fp16): fragment (r/16, block b) is 64 lanes x 8 halves at
// ((r/16) * (kp/32) + b) * 512, lane r%16 + 16 g holding K 8g + (0, 4, 2, 6, 1, 5,
// 3, 7) of the block, the order in which a weight dword's nibbles decode.
template <bool F16>
__global__ __launch_bounds__(kRowThreads) void common_quant_rows(const void *__restrict__ x, int k, int kp, int rows,
                                                                int view_from, size_t chunk_stride,
                                                                int8_t *__restrict__ values,
                                                                float *__restrict__ params,
                                                                _Float16 *__restrict__ frags) {
#pragma clang fp contract(off)
    __shared__ uint32_t scratch[kRowThreads / 64];
    const int row = blockIdx.x;
    const bool real = row < rows;
    const XRow xr = x_row<F16>(x, real ? row : 0, real ? k : 0);   // a padding row reads zeros
    uint32_t m = 0;
    for (int j0 = 0; j0 < k; j0 += 8 * kRowThreads) {
        float v[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) v[t] = x_value<F16>(xr, j0 + t * kRowThreads + static_cast<int>(threadIdx.x));
#pragma unroll
        for (int t = 0; t < 8; ++t) m = max(m, __float_as_uint(v[t]) & 0x7fffffffu);
    }
    m = block_max_bits<kRowThreads>(m, scratch);
    const float mx = m ? __uint_as_float(m) : 1.0f;
    const float scale = mx / 127.0f, inv = 127.0f / mx;
    // eight values per thread and step: two code dwords (in the view's rows) and one lane's 16
    // fragment bytes
    const bool viewed = row >= view_from;
    const int view_row = viewed ? row - view_from : 0;
    uint2 *out = reinterpret_cast<uint2 *>(values + static_cast<size_t>(view_row >> 7) * chunk_stride +
                                           static_cast<size_t>(view_row & 127) * kp);
    kk::half8 *frag = reinterpret_cast<kk::half8 *>(frags) + static_cast<size_t>(row >> 4) * (kp >> 5) * 64 + (row & 15);
    for (int d = threadIdx.x; d < kp / 8; d += kRowThreads) {
        int q[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) q[t] = kk::round_clamp(x_value<F16>(xr, 8 * d + t) * inv, 127);
        if (viewed) out[d] = make_uint2(pack4(q[0], q[1], q[2], q[3]), pack4(q[4], q[5], q[6], q[7]));
        kk::half8 h;
        h[0] = static_cast<_Float16>(q[0]); h[1] = static_cast<_Float16>(q[4]);
        h[2] = static_cast<_Float16>(q[2]); h[3] = static_cast<_Float16>(q[6]);
        h[4] = static_cast<_Float16>(q[1]); h[5] = static_cast<_Float16>(q[5]);
        h[6] = static_cast<_Float16>(q[3]); h[7] = static_cast<_Float16>(q[7]);
        frag[(d >> 2) * 64 + 16 * (d & 3)] = h;
    }
    if (threadIdx.x < 16) params[row * 16 + threadIdx.x] = scale;
}

// ---------------------------------------------------------------------------
// M = 1 GEMV over one or two weights (the gate/up pair shares the
// activations). Workgroup = one N32 tile of one weight; its 8 waves take block
// pairs in turn. In an item (blocks 2i, 2i+1) lane l loads the 16 bytes of
// column 16 (c%2) + c/2 (c = l%32) of block 2i + l/32: the wave reads 1 KB
// contiguous. A8 (EXACT false): activation per block in LDS as 16 dwords
// [component][even K, odd K][4]; the weight dword w gives 16*q of the even K
// as (w << 4) & 0xf0f0f0f0 and of the odd K as w & 0xf0f0f0f0, so
// v_dot4_i32_i8 yields 16 * sum q x_q exactly. EXACT: the activations are
// 23-bit block fixed point digits (kk::fixed_point_digits) and v_dot8_i32_i4
// takes the weight dwords as they are (natural K order).
struct GemvMatrix {
    const uint8_t *w;
    float *y;
};

// MODE: kPrepared (act = the quantized view, params its scales), kQuantize
// (act = X: every workgroup quantizes X itself, workgroup 0 also writes the
// view to view_values / view_params), kExact (act = X).
constexpr int kPrepared = 0, kQuantize = 1, kExact = 2;

template <int MODE, bool F16>
__global__ __launch_bounds__(kCqThreads) void common_gemv(GemvMatrix m0, GemvMatrix m1, int tiles_per_matrix,
                                                         const void *__restrict__ act, int x_f16,
                                                         const float *__restrict__ params,
                                                         int8_t *__restrict__ view_values,
                                                         float *__restrict__ view_params, int k, int kp, int n,
                                                         int np) {
    constexpr bool EXACT = MODE == kExact;
    constexpr bool RAW_X = MODE != kPrepared;
    extern __shared__ uint4 lds4[];
    __shared__ uint32_t scratch[kCqWaves];
    const int which = blockIdx.x / tiles_per_matrix;
    const int tile = blockIdx.x - which * tiles_per_matrix;
    const GemvMatrix mat = which ? m1 : m0;
    const int blocks = kp >> 5;
    const int pairs = blocks >> 1;
    const uint16_t *scales = reinterpret_cast<const uint16_t *>(mat.w + static_cast<size_t>(np) * kp / 2);
    constexpr int kBlockWords = EXACT ? 24 : 16;
    uint32_t *act_lds = reinterpret_cast<uint32_t *>(lds4);                       // [blocks][kBlockWords]
    float *block_scale = reinterpret_cast<float *>(act_lds + static_cast<size_t>(blocks) * kBlockWords);  // EXACT
    float *partial = block_scale + (EXACT ? blocks : 0);                         // [waves][32]

    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int chunk = lane & 31;
    const int col = tile * 32 + 16 * (chunk & 1) + (chunk >> 1);
    const size_t tile_block0 = static_cast<size_t>(tile) * blocks;

    // 1. activation loads (before the weights: the memory counter is in order)
    constexpr int kMaxPasses = 4;              // kp / 8 <= 2048 groups = 4 x 512 threads
    const int groups = kp / 8;
    uint32_t raw[kMaxPasses][4];
    float xv[kMaxPasses][8];
    const XRow xr = x_row<F16>(act, 0, k);
#pragma unroll
    for (int pass = 0; pass < kMaxPasses; ++pass) {
        const int g = min(pass * kCqThreads + static_cast<int>(threadIdx.x), groups - 1);
        if (RAW_X) {
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                xv[pass][t] = x_value<F16>(xr, 8 * g + t);
            }
        } else {
            const int8_t *codes = static_cast<const int8_t *>(act);
            const size_t at = static_cast<size_t>(g / 4) * 64 + (g % 4) * 8;
            const uint2 a = *reinterpret_cast<const uint2 *>(codes + at);
            const uint2 b = *reinterpret_cast<const uint2 *>(codes + 2 * static_cast<size_t>(kp) + at);
            raw[pass][0] = a.x;
            raw[pass][1] = a.y;
            raw[pass][2] = b.x;
            raw[pass][3] = b.y;
        }
    }
    float s0 = 0.0f, s1 = 0.0f;
    if (MODE == kPrepared) {
        s0 = params[0] * 0.0625f;              // the weights enter as 16 * q
        s1 = params[1] * 0.0625f;
    }
    __builtin_amdgcn_sched_barrier(0);

    // 2. the first weight items
    auto load_item = [&](int s, uint32_t (&buf)[5]) {
        const int it = min(wid + kCqWaves * s, pairs - 1);
        const int blk = 2 * it + (lane >> 5);
        // 1 KB contiguous per wave, read once per call: non-temporal
        const kk::u32x4_a4 v = kk::load_u32x4_stream(
            reinterpret_cast<const uint32_t *>(mat.w + (tile_block0 + blk) * 512 + chunk * 16));
        buf[0] = v.x;
        buf[1] = v.y;
        buf[2] = v.z;
        buf[3] = v.w;
        buf[4] = scales[static_cast<size_t>(blk) * np + min(col, np - 1)];
    };
    // every wave runs the same count of items (the last ones may add zero);
    // loads are unconditional (past the end they re-read a valid item): here
    // that measures faster than skipping them with a branch
    const int iters = (pairs + kCqWaves - 1) / kCqWaves;
    const int iters_padded = (iters + kCqDepth - 1) / kCqDepth * kCqDepth;
    uint32_t ring[kCqDepth][5];
#pragma unroll
    for (int d = 0; d < kCqDepth; ++d) {
        load_item(d, ring[d]);
        __builtin_amdgcn_sched_barrier(0);
    }

    // 3. activations -> LDS
    if (MODE == kQuantize) {
        // clamped duplicate groups hold copies of the last group: no effect on the maxima
        int q0[kMaxPasses][8], q1[kMaxPasses][8];
        float sc[4];
        quantize_pair<kCqThreads, kMaxPasses>(xv, q0, q1, sc, scratch);
        s0 = sc[0] * 0.0625f;
        s1 = sc[1] * 0.0625f;
#pragma unroll
        for (int pass = 0; pass < kMaxPasses; ++pass) {
            const int g = pass * kCqThreads + static_cast<int>(threadIdx.x);
            if (g < groups) {
                raw[pass][0] = pack4(q0[pass][0], q0[pass][1], q0[pass][2], q0[pass][3]);
                raw[pass][1] = pack4(q0[pass][4], q0[pass][5], q0[pass][6], q0[pass][7]);
                raw[pass][2] = pack4(q1[pass][0], q1[pass][1], q1[pass][2], q1[pass][3]);
                raw[pass][3] = pack4(q1[pass][4], q1[pass][5], q1[pass][6], q1[pass][7]);
                if (blockIdx.x == 0) write_view_group(view_values, kp, g, q0[pass], q1[pass]);
            }
        }
        if (blockIdx.x == 0) write_view_tail(view_values, kp, view_params, sc);
    }
#pragma unroll
    for (int pass = 0; pass < kMaxPasses; ++pass) {
        const int idx = pass * kCqThreads + static_cast<int>(threadIdx.x);
        const int g = min(idx, groups - 1);
        if (EXACT) {
            float m = 0.0f, bad = 0.0f;
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const float a = fabsf(xv[pass][t]);
                bad = (a <= 3.402823466e38f) ? bad : 1.0f;
                m = fmaxf(m, a);
            }
            m = fmaxf(m, kk::dpp_move<0xb1>(m));        // the 4 groups of a block: one quad
            m = fmaxf(m, kk::dpp_move<0x4e>(m));
            bad = fmaxf(bad, kk::dpp_move<0xb1>(bad));
            bad = fmaxf(bad, kk::dpp_move<0x4e>(bad));
            const int e = max(__builtin_amdgcn_frexp_expf(m), -100);
            uint32_t dig[6];
            kk::fixed_point_digits(xv[pass], ldexpf(1.0f, 22 - e), dig);
            if (idx < groups) {
#pragma unroll
                for (int l = 0; l < 6; ++l) act_lds[(g / 4) * 24 + (g % 4) * 6 + l] = dig[l];
                if ((g & 3) == 0) block_scale[g / 4] = bad != 0.0f ? __builtin_nanf("") : ldexpf(1.0f, e - 22);
            }
        } else if (idx < groups) {
            // even K: bytes 0, 2 of each dword; odd K: bytes 1, 3
            uint32_t *dst = act_lds + (g / 4) * 16 + (g % 4);
            dst[0] = __builtin_amdgcn_perm(raw[pass][1], raw[pass][0], 0x06040200u);
            dst[4] = __builtin_amdgcn_perm(raw[pass][1], raw[pass][0], 0x07050301u);
            dst[8] = __builtin_amdgcn_perm(raw[pass][3], raw[pass][2], 0x06040200u);
            dst[12] = __builtin_amdgcn_perm(raw[pass][3], raw[pass][2], 0x07050301u);
        }
    }
    __syncthreads();

    // 4. items
    float acc = 0.0f;
    auto compute_item = [&](int s, const uint32_t (&buf)[5]) {
        const int it = wid + kCqWaves * s;
        const bool live = it < pairs && col < n;
        const int blk = 2 * min(it, pairs - 1) + (lane >> 5);
        const float d = live ? kk::half_bits_to_float(buf[4]) : 0.0f;
        if (EXACT) {
            const uint4 *src = reinterpret_cast<const uint4 *>(act_lds + static_cast<size_t>(blk) * 24);
            uint32_t dg[24];
#pragma unroll
            for (int g = 0; g < 6; ++g) {
                const uint4 v4 = src[g];
                dg[4 * g] = v4.x;
                dg[4 * g + 1] = v4.y;
                dg[4 * g + 2] = v4.z;
                dg[4 * g + 3] = v4.w;
            }
            int t[6];
#pragma unroll
            for (int l = 0; l < 6; ++l) {
                t[l] = 0;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    t[l] = __builtin_amdgcn_sdot8(static_cast<int>(buf[i]), static_cast<int>(dg[i * 6 + l]), t[l], false);
            }
            int sum = t[5];
#pragma unroll
            for (int l = 4; l >= 0; --l) sum = (sum << 4) + t[l];
            acc = fmaf(static_cast<float>(sum), live ? d * block_scale[blk] : 0.0f, acc);
        } else {
            const uint4 *src = reinterpret_cast<const uint4 *>(act_lds + static_cast<size_t>(blk) * 16);
            const uint4 e0 = src[0], o0 = src[1], e1 = src[2], o1 = src[3];
            const uint32_t a0e[4] = {e0.x, e0.y, e0.z, e0.w}, a0o[4] = {o0.x, o0.y, o0.z, o0.w};
            const uint32_t a1e[4] = {e1.x, e1.y, e1.z, e1.w}, a1o[4] = {o1.x, o1.y, o1.z, o1.w};
            int p0 = 0, p1 = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int ev = static_cast<int>((buf[i] << 4) & 0xf0f0f0f0u);
                const int od = static_cast<int>(buf[i] & 0xf0f0f0f0u);
                p0 = __builtin_amdgcn_sdot4(ev, static_cast<int>(a0e[i]), p0, false);
                p0 = __builtin_amdgcn_sdot4(od, static_cast<int>(a0o[i]), p0, false);
                p1 = __builtin_amdgcn_sdot4(ev, static_cast<int>(a1e[i]), p1, false);
                p1 = __builtin_amdgcn_sdot4(od, static_cast<int>(a1o[i]), p1, false);
            }
            const float t = fmaf(static_cast<float>(p0), s0, static_cast<float>(p1) * s1);
            acc = fmaf(d, t, acc);
        }
    };
    for (int base = 0; base < iters_padded; base += kCqDepth) {
#pragma unroll
        for (int dpt = 0; dpt < kCqDepth; ++dpt) {
            if (base + dpt < iters) compute_item(base + dpt, ring[dpt]);   // uniform; no loads inside
            load_item(base + dpt + kCqDepth, ring[dpt]);     // past the end: a valid address
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // 5. column sums: the two block halves of the wave, then the waves in order
    acc += __shfl_xor(acc, 32, kk::kWave);
    if (lane < 32) partial[wid * 32 + chunk] = acc;
    __syncthreads();
    if (threadIdx.x < 32) {
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < kCqWaves; ++w) v += partial[w * 32 + threadIdx.x];
        const int c = tile * 32 + 16 * (threadIdx.x & 1) + (threadIdx.x >> 1);
        if (c < n) mat.y[c] = v;
    }
}

// ---------------------------------------------------------------------------
// M > 1 GEMM on v_mfma_f32_16x16x32_f16, one K32 block per MFMA: int8 codes and
// 4-bit weights are exact in fp16 and a block's sum (at most 32 * 127 * 8) is
// exact in F32, so D is the block's integer sum and needs one fma per output
// with the block's FP16 scale. (v_mfma_i32_16x16x32_i8, used before, needs a
// conversion as well: twice the VALU work, which is what bounds this kernel.)
//
// A workgroup of 8 waves takes 16 RT rows x 16 CG CW columns, CW = 8 / KG: wave
// (wn, kg) sums its 16 CG columns over BPW of every stage's SB = KG BPW blocks, and
// the k-groups' sums meet in LDS at the end in a fixed order. Per stage each
// wave copies RT SB / 8 fragments (1 KB each, in operand order), 1 KB of weights
// and 128 B of scales into LDS (global_load_lds), into a ring of SLOTS stages.
//
// MFMA and VALU issue hardly overlap here (a probe of independent chains, two
// waves per SIMD: 16 MFMAs 253 cycles, 64 fmas 158, both 380): K4096 x N11008 at
// 512 rows needs 29 us of it, of the 75 that the kernel takes. The rest is what a
// stage does before its first product: the wait for its copies, the barrier and
// the operand reads (CG = 2: 85 B per cycle and CU at full MFMA rate). KG splits K
// over the waves rather than the tile, so that few rows and columns per workgroup
// still fill the CUs. kk_common_gemm has the times.
template <int RT, int CG, int KG, int BPW, int SLOTS>
struct CgShape {
    static constexpr int CW = 8 / KG;                                   // column waves
    static constexpr int Cols = 16 * CG * CW;
    static constexpr int SB = KG * BPW;                                 // blocks per stage
    static constexpr int ABytes = RT * SB * 1024;
    static constexpr int StageBytes = ABytes + 8 * 1024 + 1024;         // + weights + scales
    static constexpr int ACopies = RT * SB / 8;                         // per wave
    static constexpr int LdsBytes = SLOTS * StageBytes;
    static_assert(Cols * SB == 512 && CG % 2 == 0, "8 KB of weights per stage, whole 32-column tiles");
    static_assert(RT * SB % 8 == 0 && LdsBytes <= 160 * 1024 && ACopies <= 8, "stage");
    static constexpr int RP = RT * CG * 8 * 1024 <= LdsBytes ? RT : RT * CG * 4 * 1024 <= LdsBytes ? RT / 2 : RT / 4;
    static_assert(RP >= 1 && RP * CG * 8 * 1024 <= LdsBytes, "k-group exchange");
};

template <int RT, int CG, int KG, int BPW, int SLOTS>
__device__ __forceinline__ void cg_copy_stage(const uint8_t *w, const uint8_t *scales, const uint8_t *frags, int blocks,
                                              int np, int row_tile0, int col_tile0, int wid, int lane, int stage) {
    using S = CgShape<RT, CG, KG, BPW, SLOTS>;
    extern __shared__ __attribute__((aligned(16))) uint8_t cg_lds[];
    uint8_t *buf = cg_lds + (stage % SLOTS) * S::StageBytes;
    const int b0 = stage * S::SB;
#pragma unroll
    for (int t = 0; t < S::ACopies; ++t) {
        const int c = wid + 8 * t, i = c / S::SB, j = c % S::SB;        // row tile, block
        __builtin_amdgcn_global_load_lds(frags + (static_cast<size_t>(row_tile0 + i) * blocks + b0 + j) * 1024 + lane * 16,
                                         buf + c * 1024, 16, 0, 0);
    }
    constexpr int kPer = S::SB / 2;                                     // 1 KB weight copies per column tile
    const int ct = wid / kPer, part = wid % kPer;
    __builtin_amdgcn_global_load_lds(w + (static_cast<size_t>(col_tile0 + ct) * blocks + b0) * 512 + part * 1024 + lane * 16,
                                     buf + S::ABytes + wid * 1024, 16, 0, 0);
    // scales [block][column]: bytes 128 wid .. +127 of the stage's 1 KB
    constexpr int kRow = 2 * S::Cols;                                   // bytes per block
    if (lane < 8) {
        const int pos = wid * 128 + lane * 16, b = pos / kRow, off = pos % kRow;
        __builtin_amdgcn_global_load_lds(scales + (static_cast<size_t>(b0 + b) * np + col_tile0 * 32) * 2 + off,
                                         buf + S::ABytes + 8 * 1024 + wid * 128, 16, 0, 0);
    }
}

template <int RT, int CG, int KG, int BPW, int SLOTS>
__global__ __launch_bounds__(512, (SLOTS * (RT * KG * BPW + 9) <= 80 ? 4 : 2)) void common_gemm(const uint8_t *__restrict__ w, const uint8_t *__restrict__ frags,
                                                   const float *__restrict__ row_scales, float *__restrict__ y,
                                                   int rows, int blocks, int n, int np, int col_groups, int per_xcd,
                                                   int total) {
    using S = CgShape<RT, CG, KG, BPW, SLOTS>;
    typedef float float4v __attribute__((ext_vector_type(4)));
    extern __shared__ __attribute__((aligned(16))) uint8_t cg_lds[];
    const int idx = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;        // contiguous ranges per XCD
    if (idx >= total) return;                                           // whole workgroup, before any barrier
    const int row_groups = total / col_groups;
    const int cg = idx / row_groups, rg = idx - cg * row_groups;        // one column group's rows share its weights in L2
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int wn = wid % S::CW, kg = wid / S::CW;
    const int q = lane >> 4, c16 = lane & 15;
    const int row_tile0 = rg * RT, col_tile0 = cg * (S::Cols / 32);     // 16-row and 32-column tiles
    const int stages = blocks / S::SB;
    const uint8_t *scales = w + static_cast<size_t>(np) * blocks * 16;  // after the np * kp / 2 weight bytes

    float4v acc[RT][CG];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int h = 0; h < CG; ++h) acc[i][h] = float4v{0.0f, 0.0f, 0.0f, 0.0f};

    for (int s = 0; s < min(SLOTS - 1, stages); ++s)
        cg_copy_stage<RT, CG, KG, BPW, SLOTS>(w, scales, frags, blocks, np, row_tile0, col_tile0, wid, lane, s);
    for (int s = 0; s < stages; ++s) {
        // this wave's copies of stage s landed (with three slots those of s + 1
        // may be in flight), then every wave's; all reads of the buffer filled
        // next are done
        if (SLOTS == 3 && s + 1 < stages) __builtin_amdgcn_s_waitcnt(0x0F70 | (S::ACopies + 2));
        else __builtin_amdgcn_s_waitcnt(0x0F70);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
        if (s + SLOTS - 1 < stages)
            cg_copy_stage<RT, CG, KG, BPW, SLOTS>(w, scales, frags, blocks, np, row_tile0, col_tile0, wid, lane,
                                                  s + SLOTS - 1);
        const uint8_t *buf = cg_lds + (s % SLOTS) * S::StageBytes;
        // every operand read, then MFMA m + kAhead beside the fmas of MFMA m (left to
        // itself the compiler pairs each MFMA with its own fmas and waits for it)
        constexpr int kB = RT * CG, kM = BPW * kB, kAhead = kM < 6 ? kM : 6;
        kk::half8 b[BPW][CG], a[BPW][RT];
        float d[BPW][CG];
#pragma unroll
        for (int jj = 0; jj < BPW; ++jj) {
            const int j = BPW * kg + jj;
            // 32-column tiles of the stage: [tile][block][column % 16][column / 16][16 bytes]
            const uint8_t *wb = buf + S::ABytes + (wn * (CG / 2) * S::SB + j) * 512 + c16 * 32 + 4 * q;
            const uint16_t *sc = reinterpret_cast<const uint16_t *>(buf + S::ABytes + 8 * 1024 + j * 2 * S::Cols) +
                                 wn * 16 * CG + c16;
            uint32_t nib[CG];
#pragma unroll
            for (int h = 0; h < CG; ++h) {                              // columns 16 h + c16 of the wave
                nib[h] = *reinterpret_cast<const uint32_t *>(wb + (h / 2) * S::SB * 512 + 16 * (h % 2));
                d[jj][h] = kk::half_bits_to_float(sc[16 * h]);
                asm("" : "+v"(d[jj][h]));                               // a plain F32 fma below: v_fma_mix issues at half its rate
            }
#pragma unroll
            for (int i = 0; i < RT; ++i) a[jj][i] = reinterpret_cast<const kk::half8 *>(buf)[(j + i * S::SB) * 64 + lane];
            // signed nibble + 8 is the nibble with its top bit flipped
#pragma unroll
            for (int h = 0; h < CG; ++h) b[jj][h] = kk::q4_dword_halves(nib[h] ^ 0x88888888u);
        }
        __builtin_amdgcn_sched_barrier(0);
        float4v p[kM];
#pragma unroll
        for (int m = 0; m < kM + kAhead; ++m) {
            if (m < kM) {
                const float4v zero = {0.0f, 0.0f, 0.0f, 0.0f};
                p[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[m / kB][m % kB / CG], b[m / kB][m % CG], zero, 0, 0, 0);
            }
            if (m >= kAhead) {
                const int o = m - kAhead, i = o % kB / CG, h = o % CG;
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[i][h][r] = fmaf(p[o][r], d[o / kB][h], acc[i][h][r]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // the k-groups' sums meet in LDS, RP row tiles at a time; every wave adds
    // (in k-group order) and stores its share of the 16 x 16 tiles
    constexpr int kTiles = S::CW * S::RP * CG;                          // per pass
    float4v *xfer = reinterpret_cast<float4v *>(cg_lds);
#pragma unroll
    for (int i0 = 0; i0 < RT; i0 += S::RP) {
        __syncthreads();                                                // the ring, or the pass before, is read
#pragma unroll
        for (int i = 0; i < S::RP; ++i)
#pragma unroll
            for (int h = 0; h < CG; ++h) xfer[((kg * S::CW + wn) * S::RP * CG + i * CG + h) * 64 + lane] = acc[i0 + i][h];
        __syncthreads();
        for (int t = wid; t < kTiles; t += 8) {
            float4v v = xfer[t * 64 + lane];
#pragma unroll
            for (int o = 1; o < KG; ++o) v += xfer[(o * kTiles + t) * 64 + lane];
            const int tn = t / (S::RP * CG), i = t / CG % S::RP, h = t % CG;
            const int col = col_tile0 * 32 + (tn * CG + h) * 16 + c16;
            const int row0 = (row_tile0 + i0 + i) * 16 + 4 * q;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (row0 + r < rows && col < n) y[static_cast<size_t>(row0 + r) * n + col] = v[r] * row_scales[(row0 + r) * 16];
        }
    }
}

struct CgArgs {
    const uint8_t *w, *frags;
    const float *row_scales;
    float *y;
    int rows, blocks, n, np;
};

template <int RT, int CG, int KG, int BPW, int SLOTS>
hipError_t launch_common_gemm(const CgArgs &a, hipStream_t stream) {
    using S = CgShape<RT, CG, KG, BPW, SLOTS>;
    const hipError_t rc = kk::opt_in_lds(reinterpret_cast<const void *>(&common_gemm<RT, CG, KG, BPW, SLOTS>), S::LdsBytes);
    if (rc != hipSuccess) return rc;
    const int col_groups = (a.n + S::Cols - 1) / S::Cols;
    const int total = col_groups * ((a.rows + 16 * RT - 1) / (16 * RT));
    const int per_xcd = (total + 7) / 8;
    hipLaunchKernelGGL((common_gemm<RT, CG, KG, BPW, SLOTS>), dim3(per_xcd * 8), dim3(512), S::LdsBytes, stream, a.w, a.frags,
                       a.row_scales, a.y, a.rows, a.blocks, a.n, a.np, col_groups, per_xcd, total);
    return hipGetLastError();
}

} // namespace

extern "C" int kk_common_quant_pair(const void *x, int x_f16, int k, int kp, void *values, void *params,
                                    hipStream_t stream) {
    if (!x || !values || !params || k <= 0 || kp < k || kp % 256 != 0 || kp > 16384) return hipErrorInvalidValue;
    if (x_f16)
        hipLaunchKernelGGL(common_quant_pair<true>, dim3(1), dim3(kQuantThreads), 0, stream, x, x_f16, k, kp,
                           static_cast<int8_t *>(values), static_cast<float *>(params));
    else
        hipLaunchKernelGGL(common_quant_pair<false>, dim3(1), dim3(kQuantThreads), 0, stream, x, x_f16, k, kp,
                           static_cast<int8_t *>(values), static_cast<float *>(params));
    return hipGetLastError();
}

extern "C" int kk_common_quant_rows(const void *x, int x_f16, int k, int kp, int rows, int defined_rows,
                                    int view_from, size_t chunk_stride, void *values, void *params, void *frags,
                                    hipStream_t stream) {
    if (!x || !values || !params || !frags || k <= 0 || kp < k || kp % 256 != 0 || rows <= 0 ||
        defined_rows < rows || defined_rows % 32 != 0 || view_from < 0 || view_from >= rows ||
        (reinterpret_cast<uintptr_t>(values) & 7) || (chunk_stride & 7) || (reinterpret_cast<uintptr_t>(frags) & 15))
        return hipErrorInvalidValue;
    if (x_f16)
        hipLaunchKernelGGL(common_quant_rows<true>, dim3(defined_rows), dim3(kRowThreads), 0, stream, x, k, kp, rows,
                           view_from, chunk_stride, static_cast<int8_t *>(values), static_cast<float *>(params),
                           static_cast<_Float16 *>(frags));
    else
        hipLaunchKernelGGL(common_quant_rows<false>, dim3(defined_rows), dim3(kRowThreads), 0, stream, x, k, kp, rows,
                           view_from, chunk_stride, static_cast<int8_t *>(values), static_cast<float *>(params),
                           static_cast<_Float16 *>(frags));
    return hipGetLastError();
}

extern "C" size_t kk_common_gemv_lds_bytes(int kp, int exact) {
    const size_t blocks = static_cast<size_t>(kp) / 32;
    return blocks * (exact ? 24 * 4 + 4 : 16 * 4) + static_cast<size_t>(kCqWaves) * 32 * 4;
}

extern "C" int kk_common_gemv(const void *w0, float *y0, const void *w1, float *y1, const void *act, int mode,
                              int x_f16, void *params, void *view_values, int k, int kp, int n, int np,
                              hipStream_t stream) {
    if (!w0 || !y0 || !act || mode < 0 || mode > 2 || (mode != kExact && !params) ||
        (mode == kQuantize && !view_values) || kp % 256 != 0 || kp > 16384 || np % 256 != 0 || n > np || k > kp ||
        (reinterpret_cast<uintptr_t>(w0) & 255) != 0 || (w1 && (reinterpret_cast<uintptr_t>(w1) & 255)))
        return hipErrorInvalidValue;
    const int tiles = (n + 31) / 32;
    const int count = w1 ? 2 : 1;
    const size_t lds = kk_common_gemv_lds_bytes(kp, mode == kExact);
    const GemvMatrix m0{static_cast<const uint8_t *>(w0), y0};
    const GemvMatrix m1{static_cast<const uint8_t *>(w1 ? w1 : w0), w1 ? y1 : y0};
    const dim3 grid(tiles * count), block(kCqThreads);
    int8_t *vv = static_cast<int8_t *>(view_values);
    float *pp = static_cast<float *>(params);
#define KK_COMMON_GEMV(M, F)                                                                                \
    hipLaunchKernelGGL((common_gemv<M, F>), grid, block, lds, stream, m0, m1, tiles, act, x_f16, pp, vv, pp, k, kp, n, \
                       np)
    if (mode == kExact) {
        if (x_f16) KK_COMMON_GEMV(kExact, true); else KK_COMMON_GEMV(kExact, false);
    } else if (mode == kQuantize) {
        if (x_f16) KK_COMMON_GEMV(kQuantize, true); else KK_COMMON_GEMV(kQuantize, false);
    } else {
        if (x_f16) KK_COMMON_GEMV(kPrepared, true); else KK_COMMON_GEMV(kPrepared, false);
    }
#undef KK_COMMON_GEMV
    return hipGetLastError();
}

// Tiles, and their times per workgroup and K block fitted to the sweep below (us;
// with one resident per CU, and with two where LDS allows). Measured, K4096 x
// N11008 at 32 / 128 / 512 / 1024 rows: 128 x 64 tile 30 / 32 / 94 / 187 us, 64 x
// 128 34 / 35 / 75 / 140, 32 x 64 13 / 29 / 90 / 201, 32 x 32 17 / 48 / 174 / 385;
// K4096 x N4096 29 / 31 / 34 / 64, 34 / 34 / 35 / 52, 13 / 14 / 36 / 78, 9 / 18 /
// 64 / 151. (Before: chunks of 128 rows on the int8 MFMA, 36 us each at N11008.)
extern "C" int kk_common_gemm(const void *w, const void *frags, const void *row_scales, float *y, int rows, int kp, int n,
                              int np, int cus, hipStream_t stream) {
    if (!w || !frags || !row_scales || !y || rows <= 0 || kp <= 0 || kp % 256 != 0 || np % 256 != 0 || n > np ||
        cus <= 0 || (reinterpret_cast<uintptr_t>(w) & 255) != 0 || (reinterpret_cast<uintptr_t>(frags) & 15) != 0)
        return hipErrorInvalidValue;
    const CgArgs a = {static_cast<const uint8_t *>(w), static_cast<const uint8_t *>(frags),
                      static_cast<const float *>(row_scales), y, rows, kp / 32, n, np};
    static const struct { int rows, cols, stage; double one, two; } kAll[] = {
        {128, 64, 8, 0.235, 0.0}, {64, 128, 4, 0.255, 0.39}, {32, 64, 8, 0.095, 0.145}, {32, 32, 16, 0.062, 0.0}};
    int pick = 0;
    double best = 0.0;
    for (int i = 0; i < 4; ++i) {
        if (a.blocks % kAll[i].stage != 0) continue;
        const long wgs = static_cast<long>((n + kAll[i].cols - 1) / kAll[i].cols) * ((rows + kAll[i].rows - 1) / kAll[i].rows);
        const double cost = wgs <= cus             ? kAll[i].one
                            : kAll[i].two == 0.0 ? kAll[i].one * static_cast<double>((wgs + cus - 1) / cus)
                                                 : kAll[i].two * std::max(1.0, static_cast<double>(wgs) / (2 * cus));
        if (best == 0.0 || cost < best) {
            best = cost;
            pick = i;
        }
    }
    switch (pick) {
    case 0: return launch_common_gemm<8, 4, 8, 1, 2>(a, stream);
    case 1: return launch_common_gemm<4, 2, 2, 2, 3>(a, stream);
    case 2: return launch_common_gemm<2, 2, 4, 2, 3>(a, stream);
    default: return launch_common_gemm<2, 2, 8, 2, 3>(a, stream);
    }
}
