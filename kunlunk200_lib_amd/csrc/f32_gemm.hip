// F32 weights at more than 16 columns, one pass over the weights per 64 columns,
// on fp32 MFMA (v_mfma_f32_16x16x4_f32): exact F32 products and F32 sums, the
// numerics of dense_mfma_gemv.
//
// A workgroup of 8 waves owns 16 weight rows x 16 MT columns: wave (kg, ch) sums
// the K32 slice kg of every 128-K stage for column half ch, and the four
// k-groups' sums meet in LDS at the end in order. Per stage the waves copy
// the 16 weight rows and the X rows (512 B each) into LDS
// (buffer_load_dwordx4 ... lds), all but one slot of the ring ahead. Chunk c
// (16 B) of row r sits at position c ^ (r & 15), so the 16 rows of an operand
// read hit 16 distinct bank quads; lane (n, g) reads K 8g .. 8g + 7 of its row.
//
// 16 rows per workgroup, for 256 workgroups at N4096. K4096 x N4096 at 64 columns
// has 14.5 us of fp32 MFMA and 13 us of weight reads; the kernel takes 27.5 us (51
// in passes of 16 columns), 1900 cycles per stage for 1024 of MFMA on each SIMD:
// the waves of a SIMD read their operands together after each barrier. Where
// there are more workgroups than CUs, two per CU with half the ring each overlap
// that: 128 / 256 columns 53.8 / 102.8 -> 42.9 / 84.8 us (105 / 208 in passes of 16);
// with one workgroup per CU the deep ring is faster (K11008 x N4096 at 64: 68
// against 79).
#include "device_common.h"
#include "launch.h"
#include "lds_opt_in.h"

#include <algorithm>

namespace {

using kk::kWave;

typedef float float4v __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kDgStageK = 128;
constexpr int kDgRow = kDgStageK * 4;             // bytes of a row per stage
constexpr int kDgWaves = 8, kDgThreads = kDgWaves * kWave;
constexpr int kDgGroups = 4;                     // k-groups, one K32 slice of a stage each

template <int MT, bool SHARE>
struct DgShape {
    static_assert(MT == 2 || MT == 4, "32 or 64 columns");
    static constexpr int Cols = 16 * MT;
    static constexpr int WBytes = 16 * kDgRow, XBytes = Cols * kDgRow;
    static constexpr int StageBytes = WBytes + XBytes;
    static constexpr int XCopies = XBytes / 1024 / kDgWaves;             // per wave: 2 or 4
    static_assert(WBytes == 1024 * kDgWaves, "one weight copy per wave");
    // SHARE: two workgroups per CU
    static constexpr int Slots = std::min(6, (SHARE ? 80 : 160) * 1024 / StageBytes);   // 3, 2; 6, 4
    static constexpr int LdsBytes = Slots * StageBytes;
    static_assert(Slots >= 2 && (Slots - 2) * (XCopies + 1) <= 63, "ring");
};

template <int N>
__device__ __forceinline__ void dg_wait() {
    static_assert(N >= 0 && N <= 63, "vmcnt");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0F70);
}

// One stage's copies of wave `wid` (a separate function: the host pass rejects
// a kernel-local lambda that hands captured values to these builtins).
template <int MT, bool SHARE>
__device__ __forceinline__ void dg_copy(const uint8_t *w, int w_bytes, const float *x, int x_bytes, uint32_t w_off,
                                        const uint32_t (&x_off)[DgShape<MT, SHARE>::XCopies], int wid, int s) {
    using D = DgShape<MT, SHARE>;
    extern __shared__ __align__(16) uint8_t dg_lds[];
    // the stage's offset moves the base and the extent, so that a lane past the matrix (a
    // last stage that K does not fill) is past the extent by its own offset
    const int at = s * kDgRow;
    const __amdgpu_buffer_rsrc_t w_rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(w) + at, 0, w_bytes - at, 0x00020000);
    const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(reinterpret_cast<const uint8_t *>(x)) + at, 0, x_bytes - at, 0x00020000);
    __attribute__((address_space(3))) uint8_t *buf =
        (__attribute__((address_space(3))) uint8_t *)dg_lds + (s % D::Slots) * D::StageBytes;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(w_rsrc, buf + wid * 1024, 16, w_off, 0, 0, 2);   // read once
#pragma unroll
    for (int t = 0; t < D::XCopies; ++t)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(x_rsrc, buf + D::WBytes + (wid + kDgWaves * t) * 1024, 16, x_off[t],
                                                 0, 0, 0);
}

template <int MT, bool SHARE>
__global__ __launch_bounds__(kDgThreads) void f32_gemm(const uint8_t *__restrict__ w, const float *__restrict__ x,
                                                         float *__restrict__ y, int k, int n, int batch, int chunks,
                                                         int total, int per_xcd) {
    using D = DgShape<MT, SHARE>;
    extern __shared__ __align__(16) uint8_t dg_lds[];
    const int idx = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;    // a tile's column chunks share an XCD's L2
    if (idx >= total) return;                                       // whole workgroup, before any barrier
    const int tile = idx / chunks, m0 = (idx - tile * chunks) * D::Cols;
    const int n0 = tile * 16;
    const int lane = threadIdx.x & (kWave - 1);
    const int wid = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int kg = wid & 3, ch = wid >> 2;
    const int c16 = lane & 15, g = lane >> 4;
    const int stages = (k + kDgStageK - 1) / kDgStageK;
    const uint32_t w_row_bytes = static_cast<uint32_t>(k) * 4u;
    const int w_bytes = n * static_cast<int>(w_row_bytes), x_bytes = batch * k * 4;

    // copy sources: rows past the matrix repeat its last row (never stored)
    const int wr = 2 * wid + lane / 32;
    const uint32_t w_off = static_cast<uint32_t>(min(n0 + wr, n - 1)) * w_row_bytes + 16u * ((lane % 32) ^ wr);
    uint32_t x_off[D::XCopies];
#pragma unroll
    for (int t = 0; t < D::XCopies; ++t) {
        const int r = 2 * (wid + kDgWaves * t) + lane / 32;
        x_off[t] = static_cast<uint32_t>(min(m0 + r, batch - 1)) * static_cast<uint32_t>(k) * 4u + 16u * ((lane % 32) ^ (r & 15));
    }

    float4v acc[MT / 2][2], tot[MT / 2];
#pragma unroll
    for (int i = 0; i < MT / 2; ++i) tot[i] = acc[i][0] = acc[i][1] = float4v{0.0f, 0.0f, 0.0f, 0.0f};

    for (int s = 0; s < min(D::Slots - 1, stages); ++s) dg_copy<MT, SHARE>(w, w_bytes, x, x_bytes, w_off, x_off, wid, s);
    for (int s = 0; s < stages; ++s) {
        // copies of stages s + 1 .. s + Slots - 2 may be in flight (near the end: none)
        if (s + D::Slots - 2 >= stages) dg_wait<0>();
        else dg_wait<(D::Slots - 2) * (D::XCopies + 1)>();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();                               // every wave's copies landed; the slot refilled next is read
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
        if (s + D::Slots - 1 < stages) dg_copy<MT, SHARE>(w, w_bytes, x, x_bytes, w_off, x_off, wid, s + D::Slots - 1);
        if (s * kDgStageK + 32 * kg >= k) continue;                 // a slice past K (wave-uniform)
        const uint8_t *buf = dg_lds + (s % D::Slots) * D::StageBytes;
        float b[8];
        const float4v lo = *reinterpret_cast<const float4v *>(buf + c16 * kDgRow + 16 * ((8 * kg + 2 * g) ^ c16));
        const float4v hi = *reinterpret_cast<const float4v *>(buf + c16 * kDgRow + 16 * ((8 * kg + 2 * g + 1) ^ c16));
#pragma unroll
        for (int t = 0; t < 4; ++t) { b[t] = lo[t]; b[4 + t] = hi[t]; }
        float4v a[MT / 2][2];
#pragma unroll
        for (int i = 0; i < MT / 2; ++i) {
            const uint8_t *xr = buf + D::WBytes + (16 * (ch * (MT / 2) + i) + c16) * kDgRow;
            a[i][0] = *reinterpret_cast<const float4v *>(xr + 16 * ((8 * kg + 2 * g) ^ c16));
            a[i][1] = *reinterpret_cast<const float4v *>(xr + 16 * ((8 * kg + 2 * g + 1) ^ c16));
        }
#pragma unroll
        for (int t = 0; t < 8; ++t)
#pragma unroll
            for (int i = 0; i < MT / 2; ++i)
                acc[i][t & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][t >> 2][t & 3], b[t], acc[i][t & 1], 0, 0, 0);
        // sums of 8 stages join the totals: chains as short as the K-split kernel's
        if ((s & 7) == 7) {
#pragma unroll
            for (int i = 0; i < MT / 2; ++i) {
                tot[i] += acc[i][0] + acc[i][1];
                acc[i][0] = acc[i][1] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
            }
        }
    }

    __syncthreads();                                                // the ring is idle
    float4v *xfer = reinterpret_cast<float4v *>(dg_lds);
#pragma unroll
    for (int i = 0; i < MT / 2; ++i) xfer[(kg * MT + ch * (MT / 2) + i) * kWave + lane] = tot[i] + (acc[i][0] + acc[i][1]);
    __syncthreads();
    // wave t adds and stores column tile t: D reg r of lane (n, g) is column 4g + r, row n
    if (wid >= MT) return;
    float4v sum = xfer[wid * kWave + lane];
#pragma unroll
    for (int h = 1; h < kDgGroups; ++h) sum += xfer[(h * MT + wid) * kWave + lane];
    if (n0 + c16 >= n) return;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int m = m0 + 16 * wid + 4 * g + r;
        if (m < batch) y[static_cast<size_t>(m) * n + n0 + c16] = sum[r];
    }
}

template <int MT, bool SHARE>
hipError_t launch_f32_gemm(const uint8_t *w, const float *x, float *y, int k, int n, int batch, hipStream_t stream) {
    using D = DgShape<MT, SHARE>;
    const hipError_t rc = kk::opt_in_lds(reinterpret_cast<const void *>(&f32_gemm<MT, SHARE>), D::LdsBytes);
    if (rc != hipSuccess) return rc;
    const int chunks = (batch + D::Cols - 1) / D::Cols;
    const int total = (n + 15) / 16 * chunks, per_xcd = (total + 7) / 8;
    hipLaunchKernelGGL((f32_gemm<MT, SHARE>), dim3(per_xcd * 8), dim3(kDgThreads), D::LdsBytes, stream, w, x, y, k, n,
                       batch, chunks, total, per_xcd);
    return hipGetLastError();
}

} // namespace

extern "C" int kk_f32_gemm(const void *w, const float *x, float *y, int k, int n, int batch, int cus,
                           hipStream_t stream) {
    const uintptr_t bits = reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(x);
    if (!w || !x || !y || k <= 0 || (k & 31) || n <= 0 || batch < 1 || (bits & 15) ||
        static_cast<size_t>(n) * k * 4 > 0x7fffffffu || static_cast<size_t>(batch) * k * 4 > 0x7fffffffu)
        return hipErrorInvalidValue;
    const uint8_t *wb = static_cast<const uint8_t *>(w);
    const bool share = static_cast<long>((n + 15) / 16) * ((batch + 63) / 64) > cus;
    if (batch <= 32)
        return share ? launch_f32_gemm<2, true>(wb, x, y, k, n, batch, stream)
                     : launch_f32_gemm<2, false>(wb, x, y, k, n, batch, stream);
    return share ? launch_f32_gemm<4, true>(wb, x, y, k, n, batch, stream)
                 : launch_f32_gemm<4, false>(wb, x, y, k, n, batch, stream);
}
