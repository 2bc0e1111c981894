// Q4_0 GEMV for 3..32 activation columns in one pass over the weights, on
// gfx950 fp16 MFMA, with K split over workgroups.
//
// Y[b, r] = sum_k X[b, k] * W[r, k] (reference kernels/kunlun-matvec.xpu:24-79).
//
// Products: per 32-value block the exact fp16 q - 8 (B) times
// the activations as fp16 hi + lo of x * 2^s (A, about 22 bits), block sums in
// F32, scaled by the block's F16 scale in F32.
//
// Work split. A workgroup (16 waves) owns one of S ranges of K and a run of
// 16-row weight tiles; wave (wt, kg) sums tiles wt, wt + 16 / KG, ... over k-group
// kg's part of the range. The range's activations are converted into MFMA A
// fragments in LDS by the workgroup itself (no prepass launch), in chunks of
// at most 128 KiB. With S > 1 the F32 sums go to a workspace
// [range][matrix][column][row], and q4_split_sum adds the ranges in order (and
// applies SiLU * up); one range stores y directly. A range of one chunk keeps
// its fragments for any number of tiles; one of several chunks keeps one
// tile's sums per wave over them.
//
// Weights stream straight into registers: a step is 8 blocks (144 bytes) of
// 16 rows, lane (row, g) loading the 36 bytes of block pair g (x4 + x4 + x1:
// 144 contiguous bytes per row and step). MFMA wants nibble dword g of one
// block in lane (row, g), so the four lanes of a row transpose their dwords
// with v_permlane32_swap / v_permlane16_swap (one swap per fragment), and the
// scales are gathered the same way. One step is in flight per wave; two, three
// and four measured slower (K4096 x N4096, 16 columns: 10.6, 10.8, 11.7, 12.8 us).
//
// What bounds it: latency, not bandwidth. K4096 x N11008 at 32 columns takes
// 20 us; without the conversion and the products the same kernel takes 16
// (launch, X, weights, partial sums and the summing launch in turn), against
// 5.4 us for reading its 25 MB. Against the kernels before (64 rows per
// workgroup over all of K, activations from a prepass, 16 columns per pass),
// us per call: K11008 x N4096 at 8 / 16 / 32 columns 37.8 / 38.0 / 75.6 -> 13.0 /
// 14.6 / 19.5; K4096 x N11008 at 16 / 32 15.7 / 30.9 -> 14.5 / 20.6; K4096 x
// N4096 14.6 / 28.6 -> 10.3 / 13.9; pair K4096 x 2 x N11008 27.5 / 54.4 ->
// 23.2 / 33.
//
// Scales. Each (column, 256-value step) has its own power of two with
// max |x * 2^s| < 2^14; a step's sums are multiplied by 2^-s and added to the
// wave's totals. A step holding Inf or NaN makes its column NaN; for the shapes the
// batch-1 kernels leave to F32 arithmetic (K % 64 != 0, weights off a dword) an Inf
// is multiplied as one instead: +-Inf, NaN where its weight is zero or infinities cancel.
#include "device_common.h"
#include "launch.h"
#include "lds_opt_in.h"
#include <kunlun/k200_c.h>

#include <algorithm>

namespace {

using kk::half8;
using kk::kWave;

typedef float float4v __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kStepBlocks = 8;                       // blocks per step
constexpr int kStepK = 32 * kStepBlocks;
constexpr int kStepBytes = 18 * kStepBlocks;         // 144
constexpr int kFragBytes = kWave * 16;               // one A fragment: 1 KiB
constexpr int kXcds = 8;

// MT 16-column tiles (PACK: at most 8 columns, hi parts in A rows 0..7 and lo
// parts in rows 8..15 of one fragment). 16 waves of at most 128 VGPRs: two row
// tiles per wave on 8 waves (half the fragment reads) and 48- and 64-column
// forms were slower (K4096 x N11008: 32 columns 22.9 against 18.3 us, 64
// columns 46 us against two calls of 32).
constexpr int kQsWaves = 16;
constexpr int kQsThreads = kQsWaves * kWave;

template <int MT, bool PACK>
struct QsShape {
    static_assert(MT == 1 || (MT == 2 && !PACK), "up to 32 columns");
    static constexpr int Frags = PACK ? 1 : 2 * MT;                      // per block
    static constexpr int StepBytes = kStepBlocks * Frags * kFragBytes;   // A fragments of one step
    static constexpr int Cols = PACK ? 8 : 16 * MT;
    static constexpr int ChunkSteps = 128 * 1024 / StepBytes;            // 16 (PACK), 8, 4
    // conversion: a wave's item is one column and two steps (512 values)
    static constexpr int Items = (Cols * (ChunkSteps / 2) + kQsWaves - 1) / kQsWaves;
    static constexpr int InvBytes = ChunkSteps * Cols * 4;
    static constexpr int RingBytes = ChunkSteps * StepBytes + InvBytes;
    static constexpr int XferBytes = (kQsWaves - 1) * MT * kWave * 16;   // k-group sums
    static constexpr int LdsBytes = RingBytes + XferBytes;
    static_assert(ChunkSteps % 2 == 0 && Items <= 8 && LdsBytes <= 160 * 1024, "LDS chunk");
};

template <int Ctrl>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), Ctrl, 0xf, 0xf, false));
}

// Transposes dwords across the four 16-lane groups: v[i] of group g -> v[g] of
// group i.
__device__ __forceinline__ void swap32(uint32_t &a, uint32_t &b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
__device__ __forceinline__ void swap16(uint32_t &a, uint32_t &b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
__device__ __forceinline__ void transpose4(uint32_t (&v)[4]) {
    swap32(v[0], v[2]);
    swap32(v[1], v[3]);
    swap16(v[0], v[1]);
    swap16(v[2], v[3]);
}
// v[i] = group i's value, in every lane of its row
__device__ __forceinline__ void gather4(uint32_t own, uint32_t (&v)[4]) {
    uint32_t a = own, b = own;
    swap32(a, b);            // a: groups 0 1 0 1, b: groups 2 3 2 3
    v[0] = a;
    v[1] = a;
    swap16(v[0], v[1]);
    v[2] = b;
    v[3] = b;
    swap16(v[2], v[3]);
}

// The 36 bytes of one block pair (GEN: 40, from the dword its bytes start in).
template <bool GEN>
struct QsRaw {
    uint32_t d[GEN ? 10 : 9];
};

// The step's offset soff moves GEN's base and extent: its lanes past the matrix (a last step
// that K does not fill) are past the extent by their own offset. The others read inside a row.
template <bool GEN>
__device__ __forceinline__ QsRaw<GEN> qs_load(const uint8_t *base, uint32_t extent, uint32_t off, int soff) {
    QsRaw<GEN> r;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(base) + (GEN ? soff : 0), 0, static_cast<int>(GEN ? extent - soff : extent), 0x00020000);
    if constexpr (GEN) {
#pragma unroll
        for (int i = 0; i < 10; ++i) r.d[i] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, off + 4 * i, 0, 0);
    } else {
        const u32x4 a = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, soff, 0);
        const u32x4 b = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off + 16, soff, 0);
        r.d[8] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, off + 32, soff, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            r.d[i] = a[i];
            r.d[4 + i] = b[i];
        }
    }
    return r;
}

struct QsArgs {
    const uint8_t *w, *w2;      // weight matrices (w2: the up matrix of a pair, else null)
    const float *x;
    float *out;                 // y (one range) or the partial sums
    int k, n, batch;
    int steps;                  // K in steps, the last one partial when K % 256 != 0
    int ranges, kgroups;        // S, KG
    int tiles;                  // 16-row tiles of one matrix
    int per_group, groups;      // tiles of a workgroup, workgroups per range
    int per_xcd, total;         // workgroups
    int at_once;                // SERIAL: ranges at a time
    int row_stride;             // row stride of `out` (n, or the padded rows of a partial)
    uint32_t inf_bits;          // GEN: magnitude that is multiplied as infinity (above every value's: none)
};

// One column's 512 values (two steps; lane: block lane / 4, block positions
// 8 (lane % 4) ..) into the chunk's A fragments and inverse scales.
template <int MT, bool PACK, bool GEN>
__device__ __forceinline__ void qs_convert(const float (&v)[8], int item, int lane, uint32_t inf_bits, _Float16 *frag,
                                           float *inv_lds) {
    using Q = QsShape<MT, PACK>;
    const int col = item % Q::Cols, pr = item / Q::Cols;
    // the largest magnitude of each 32-lane half (one step) as bits: a NaN's
    // or Inf's are above every finite value's (inf_bits: an Inf beside finite values does not count)
    uint32_t mb = 0u;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const uint32_t bits = __float_as_uint(v[t]) & 0x7fffffffu;
        mb = max(mb, GEN && bits == inf_bits ? 0u : bits);
    }
    mb = max(mb, dpp_u32<0xb1>(mb));
    mb = max(mb, dpp_u32<0x4e>(mb));
    mb = max(mb, dpp_u32<0x141>(mb));
    mb = max(mb, dpp_u32<0x140>(mb));
    uint32_t other = mb;
    swap16(mb, other);                                          // rows 0 1 and 2 3
    mb = max(mb, other);
    int e = __builtin_amdgcn_frexp_expf(__uint_as_float(mb));
    e = mb < 0x7f800000u && mb != 0u ? max(e, -100) : 14;   // at most 128: 2^(14-e) and 2^(e-14) stay normal
    const float s = ldexpf(1.0f, 14 - e);
    const int step = 2 * pr + (lane >> 5);
    if ((lane & 31) == 0 && step < Q::ChunkSteps) inv_lds[step * Q::Cols + col] = ldexpf(1.0f, e - 14);
    half8 hi, lo;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const float a = v[t] * s;
        hi[t] = static_cast<_Float16>(a);
        lo[t] = static_cast<_Float16>(GEN && (__float_as_uint(v[t]) & 0x7fffffffu) == inf_bits
                                          ? 0.0f : a - static_cast<float>(hi[t]));   // Inf - Inf: NaN, the column's
    }
    const int blk = 2 * pr * kStepBlocks + (lane >> 2);
    const int alane = (lane & 3) * 16 + (col & 15);             // A row col % 16, positions 8 (lane % 4) ..
    if constexpr (PACK) {
        half8 *dst = reinterpret_cast<half8 *>(frag) + blk * kWave + alane;
        dst[0] = hi;
        dst[8] = lo;
    } else {
        half8 *dst = reinterpret_cast<half8 *>(frag) + (blk * Q::Frags + 2 * (col >> 4)) * kWave + alane;
        dst[0] = hi;
        dst[kWave] = lo;
    }
}

// One step of one tile: tot += 2^-s * (the step's products). a: the step's
// fragments at this lane, inv: the step's inverse scales. `next` loads the next
// step into raw: behind the products, once this step's bytes are in operand order
// (after them the products do not cover its latency: K4096 x N14336 at 16 columns 16.4
// against 16.9 us, N11008 14.6 / 15.6); with two column tiles, whose registers are full,
// after them (K4096 x N4096 at 32 columns 13.8 against 14.1).
template <int MT, bool PACK, bool GEN, typename Next>
__device__ __forceinline__ void qs_step(QsRaw<GEN> &raw, Next next, uint32_t shift, int step, int blocks, int g,
                                        const half8 *a, const float *inv, float4v (&tot)[MT]) {
    using Q = QsShape<MT, PACK>;
    uint32_t d[9], ev[4], od[4], sc[4];
#pragma unroll
    for (int i = 0; i < 9; ++i) d[i] = GEN ? kk::align_bytes(raw.d[GEN ? i + 1 : i], raw.d[i], shift) : raw.d[i];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        ev[i] = kk::align_bytes(d[i + 1], d[i], 2);             // block 2g: scale in d[0], nibbles after it
        od[i] = d[5 + i];                                       // block 2g + 1: scale in d[4]'s high half
    }
    uint32_t s2 = (d[0] & 0xffffu) | (d[4] & 0xffff0000u);
    if (GEN) {                                                  // blocks past K: scale 0 (their A is 0 too)
        const int b = step * kStepBlocks + 2 * g;
        s2 = b + 1 < blocks ? s2 : b < blocks ? s2 & 0xffffu : 0u;
    }
    transpose4(ev);
    transpose4(od);
    gather4(s2, sc);
    if (MT == 1) {
        __builtin_amdgcn_sched_barrier(0);
        raw = next();
        __builtin_amdgcn_sched_barrier(0);
    }
    float4v acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int b = 0; b < kStepBlocks; ++b) {
        const half8 bf = kk::q4_dword_halves((b & 1) ? od[b >> 1] : ev[b >> 1]);
        const float sd = kk::half_bits_to_float((b & 1) ? sc[b >> 1] >> 16 : sc[b >> 1] & 0xffffu);
        asm volatile("" ::: "memory");                          // few fragments live at once
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const half8 *f = a + (b * Q::Frags + 2 * t) * kWave;
            float4v q = {0.0f, 0.0f, 0.0f, 0.0f};
            q = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[0], bf, q, 0, 0, 0);
            if (!PACK) q = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[kWave], bf, q, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[t][r] = fmaf(sd, q[r], acc[t][r]);
        }
    }
    // columns 16 t + 4 g + r (PACK: column 4 (g % 2) + r, hi or lo part)
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const float4v iv = *reinterpret_cast<const float4v *>(inv + (PACK ? 4 * (g & 1) : 16 * t + 4 * g));
#pragma unroll
        for (int r = 0; r < 4; ++r) tot[t][r] = fmaf(acc[t][r], iv[r], tot[t][r]);
    }
    if (MT != 1) raw = next();
}

// GEN: any K % 32 == 0 and any weight alignment (dword loads, byte shifts,
// blocks past K masked); else K % 256 == 0 and 4-byte aligned weights.
// kSerial (one matrix, one tile per wave): a workgroup takes its tiles' ranges in turn, at_once
// of them at a time (whose fragments fit one chunk), and adds their sums in range order, as
// q4_split_sum does, so that no partial sum leaves it.
// kFused (a pair of one range): a gate tile and the up tile of the same rows go to two waves
// side by side, and the gate tile's wave stores SiLU(gate) * up; the summing launch and the
// trip through the workspace are 1.5 - 2 us of such a call (K1536 at 9 / 16 columns, us: N1000
// 11.0 / 11.2 with them, 9.2 / 9.4 without; N4096 11.2 / 11.4, 9.3 / 9.6; N11008 15.4 / 15.8,
// 13.8 / 14.0).
constexpr int kRanges = 0, kSerial = 1, kFused = 2;

template <int MT, bool PACK, bool GEN, int FORM>
__global__ __launch_bounds__(kQsThreads) void q4_split_gemv(const QsArgs p) {
    using Q = QsShape<MT, PACK>;
    constexpr bool SERIAL = FORM == kSerial, FUSED = FORM == kFused;
    extern __shared__ __align__(16) uint8_t qs_lds[];
    const int bid = blockIdx.x;
    const int idx = (bid % kXcds) * p.per_xcd + bid / kXcds;    // contiguous ranges per XCD share X in its L2
    if (idx >= p.total) return;                                 // whole workgroup, before any barrier
    const int range0 = SERIAL ? 0 : idx / p.groups, range1 = SERIAL ? p.ranges : range0 + 1;
    const int group = SERIAL ? idx : idx - range0 * p.groups;
    const int lane = threadIdx.x & (kWave - 1);
    const int wid = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int c16 = lane & 15, g = lane >> 4;
    const int at_once = SERIAL ? p.at_once : 1;
    const int tw = kQsWaves / (p.kgroups * at_once);            // waves along the tiles
    const int wt = wid % tw, kg = SERIAL ? wid / tw % p.kgroups : wid / tw;
    const int slot = SERIAL ? wid / (tw * p.kgroups) : 0;       // the wave's range of those at a time
    const int blocks = p.k >> 5;
    const uint32_t row_bytes = static_cast<uint32_t>(blocks) * 18u;
    // of a pair the gate matrix's tiles, then the up matrix's (FUSED: in turn, from an even tile)
    const int all_tiles = p.w2 ? 2 * p.tiles : p.tiles;
    const int first = group * p.per_group, end = min(first + p.per_group, all_tiles);
    const int rounds = SERIAL ? 1 : (p.per_group + tw - 1) / tw;   // tiles per wave (1 with several chunks)

    _Float16 *frag = reinterpret_cast<_Float16 *>(qs_lds);
    float *inv_lds = reinterpret_cast<float *>(qs_lds + Q::ChunkSteps * Q::StepBytes);

    const __amdgpu_buffer_rsrc_t x_rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p.x), 0, p.batch * p.k * 4, 0x00020000);
    for (int round = 0; round < rounds; ++round) {
        const int tile = first + round * tw + wt;
        const bool live = tile < end;                           // wave-uniform; an idle wave helps to convert X
        const bool up = FUSED ? tile & 1 : live && tile >= p.tiles;
        const int row = (FUSED ? tile >> 1 : up ? tile - p.tiles : tile) * 16 + c16;
        const uint8_t *m = up ? p.w2 : p.w;
        const uint32_t mis = GEN ? static_cast<uint32_t>(reinterpret_cast<uintptr_t>(m) & 3) : 0u;
        const uint32_t pos = mis + static_cast<uint32_t>(min(row, p.n - 1)) * row_bytes + 36u * g;
        const uint32_t off = GEN ? pos & ~3u : pos, shift = pos & 3u;
        // whole dwords up to the one that holds the matrix's last byte
        const uint32_t extent = (mis + static_cast<uint32_t>(p.n) * row_bytes + 3u) & ~3u;

        float4v sum[MT];                                        // SERIAL: the ranges'
#pragma unroll
        for (int t = 0; t < MT; ++t) sum[t] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
        for (int range = range0; range < range1; range += at_once) {
            const int here = SERIAL ? min(at_once, range1 - range) : 1;
            const int step0 = p.steps * range / p.ranges, step1 = p.steps * (range + here) / p.ranges;
            float4v tot[MT];
#pragma unroll
            for (int t = 0; t < MT; ++t) tot[t] = float4v{0.0f, 0.0f, 0.0f, 0.0f};

            for (int c0 = step0; c0 < step1; c0 += Q::ChunkSteps) {
                const int csteps = min(Q::ChunkSteps, step1 - c0);
                int from = c0, count = csteps;                  // the k-groups' steps of this chunk
                if (SERIAL && at_once > 1) {                    // one chunk: this wave's range of it
                    from = p.steps * min(range + slot, range1) / p.ranges;
                    count = p.steps * min(range + slot + 1, range1) / p.ranges - from;
                }
                const int s0 = from + count * kg / p.kgroups;
                const int s1 = live ? from + count * (kg + 1) / p.kgroups : s0;
                const int last = max(s1 - 1, c0);                   // past the end: re-read, not used
                QsRaw<GEN> raw;
                if (round == 0) {
                    // X of this chunk, then the first weight step: the memory counter
                    // is in order, so waiting for X leaves the weights in flight
                    const int items = Q::Cols * ((csteps + 1) >> 1);
                    float v[Q::Items][8];
#pragma unroll
                    for (int it = 0; it < Q::Items; ++it) {
                        const int item = wid + kQsWaves * it;
                        const int col = item % Q::Cols, pr = item / Q::Cols;
                        const int blk = (c0 + 2 * pr) * kStepBlocks + (lane >> 2);   // lane: block lane / 4, dword lane % 4
                        const bool in = item < items && col < p.batch && blk < blocks && blk < (c0 + csteps) * kStepBlocks;
                        // outside: past the extent, zeros without a memory access
                        const uint32_t xo = in ? (static_cast<uint32_t>(col) * p.k + 32 * blk + 4 * (lane & 3)) * 4u : 0x80000000u;
                        const u32x4 lo = __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, xo, 0, 0);
                        const u32x4 hi = __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, xo, 64, 0);
                        const uint32_t order[8] = {lo[0], lo[2], lo[1], lo[3], hi[0], hi[2], hi[1], hi[3]};
#pragma unroll
                        for (int t = 0; t < 8; ++t) v[it][t] = __uint_as_float(order[t]);
                    }
                    raw = qs_load<GEN>(m - mis, extent, off, min(s0, last) * kStepBytes);
                    if (c0 != step0 || (SERIAL && range > 0)) kk::lds_barrier();   // the last chunk's fragments are read
#pragma unroll
                    for (int it = 0; it < Q::Items; ++it) {
                        const int item = wid + kQsWaves * it;       // wave-uniform
                        if (item >= items) break;
                        qs_convert<MT, PACK, GEN>(v[it], item, lane, p.inf_bits, frag, inv_lds);
                    }
                    kk::lds_barrier();
                } else {
                    raw = qs_load<GEN>(m - mis, extent, off, min(s0, last) * kStepBytes);
                }
                for (int s = s0; s < s1; ++s) {
                    auto next = [&] { return qs_load<GEN>(m - mis, extent, off, min(s + 1, last) * kStepBytes); };
                    qs_step<MT, PACK, GEN>(raw, next, shift, s, blocks, g, reinterpret_cast<const half8 *>(frag) +
                                           (s - c0) * (kStepBlocks * Q::Frags * kWave) + lane, inv_lds + (s - c0) * Q::Cols, tot);
                }
            }

            // k-groups 1 .. KG-1 hand their sums to k-group 0, which adds them in
            // order (with several rounds the fragments stay: the exchange has LDS of its own)
            if (p.kgroups > 1) {
                float4v *xfer = reinterpret_cast<float4v *>(qs_lds + Q::RingBytes);
                if (round > 0) __syncthreads();                     // the round before's sums are read
                if (kg > 0) {
#pragma unroll
                    for (int t = 0; t < MT; ++t) xfer[((wid - tw) * MT + t) * kWave + lane] = tot[t];
                }
                __syncthreads();
                if (kg == 0)
                    for (int h = 1; h < p.kgroups; ++h)
#pragma unroll
                        for (int t = 0; t < MT; ++t) tot[t] += xfer[((wid + (h - 1) * tw) * MT + t) * kWave + lane];
            }
            if constexpr (PACK) {
                // A rows 8..15 (lanes 32..63) are the lo parts of columns 0..7
#pragma unroll
                for (int r = 0; r < 4; ++r) tot[0][r] += __shfl_down(tot[0][r], 32);
            }
#pragma unroll
            for (int t = 0; t < MT; ++t) sum[t] = SERIAL ? sum[t] + tot[t] : tot[t];
            if (SERIAL && at_once > 1) {
                // slots 1 .. hand theirs to slot 0 (in places that no k-group used)
                float4v *xfer = reinterpret_cast<float4v *>(qs_lds + Q::RingBytes);
                if (slot > 0 && kg == 0) {
#pragma unroll
                    for (int t = 0; t < MT; ++t) xfer[((wid - tw) * MT + t) * kWave + lane] = tot[t];
                }
                __syncthreads();
                if (slot == 0 && kg == 0)
                    for (int h = 1; h < here; ++h)
#pragma unroll
                        for (int t = 0; t < MT; ++t) sum[t] += xfer[((wid + (h * p.kgroups - 1) * tw) * MT + t) * kWave + lane];
            }
        }
        if constexpr (FUSED) {
            // in places that no k-group used (tw / 2 of the tw - 1 that are left)
            float4v *xfer = reinterpret_cast<float4v *>(qs_lds + Q::RingBytes) + (kQsWaves - tw + (wt >> 1)) * MT * kWave + lane;
            if (p.kgroups == 1 && round > 0) __syncthreads();   // the round before's are read
            if (up && kg == 0) {
#pragma unroll
                for (int t = 0; t < MT; ++t) xfer[t * kWave] = sum[t];
            }
            __syncthreads();
            if (!up && kg == 0) {
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    const float4v u = xfer[t * kWave];
#pragma unroll
                    for (int r = 0; r < 4; ++r) sum[t][r] = kk::swiglu_value(sum[t][r], u[r]);
                }
            }
        }
        if (live && kg == 0 && slot == 0 && !(FUSED && up) && row < p.n && !(PACK && g >= 2)) {
            float *out = p.out + (SERIAL ? 0 : static_cast<size_t>(range0) * (p.w2 ? 2 : 1) + (up ? 1 : 0)) * p.batch * p.row_stride + row;
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int col = 16 * t + 4 * g + r;
                    if (col < p.batch) out[static_cast<size_t>(col) * p.row_stride] = sum[t][r];
                }
        }
    }
}

// y[b][r] = the partial sums of the ranges, added in range order (PAIR:
// SiLU(gate) * up of the two matrices' sums). Four rows per thread.
constexpr int kSumThreads = 256;

template <bool PAIR>
__global__ __launch_bounds__(kSumThreads) void q4_split_sum(const float *__restrict__ part, float *__restrict__ y,
                                                            int n, int batch, int stride, int ranges) {
    const int quads = stride >> 2;
    const int i = blockIdx.x * kSumThreads + threadIdx.x;
    if (i >= batch * quads) return;
    const int col = i / quads, r0 = 4 * (i - col * quads);
    const size_t plane = static_cast<size_t>(batch) * stride;
    const float *src = part + static_cast<size_t>(col) * stride + r0;
    float4v a = {0.0f, 0.0f, 0.0f, 0.0f}, b = a;
#pragma unroll 4
    for (int s = 0; s < ranges; ++s) {
        a += *reinterpret_cast<const float4v *>(src + static_cast<size_t>(PAIR ? 2 * s : s) * plane);
        if (PAIR) b += *reinterpret_cast<const float4v *>(src + static_cast<size_t>(2 * s + 1) * plane);
    }
    if (PAIR) {
#pragma unroll
        for (int t = 0; t < 4; ++t) a[t] = kk::swiglu_value(a[t], b[t]);
    }
    float *dst = y + static_cast<size_t>(col) * n + r0;
    if ((n & 3) == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0) {
        *reinterpret_cast<float4v *>(dst) = a;
    } else {
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (r0 + t < n) dst[t] = a[t];
    }
}

struct QsPlan {
    int kgroups, ranges;   // KG, S
    int tiles, per_group, groups;   // 16-row tiles of one matrix; tiles of a workgroup; workgroups per range
    int stride;            // row stride of a partial sum
    size_t part_bytes;     // partial sums (0: one range stores y directly)
    bool fused;            // a pair of one range: kFused
};

// The partial sums of one matrix stay within the no-allocation entry point's
// scratch, so both entry points split alike.
constexpr size_t kMaxPartBytes = KUNLUN_NOALLOC_SCRATCH_BYTES;

int floor_pow2(int v) {
    int p = 1;
    while (2 * p <= v) p *= 2;
    return p;
}

// Steps whose fragments fit in LDS.
int qs_chunk(int batch) {
    return batch <= 8    ? QsShape<1, true>::ChunkSteps
           : batch <= 16 ? QsShape<1, false>::ChunkSteps : QsShape<2, false>::ChunkSteps;
}

// S: at most 6 steps (1536 values) per range, 4 above 16 columns, as a power of
// two, so that the fragments fit one chunk and the ranges' workgroups fill the
// CUs; up to 8 steps in one range where they fit one chunk, which saves the
// summing launch. Measured (us, 8 / 16 / 32 columns): K4096 x N4096 S = 4 10.0 /
// 10.3 / 13.9, S = 2 10.4 / 10.8 / 19.9, S = 8 10.3 / 10.6 / 13.8; K11008 x
// N4096 S = 16 13.8 / 15.1 / 19.5, 8 13.0 / 14.6 / 22.2, 4 13.4 / 18.4 / 29.8;
// K2048 x N5632 at 16 S = 1 8.7, 2 10.0, 4 9.8.
// Up to 16 columns, wide matrices take fewer and longer ranges as long as one chunk holds
// them: where a range's tiles are more than the 16 waves of its workgroups, each S writes
// and re-reads sums for nothing (S that the rule above gives / this, us): K8192 x N14336 at
// 8 columns 23.6 / 22.0 (S = 4), N28672 41.3 / 36.4 (2), K16384 x N14336 42.5 / 36.4 (4);
// at 16 K4096 x N32000 28.8 / 25.5 (2), K8192 x N28672 44.9 / 40.1 (4), pair K8192 x 2 x
// N14336 45.7 / 41.0; but K4096 x N14336 at 16 S = 4 16.4, 2 17.1, K8192 x N8192 at 8 S = 8 16.6.
// KG: the waves a CU's tiles leave idle (K4096 x N4096 S = 4: KG = 4 10.3,
// KG = 2 10.5, KG = 1 12.1). A pair takes its matrices' S and KG, so its sums
// are those of two single calls.
QsPlan qs_plan(int k, int n, int batch, bool pair, int cus) {
    QsPlan p;
    const int steps = (k + kStepK - 1) / kStepK;
    const int chunk = qs_chunk(batch);
    p.stride = (n + 3) & ~3;
    p.ranges = 1;
    if (steps > 8 || steps > chunk)
        while (p.ranges * (batch <= 16 ? 6 : 4) < steps) p.ranges *= 2;
    p.tiles = (n + 15) / 16;
    if (batch <= 16)
        while (p.ranges > 1 && static_cast<long>(p.tiles) * p.ranges > static_cast<long>(kQsWaves) * cus &&
               steps <= p.ranges / 2 * chunk)
            p.ranges /= 2;
    const size_t one = static_cast<size_t>(batch) * p.stride * 4;   // one range's sums
    while (p.ranges > 1 && p.ranges * one > kMaxPartBytes) p.ranges /= 2;
    // one workgroup per CU where the tiles allow; a range of several chunks
    // holds one tile per wave
    const int max_groups = std::max(1, cus / p.ranges);
    auto per_cu = [&](int tiles) { return (tiles + max_groups - 1) / max_groups; };
    p.kgroups = floor_pow2(std::max(1, std::min(kQsWaves / std::min(kQsWaves, per_cu(p.tiles)), steps / p.ranges)));
    const int all = pair ? 2 * p.tiles : p.tiles;
    p.fused = pair && p.ranges == 1 && p.kgroups <= kQsWaves / 2;   // two waves for a k-group's two tiles
    p.part_bytes = p.ranges == 1 && (!pair || p.fused) ? 0 : static_cast<size_t>(p.ranges) * (pair ? 2 : 1) * one;
    p.per_group = p.fused ? 2 * per_cu(p.tiles) : per_cu(all);
    if ((steps + p.ranges - 1) / p.ranges > chunk) p.per_group = std::min(p.per_group, kQsWaves / p.kgroups);
    p.groups = (all + p.per_group - 1) / p.per_group;
    return p;
}

template <int MT, bool PACK, bool GEN, int FORM>
hipError_t qs_launch(const QsArgs &a, hipStream_t stream) {
    using Q = QsShape<MT, PACK>;
    const hipError_t rc = kk::opt_in_lds(reinterpret_cast<const void *>(&q4_split_gemv<MT, PACK, GEN, FORM>), Q::LdsBytes);
    if (rc != hipSuccess) return rc;
    hipLaunchKernelGGL((q4_split_gemv<MT, PACK, GEN, FORM>), dim3(a.per_xcd * kXcds), dim3(kQsThreads), Q::LdsBytes, stream, a);
    return hipGetLastError();
}

template <int MT, bool PACK>
hipError_t qs_launch_form(const QsArgs &a, bool gen, int form, hipStream_t stream) {
    if (form == kSerial) return gen ? qs_launch<MT, PACK, true, kSerial>(a, stream) : qs_launch<MT, PACK, false, kSerial>(a, stream);
    if (form == kFused) return gen ? qs_launch<MT, PACK, true, kFused>(a, stream) : qs_launch<MT, PACK, false, kFused>(a, stream);
    return gen ? qs_launch<MT, PACK, true, kRanges>(a, stream) : qs_launch<MT, PACK, false, kRanges>(a, stream);
}

// Runs `p` (w2 null: one matrix); `workspace` holds p.part_bytes, or is null for one matrix:
// then the ranges of a tile run in one workgroup, with the same sums.
hipError_t qs_run(const QsPlan &p, const uint8_t *w, const uint8_t *w2, const float *x, float *y, int k, int n,
                  int batch, void *workspace, int cus, hipStream_t stream) {
    QsArgs a;
    a.w = w;
    a.w2 = w2;
    a.x = x;
    const bool serial = p.part_bytes && !workspace, split = p.part_bytes && workspace;
    a.out = split ? static_cast<float *>(workspace) : y;
    a.k = k;
    a.n = n;
    a.batch = batch;
    a.steps = (k + kStepK - 1) / kStepK;
    a.ranges = p.ranges;
    a.kgroups = p.kgroups;
    a.tiles = p.tiles;
    a.per_group = p.per_group;
    a.groups = p.groups;
    a.at_once = 1;
    if (serial) {   // one tile per wave, over all of K; the waves that the CUs' tiles leave idle take more ranges at a time
        a.per_group = std::min(kQsWaves / p.kgroups, (p.tiles + cus - 1) / cus);
        a.groups = (p.tiles + a.per_group - 1) / a.per_group;
        const int fit = qs_chunk(batch) / ((a.steps + p.ranges - 1) / p.ranges);
        while (2 * a.at_once <= std::min(fit, p.ranges) && 2 * a.at_once * p.kgroups * a.per_group <= kQsWaves) a.at_once *= 2;
    }
    a.total = serial ? a.groups : p.groups * p.ranges;
    a.per_xcd = (a.total + kXcds - 1) / kXcds;
    a.row_stride = split ? p.stride : n;
    const uintptr_t bits = reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(w2);
    const bool gen = k % kStepK != 0 || (bits & 3) != 0;
    a.inf_bits = k % 64 != 0 || (bits & 3) != 0 ? 0x7f800000u : 0xffffffffu;
    const int form = serial ? kSerial : p.fused ? kFused : kRanges;
    hipError_t rc = batch <= 8    ? qs_launch_form<1, true>(a, gen, form, stream)
                    : batch <= 16 ? qs_launch_form<1, false>(a, gen, form, stream)
                                  : qs_launch_form<2, false>(a, gen, form, stream);
    if (rc != hipSuccess || !split) return rc;
    const int threads = batch * (p.stride / 4);
    const dim3 grid((threads + kSumThreads - 1) / kSumThreads), block(kSumThreads);
    if (w2)
        hipLaunchKernelGGL(q4_split_sum<true>, grid, block, 0, stream, static_cast<const float *>(workspace), y, n, batch,
                           p.stride, p.ranges);
    else
        hipLaunchKernelGGL(q4_split_sum<false>, grid, block, 0, stream, static_cast<const float *>(workspace), y, n,
                           batch, p.stride, p.ranges);
    return hipGetLastError();
}

} // namespace

extern "C" size_t kk_q4_split_workspace_bytes(int k, int n, int batch, int pair, int cus) {
    return qs_plan(k, n, batch, pair != 0, cus).part_bytes;
}

extern "C" int kk_q4_split_gemv(const void *w, const void *w_up, const float *x, float *y, int k, int n, int batch,
                                void *workspace, int cus, hipStream_t stream) {
    if (!w || !x || !y || k <= 0 || (k & 31) || k > 16384 || n <= 0 || batch < 1 || batch > 32 || cus <= 0 ||
        static_cast<size_t>(n) * (k / 32 * 18) > 0x7fffffffu || (reinterpret_cast<uintptr_t>(x) & 3))
        return hipErrorInvalidValue;
    const QsPlan p = qs_plan(k, n, batch, w_up != nullptr, cus);
    if (p.part_bytes && !workspace && w_up) return hipErrorInvalidValue;
    return qs_run(p, static_cast<const uint8_t *>(w), static_cast<const uint8_t *>(w_up), x, y, k, n, batch, workspace,
                  cus, stream);
}
