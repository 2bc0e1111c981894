// kunlun::Kernel and kunlun::matmul: argument validation exactly as the
// reference (reference src/k200.cpp:268-279), then submission of the HIP
// kernels for the weight format (reference dispatch src/k200.cpp:187-247).
#include "launch.h"
#include "runtime_internal.h"
#include "tuning.h"

#include <kunlun/k200_c.h>

#include <algorithm>
#include <climits>
#include <cstdint>

namespace kunlun {
namespace detail {
thread_local const char * last_route = nullptr;
const char * route_of_last_matmul() { return last_route; }
void note_route(const char * route) { last_route = route; }
} // namespace detail

namespace {

// Grows a Kernel-owned device workspace; waits for work that may still use
// the old one before releasing it.
void * grow(int id, detail::DeviceContext & ctx, void *& ptr, size_t & size, size_t need) {
    if (size < need) {
        if (ptr) {
            detail::check_hip(hipStreamSynchronize(ctx.stream), "hipStreamSynchronize");
            release(id, ptr, size);
            ptr = nullptr;
            size = 0;
        }
        ptr = allocate(id, need);
        require(ptr != nullptr);
        size = need;
    }
    return ptr;
}

// The split GEMV's partial sums differ from call to call of one program: what
// needs more than 1 MiB takes the no-allocation scratch's size at once, so a
// decode loop's first pass allocates once (each regrowth waits for the stream
// and frees, 25 us and at times some hundred).
void grow_split(int id, detail::DeviceContext & ctx, Kernel::Impl & impl, size_t need) {
    if (need > impl.gemm_workspace_size)
        need = std::max<size_t>(need, need > (1u << 20) ? KUNLUN_NOALLOC_SCRATCH_BYTES : 1u << 20);
    grow(id, ctx, impl.gemm_workspace, impl.gemm_workspace_size, need);
}

} // namespace
} // namespace kunlun

namespace kk {

// Route predicates, shared with the allocation-free entry point (noalloc.hip).
//
// Smallest batch that uses the fp16-MFMA prefill GEMM (F16 and Q4_0 weights);
// smaller batches keep the F32-accumulate GEMV kernels.
int gemm_min_batch() {
    const int v = kk::tuning(kk::kGemmMinBatch);
    return v > 0 ? v : 64;
}

// Batch range of the single-pass Q4_0 MFMA GEMV (within 1..16). Below the
// minimum the batch-1 kernel's passes (two columns each) are faster: the
// streamed kernel (K % 256 == 0, 16-byte aligned weights) wins from 3
// columns, the register-staged one from 5.
bool q4_mfma_batch(int batch, bool streamed) {
    const int min_b = std::max(1, kk::tuning_or(kk::kQ4MfmaMin, streamed ? 3 : 5));
    const int max_b = std::min(16, kk::tuning_or(kk::kQ4MfmaMax, 16));
    return batch >= min_b && batch <= max_b;
}

// Shapes that the batch-1 and -2 kernels take; the others are F32 arithmetic there
// (gemv_general), which the K-split kernel follows for an infinite activation.
bool q4_whole(const void * w, int k) { return k % 64 == 0 && ((uintptr_t)w & 3) == 0; }

// Whether the K-split Q4_0 MFMA GEMV may take a call (or a gate/up pair) that no faster
// route took: the single-pass MFMA GEMV's batch range (above 16 columns: where it holds
// 16), in which shapes the batch-1 kernels cannot take (K % 64 != 0, weights off a dword)
// count from 3 columns (K5600 x N3000: 3 / 8 / 16 columns 27 / 63 / 123 us on
// the general GEMV, 13 / 13 / 14 us split).
bool q4_split_range(const void * w, int k, int batch) {
    const bool whole = q4_whole(w, k);
    return q4_mfma_batch(std::min(batch, 16), !whole || (k % 256 == 0 && ((uintptr_t)w & 15) == 0));
}

// One matrix: not where the general GEMV has little to do. It gives a wave one row of 64
// blocks at a time and up to 8 columns per pass, so its time goes with those passes x
// columns x the workgroups (4 rows) that share a CU. us general / split at N300, N1000:
// K544 8 columns 7.3 / 8.1, K1056 3 columns 6.7 / 8.9, 8 columns 8.5 / 8.9, 12 columns
// 12.6 / 9.5; K2976 (two passes) 3 columns 8.6 / 11.6, 5 columns 11.3 / 11.7, 6 columns
// 12.6 / 11.7; K4128 3 columns 11.2 / 11.2; at N3000 K544 3 columns 7.7 / 8.2, 4 columns 8.9 / 8.2.
bool q4_split_route(const void * w, int k, int n, int batch, int cus) {
    const long general = (k + 2047L) / 2048 * batch * ((n + 4L * cus - 1) / (4L * cus));
    return q4_split_range(w, k, batch) && (q4_whole(w, k) || batch > 8 || general > 10);
}

// F32 weights above the single-pass GEMV's 16 columns (K4096 x N4096 at 17
// columns: 28.4 us in passes of 16, 18.4 us), except up to 48 columns of a part of one
// row tile (K8192 x N1 at 17 / 33 / 48 / 64 columns: 22.9 / 38.1 / 46.0 / 61.0 us in passes, 30.0 /
// 48.5 / 48.5 / 48.7) and 17 of few rows (K4096 x N17 16.1 / 17.6, at 18 20.2 / 16.8).
bool f32_gemm_route(int type, const void * w, const void * x, int n, int batch) {
    return type == 0 && batch > 16 && batch > (n < 16 ? 48 : n <= 48 ? 17 : 16) && dense_mfma_batch(16) &&
           (((uintptr_t)w | (uintptr_t)x) & 15) == 0;
}

// Columns of such a call on the F32 GEMM: its 33rd alone would double the column tile, which
// on few and long rows takes longer than a pass of its own (K8192 x N65 at 33 columns: 47.7 us
// in passes of 16, 49.2 in one tile of 64, 42.0 as 32 + 1; K11008 x N300 66.7 / 65.5 / 55.3).
int f32_gemm_columns(int k, int n, int batch) { return batch == 33 && k >= 4096 && n <= 1024 ? 32 : batch; }

// Columns of one pass of batches above the small-batch kernels and off the GEMM.
int gemv_chunk(int type) { return type == 2 && q4_mfma_batch(16, true) ? 32 : 16; }

// Batch range of the block-diagonal Q4_0 MFMA GEMV (the single-pass kernel's
// range, unless KUNLUN_Q4_BDIAG=0 leaves it to the K-split kernel).
bool q4_bdiag_batch(int batch) {
    return kk::tuning_or(kk::kQ4Bdiag, 1) != 0 && q4_mfma_batch(batch, true);
}

// Batch range of the streamed Q4_0 GEMV at K = 4096: KUNLUN_Q4_STREAM_MIN
// (default 5) to 8; a minimum above 8 turns it off.
bool q4_stream_batch(int batch) {
    const int min_b = kk::tuning_or(kk::kQ4StreamMin, 5);
    return batch >= std::max(1, min_b) && batch <= 8;
}

// Batch range of the single-pass F32/F16 MFMA GEMV (within 1..16).
bool dense_mfma_batch(int batch) {
    const int min_b = std::max(1, kk::tuning_or(kk::kDenseMfmaMin, 2));
    const int max_b = std::min(16, kk::tuning_or(kk::kDenseMfmaMax, 16));
    return batch >= min_b && batch <= max_b;
}

} // namespace kk

namespace kunlun {
using kk::dense_mfma_batch;
using kk::gemm_min_batch;
using kk::q4_mfma_batch;

namespace {

// The reference's matmul argument rules (reference src/k200.cpp:271-275):
// supported type, K % 32 == 0, K <= 16384, products that fit int, and a
// weight matrix of at most INT_MAX bytes.
void validate_shape(const void * y, const void * w, const void * x, int k, int n, int batch, WeightType type,
                    int tile) {
    require(type == WeightType::f32 || type == WeightType::f16 || type == WeightType::q4_0 ||
            type == WeightType::rowwise_i8);
    require(k > 0 && k <= 16384 && k % 32 == 0 && n > 0 && batch > 0 && n <= INT_MAX / batch &&
            k <= INT_MAX / batch);
    require((size_t)n * batch <= INT_MAX / 4 && (size_t)k * batch <= INT_MAX / 4);
    const size_t row_bytes = type == WeightType::f32   ? (size_t)k * 4
                             : type == WeightType::f16 ? (size_t)k * 2
                             : type == WeightType::q4_0 ? (size_t)k / 32 * 18
                                                        : (size_t)k;
    require(y && w && x && (size_t)n <= INT_MAX / row_bytes && (tile == 1 || tile == 16));
}

} // namespace

Kernel::Kernel() : impl_(new Impl{}) {}

Kernel::~Kernel() {
    std::lock_guard<std::recursive_mutex> lock(detail::mutex());
    if (impl_->id >= 0) {
        select(impl_->id);
        check(wait());
        release(impl_->id, impl_->i8_workspace, impl_->i8_workspace_size);
        release(impl_->id, impl_->gemm_workspace, impl_->gemm_workspace_size);
        release(impl_->id, impl_->pair_workspace, impl_->pair_workspace_size);
    }
    delete impl_;
}

// The F32/F16/Q4_0 product's route for one matrix (matmul's, and each half of
// an unfused gate/up pair): the prefill GEMM, the small-batch MFMA GEMVs,
// else the single-pass GEMVs.
static void dispatch_dense(Kernel::Impl & impl, detail::DeviceContext & ctx, int id, void * y, const void * w,
                    const void * x, int k, int n, int batch, WeightType type) {
    const bool gemm = (type == WeightType::q4_0 || (type == WeightType::f16 && ((uintptr_t)w & 15) == 0)) &&
                      batch >= gemm_min_batch() && ((uintptr_t)x & 15) == 0;
    if (kk::f32_gemm_route((int)type, w, x, n, batch)) {
        const int columns = kk::f32_gemm_columns(k, n, batch);
        detail::check_hip((hipError_t)kk_f32_gemm(w, static_cast<const float *>(x), static_cast<float *>(y), k, n,
                                                  columns, ctx.cus, ctx.stream),
                          "kk_f32_gemm");
        if (columns < batch)
            dispatch_dense(impl, ctx, id, static_cast<char *>(y) + (size_t)columns * n * 4, w,
                           static_cast<const char *>(x) + (size_t)columns * k * 4, k, n, batch - columns, type);
        impl.route = "f32_mfma_gemv";
        return;
    }
    const int chunk = kk::gemv_chunk((int)type);
    if (!gemm && batch > chunk) {
        // batches between the small-batch kernels and the GEMM: chunks of 32
        // (Q4_0) or 16 columns, each on the route a call of that many columns
        // takes (one pass over the weights per chunk). X and Y chunks keep
        // their alignment (K % 32 == 0).
        const char * first = nullptr;
        for (int b0 = 0; b0 < batch; b0 += chunk) {
            dispatch_dense(impl, ctx, id, static_cast<char *>(y) + (size_t)b0 * n * 4, w,
                           static_cast<const char *>(x) + (size_t)b0 * k * 4, k, n, std::min(chunk, batch - b0), type);
            if (!first) first = impl.route;
        }
        impl.route = first;
        return;
    }
    if (gemm) {
        grow(id, ctx, impl.gemm_workspace, impl.gemm_workspace_size, kk_gemm_workspace_bytes(k, n, batch, 0));
        detail::check_hip((hipError_t)kk_gemm((int)type, w, static_cast<const float *>(x), static_cast<float *>(y), k,
                                              n, batch, impl.gemm_workspace, ctx.stream, &impl.route),
                          "kk_gemm");
    } else if ((type == WeightType::f32 || type == WeightType::f16) && dense_mfma_batch(batch) &&
               ((uintptr_t)w & 15) == 0 && ((uintptr_t)x & 15) == 0) {
        detail::check_hip((hipError_t)kk_dense_mfma_gemv((int)type, w, static_cast<const float *>(x),
                                                         static_cast<float *>(y), k, n, batch, ctx.stream),
                          "kk_dense_mfma_gemv");
        impl.route = type == WeightType::f16 ? "f16_mfma_gemv" : "f32_mfma_gemv";
    } else if (type == WeightType::q4_0 && kk::q4_stream_batch(batch) &&
               kk_q4_stream_gemv_supported(w, static_cast<const float *>(x), k, n, batch)) {
        detail::check_hip((hipError_t)kk_q4_stream_gemv(w, static_cast<const float *>(x), static_cast<float *>(y), k, n,
                                                        batch, ctx.cus, ctx.stream),
                          "kk_q4_stream_gemv");
        impl.route = "q4_stream_gemv";
    } else if (type == WeightType::q4_0 && kk::q4_bdiag_batch(batch) &&
               kk_q4_bdiag_gemv_supported(w, static_cast<const float *>(x), k, n, batch)) {
        detail::check_hip((hipError_t)kk_q4_bdiag_gemv(w, static_cast<const float *>(x), static_cast<float *>(y), k, n,
                                                       batch, ctx.cus, ctx.stream),
                          "kk_q4_bdiag_gemv");
        impl.route = "q4_bdiag_gemv";
    } else if (type == WeightType::q4_0 && kk::q4_split_route(w, k, n, batch, ctx.cus)) {
        grow_split(id, ctx, impl, kk_q4_split_workspace_bytes(k, n, batch, 0, ctx.cus));
        detail::check_hip((hipError_t)kk_q4_split_gemv(w, nullptr, static_cast<const float *>(x),
                                                       static_cast<float *>(y), k, n, batch, impl.gemm_workspace,
                                                       ctx.cus, ctx.stream),
                          "kk_q4_split_gemv");
        impl.route = "q4_mfma_gemv";
    } else {
        detail::check_hip((hipError_t)kk_dense_matmul((int)type, w, static_cast<const float *>(x),
                                                      static_cast<float *>(y), k, n, batch, ctx.stream,
                                                      &impl.route),
                          "kk_dense_matmul");
    }
}

void matmul(Kernel & kernel, int id, void * y, const void * w, const void * x, int k, int n, int batch,
            WeightType type, const float * scales, const float * maximum, int tile) {
    std::lock_guard<std::recursive_mutex> lock(detail::mutex());
    validate_shape(y, w, x, k, n, batch, type, tile);
    require(kernel.impl_->id == -1 || kernel.impl_->id == id);
    require(type != WeightType::rowwise_i8 || (scales && maximum));
    // F32 activations and outputs must be element aligned (an F32 array always is).
    require(((uintptr_t)x & 3) == 0 && ((uintptr_t)y & 3) == 0);

    detail::DeviceContext & ctx = detail::context(id);
    Kernel::Impl & impl = *kernel.impl_;
    impl.id = id;
    if (type == WeightType::rowwise_i8) {
        require(((uintptr_t)w & 3) == 0 && ((uintptr_t)scales & 3) == 0 && ((uintptr_t)maximum & 3) == 0);
        if (kk_i8_gemv_rows_supported(k, batch)) {
            detail::check_hip((hipError_t)kk_i8_gemv_rows(static_cast<const float *>(x), static_cast<const int8_t *>(w),
                                                          scales, maximum, static_cast<float *>(y), k, n, ctx.cus,
                                                          ctx.status, ctx.stream),
                              "kk_i8_gemv_rows");
            ctx.status_pending = true;
            impl.route = "i8_rows_gemv";
            detail::last_route = impl.route;
            detail::count_matmul(id);
            return;
        }
        if (kk_i8_gemv_fused_supported(k, batch)) {
            detail::check_hip((hipError_t)kk_i8_gemv_fused(static_cast<const float *>(x),
                                                           static_cast<const int8_t *>(w), scales, maximum,
                                                           static_cast<float *>(y), k, n, batch, ctx.status,
                                                           ctx.stream),
                              "kk_i8_gemv_fused");
            ctx.status_pending = true;
            impl.route = "i8_fused_gemv";
            detail::last_route = impl.route;
            detail::count_matmul(id);
            return;
        }
        grow(id, ctx, impl.i8_workspace, impl.i8_workspace_size, kk_i8_workspace_bytes(k, batch));
        detail::check_hip((hipError_t)kk_i8_quantize(static_cast<const float *>(x), k, batch, impl.i8_workspace,
                                                     ctx.status, ctx.stream),
                          "kk_i8_quantize");
        ctx.status_pending = true;
        detail::check_hip((hipError_t)kk_i8_matmul(impl.i8_workspace, static_cast<const int8_t *>(w), scales,
                                                   maximum, static_cast<float *>(y), k, n, batch, ctx.stream,
                                                   &impl.route),
                          "kk_i8_matmul");
    } else {
        dispatch_dense(impl, ctx, id, y, w, x, k, n, batch, type);
    }
    detail::last_route = impl.route;
    detail::count_matmul(id);
}

// Q4_0 gate/up pair of `batch` columns, batch 1..32: the batch-1/2 GEMV's, the
// streamed, block-diagonal or K-split GEMV's pair form, whichever takes the
// shape; none: two GEMVs and SwiGLU instead.
enum class Q4PairRoute { none, dot8, stream, bdiag, split };

static Q4PairRoute q4_pair_route(const void * w_gate, const void * w_up, const float * x, int k, int n, int batch) {
    if (kk_q4_gemv_pair_swiglu_supported(w_gate, w_up, x, k, n, batch)) return Q4PairRoute::dot8;
    if (kk::q4_stream_batch(batch) && kk_q4_stream_gemv_supported(w_gate, x, k, n, batch) &&
        kk_q4_stream_gemv_supported(w_up, x, k, n, batch))
        return Q4PairRoute::stream;
    if (kk::q4_bdiag_batch(batch) && kk_q4_bdiag_gemv_supported(w_gate, x, k, n, batch) &&
        kk_q4_bdiag_gemv_supported(w_up, x, k, n, batch))
        return Q4PairRoute::bdiag;
    // (one matrix on a dword and one off it: each on its own rule for infinities)
    if (kk::q4_split_range(w_gate, k, batch) && kk::q4_split_range(w_up, k, batch) &&
        kk::q4_whole(w_gate, k) == kk::q4_whole(w_up, k))
        return Q4PairRoute::split;
    return Q4PairRoute::none;
}

static void run_q4_pair(Q4PairRoute route, Kernel::Impl & impl, detail::DeviceContext & ctx, int id, float * y,
                        const void * w_gate, const void * w_up, const float * x, int k, int n, int batch) {
    switch (route) {
    case Q4PairRoute::dot8:
        // decode: both matrices in one GEMV pass, SwiGLU in its epilogue
        detail::check_hip((hipError_t)kk_q4_gemv_pair_swiglu(w_gate, w_up, x, y, k, n, batch, ctx.stream),
                          "kk_q4_gemv_pair_swiglu");
        impl.route = "q4_gemv_fused_pair_swiglu";
        break;
    case Q4PairRoute::stream:
        detail::check_hip((hipError_t)kk_q4_stream_gemv_pair_swiglu(w_gate, w_up, x, y, k, n, batch, ctx.cus, ctx.stream),
                          "kk_q4_stream_gemv_pair_swiglu");
        impl.route = "q4_stream_pair_swiglu";
        break;
    case Q4PairRoute::bdiag:
        detail::check_hip((hipError_t)kk_q4_bdiag_gemv_pair_swiglu(w_gate, w_up, x, y, k, n, batch, ctx.cus, ctx.stream),
                          "kk_q4_bdiag_gemv_pair_swiglu");
        impl.route = "q4_bdiag_pair_swiglu";
        break;
    case Q4PairRoute::split:
        // both products' K ranges in one launch, their sums and SwiGLU in the next (one range: in the same)
        grow_split(id, ctx, impl, kk_q4_split_workspace_bytes(k, n, batch, 1, ctx.cus));
        detail::check_hip((hipError_t)kk_q4_split_gemv(w_gate, w_up, x, y, k, n, batch, impl.gemm_workspace, ctx.cus,
                                                       ctx.stream),
                          "kk_q4_split_gemv");
        impl.route = "q4_mfma_pair_swiglu";
        break;
    case Q4PairRoute::none:
        break;
    }
}

void matmul_swiglu(Kernel & kernel, int id, void * y, const void * w_gate, const void * w_up, const void * x,
                   int k, int n, int batch, WeightType type) {
    std::lock_guard<std::recursive_mutex> lock(detail::mutex());
    require(type == WeightType::f32 || type == WeightType::f16 || type == WeightType::q4_0);
    validate_shape(y, w_gate, x, k, n, batch, type, 16);
    require(w_up != nullptr);
    require(kernel.impl_->id == -1 || kernel.impl_->id == id);
    require(((uintptr_t)x & 3) == 0 && ((uintptr_t)y & 3) == 0);

    detail::DeviceContext & ctx = detail::context(id);
    Kernel::Impl & impl = *kernel.impl_;
    impl.id = id;
    const int chunk = kk::gemv_chunk((int)type);
    const bool f16_aligned = ((uintptr_t)w_gate & 15) == 0 && ((uintptr_t)w_up & 15) == 0;
    if ((type == WeightType::q4_0 || (type == WeightType::f16 && f16_aligned)) && batch >= gemm_min_batch() &&
        ((uintptr_t)x & 15) == 0) {
        grow(id, ctx, impl.gemm_workspace, impl.gemm_workspace_size, kk_gemm_workspace_bytes(k, n, batch, 1));
        detail::check_hip((hipError_t)kk_gemm_swiglu((int)type, w_gate, w_up, static_cast<const float *>(x),
                                                     static_cast<float *>(y), k, n, batch, impl.gemm_workspace,
                                                     ctx.stream, &impl.route),
                          "kk_gemm_swiglu");
    } else if (type == WeightType::q4_0 && batch <= chunk &&
               q4_pair_route(w_gate, w_up, static_cast<const float *>(x), k, n, batch) != Q4PairRoute::none) {
        // decode and small batch: both products and SwiGLU in one launch
        run_q4_pair(q4_pair_route(w_gate, w_up, static_cast<const float *>(x), k, n, batch), impl, ctx, id,
                    static_cast<float *>(y), w_gate, w_up, static_cast<const float *>(x), k, n, batch);
    } else if (type == WeightType::q4_0 && batch > chunk &&
               q4_pair_route(w_gate, w_up, static_cast<const float *>(x), k, n, chunk) != Q4PairRoute::none &&
               (batch % chunk == 0 || q4_pair_route(w_gate, w_up, static_cast<const float *>(x), k, n, batch % chunk) !=
                                          Q4PairRoute::none)) {
        // batches between the small-batch kernels and the GEMM: chunks of
        // columns, each on its own pair route (X and Y chunks keep their
        // alignment: K % 32 == 0)
        const char * first = nullptr;
        for (int b0 = 0; b0 < batch; b0 += chunk) {
            const int cols = std::min(chunk, batch - b0);
            const float * xc = reinterpret_cast<const float *>(static_cast<const char *>(x) + (size_t)b0 * k * 4);
            run_q4_pair(q4_pair_route(w_gate, w_up, xc, k, n, cols), impl, ctx, id,
                        reinterpret_cast<float *>(static_cast<char *>(y) + (size_t)b0 * n * 4), w_gate, w_up, xc, k, n,
                        cols);
            if (!first) first = impl.route;
        }
        impl.route = first;
    } else {
        // gate and up rows side by side in the workspace: [batch][2n] F32
        const size_t half = (size_t)batch * n * 4;
        grow(id, ctx, impl.pair_workspace, impl.pair_workspace_size, 2 * half);
        float * gate = static_cast<float *>(impl.pair_workspace);
        float * up = reinterpret_cast<float *>(static_cast<char *>(impl.pair_workspace) + half);
        // each product on matmul's own route for its shape
        dispatch_dense(impl, ctx, id, gate, w_gate, x, k, n, batch, type);
        dispatch_dense(impl, ctx, id, up, w_up, x, k, n, batch, type);
        detail::check_hip((hipError_t)kk_swiglu(y, gate, up, n, batch, n * 4, n * 4, n * 4, 4, ctx.stream),
                          "kk_swiglu");
        impl.route = type == WeightType::q4_0 ? "q4_gemv_pair_swiglu"
                     : type == WeightType::f16 ? "f16_gemv_pair_swiglu"
                                               : "f32_gemv_pair_swiglu";
    }
    detail::last_route = impl.route;
    detail::count_matmul(id);
    detail::count_matmul(id);
}

} // namespace kunlun
