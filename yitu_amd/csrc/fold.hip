// Sums of row ranges: out[range r, row i] = act_r((sum_k x[source_rk + i]) * factor_r), and its
// backward. The batched form of a heterogeneous model keeps the rows of all its relations in
// one buffer (yitu_amd/xgnn_h/batch.py); what stands between two batched products (the sum
// over the relations that reach a node type, the division by their number, the activation;
// test/common/model.py:137-171, 198-236) is this one pass, and so is the sum of the gradients
// of the places that read one node type.
// Bound by memory at large sizes (each row of x read once, each row of out written once) and
// by the launch at small ones: one thread per 4 floats of the output, the range of a row
// looked up in a table of a few dozen entries that stays in cache. 7,262 rows of 32 floats in
// five ranges: 2.5 us, where the division and the ReLU of each range were ten launches of 2.3.
#include <hip/hip_runtime.h>

#include "../../include/yitu_hip.h"
#include "common.hpp"

namespace yitu {
namespace {

static_assert(sizeof(YituFoldRange) == 32, "the table is read as 32-byte entries");

// The range that holds output row `row` (ranges tile the rows in ascending order).
__device__ __forceinline__ int range_of(const YituFoldRange *ranges, int n_ranges, int row) {
    int lo = 0, hi = n_ranges;  // ranges[lo].out_begin <= row < ranges[hi].out_begin
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (ranges[mid].out_begin <= row) lo = mid; else hi = mid;
    }
    return lo;
}

template <int VEC>
__global__ __launch_bounds__(kBlock) void fold_rows_kernel(float *__restrict__ out,
                                                           const float *__restrict__ x,
                                                           const YituFoldRange *__restrict__ ranges,
                                                           const int32_t *__restrict__ sources,
                                                           int n_ranges, int64_t n_vec, int row_vecs) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n_vec) return;
    const int row = (int)(i / row_vecs), c = (int)(i % row_vecs);
    const YituFoldRange r = ranges[range_of(ranges, n_ranges, row)];
    float v[VEC] = {};
    for (int k = 0; k < r.n_sources; k++) {
        float t[VEC];
        const int64_t from = (int64_t)sources[r.first_source + k] + row - r.out_begin;
        RowLoad<VEC, float>::ld(x + (from * row_vecs + c) * VEC, t);
#pragma unroll
        for (int j = 0; j < VEC; j++) v[j] += t[j];
    }
#pragma unroll
    for (int j = 0; j < VEC; j++) {
        if (r.factor != 1.0f) v[j] *= r.factor;
        if (r.act == YITU_FOLD_RELU) v[j] = v[j] > 0.0f || v[j] != v[j] ? v[j] : 0.0f;
        if (r.act == YITU_FOLD_ELU) v[j] = v[j] > 0.0f ? v[j] : r.alpha * expm1f(v[j]);
    }
    store_row<VEC>(out + i * VEC, v);
}

// grad_x of every source of a range = grad_out act'(out) factor. ReLU and ELU are
// differentiated at their own result (out > 0; alpha e^v = out + alpha).
template <int VEC>
__global__ __launch_bounds__(kBlock) void fold_rows_bwd_kernel(
    float *__restrict__ grad_x, const float *__restrict__ grad_out, const float *__restrict__ out,
    const YituFoldRange *__restrict__ ranges, const int32_t *__restrict__ sources, int n_ranges,
    int64_t n_vec, int row_vecs) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n_vec) return;
    const int row = (int)(i / row_vecs), c = (int)(i % row_vecs);
    const YituFoldRange r = ranges[range_of(ranges, n_ranges, row)];
    float g[VEC];
    RowLoad<VEC, float>::ld(grad_out + i * VEC, g);
    if (r.act != YITU_FOLD_NONE) {
        float y[VEC];
        RowLoad<VEC, float>::ld(out + i * VEC, y);
#pragma unroll
        for (int j = 0; j < VEC; j++) {
            if (r.act == YITU_FOLD_RELU) g[j] = y[j] <= 0.0f ? 0.0f : g[j];
            else g[j] = y[j] <= 0.0f ? g[j] * (y[j] + r.alpha) : g[j];
        }
    }
#pragma unroll
    for (int j = 0; j < VEC; j++)
        if (r.factor != 1.0f) g[j] *= r.factor;
    for (int k = 0; k < r.n_sources; k++) {
        const int64_t to = (int64_t)sources[r.first_source + k] + row - r.out_begin;
        store_row<VEC>(grad_x + (to * row_vecs + c) * VEC, g);
    }
}

}  // namespace
}  // namespace yitu

using namespace yitu;
#define YITU_API extern "C" __attribute__((visibility("default")))

// 16-byte vectors where the rows allow it, single floats otherwise.
YITU_API int yitu_fold_rows(float *out, const float *x, const YituFoldRange *ranges,
                            const int32_t *sources, int64_t n_ranges, int64_t n_rows, int64_t width,
                            void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    YITU_REQUIRE(n_ranges >= 0 && n_rows >= 0 && width >= 0 && n_rows < INT32_MAX &&
                     width < INT32_MAX, "size out of range");
    if (n_rows == 0 || width == 0) return 0;
    YITU_REQUIRE(out && x && ranges && sources && n_ranges > 0, "null operand");
    const bool wide = width % 4 == 0 && aligned16(out) && aligned16(x);
    const int row_vecs = (int)(wide ? width / 4 : width);
    const int64_t n_vec = n_rows * row_vecs, grid = ceil_div(n_vec, kBlock);
    YITU_REQUIRE(grid < INT32_MAX, "size out of range");
    if (wide)
        fold_rows_kernel<4><<<(int)grid, kBlock, 0, stream>>>(out, x, ranges, sources, (int)n_ranges,
                                                              n_vec, row_vecs);
    else
        fold_rows_kernel<1><<<(int)grid, kBlock, 0, stream>>>(out, x, ranges, sources, (int)n_ranges,
                                                              n_vec, row_vecs);
    YITU_LAUNCH_CHECK();
    return 0;
}

YITU_API int yitu_fold_rows_backward(float *grad_x, const float *grad_out, const float *out,
                                     const YituFoldRange *ranges, const int32_t *sources,
                                     int64_t n_ranges, int64_t n_rows, int64_t width,
                                     void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    YITU_REQUIRE(n_ranges >= 0 && n_rows >= 0 && width >= 0 && n_rows < INT32_MAX &&
                     width < INT32_MAX, "size out of range");
    if (n_rows == 0 || width == 0) return 0;
    YITU_REQUIRE(grad_x && grad_out && out && ranges && sources && n_ranges > 0, "null operand");
    const bool wide = width % 4 == 0 && aligned16(grad_x) && aligned16(grad_out) && aligned16(out);
    const int row_vecs = (int)(wide ? width / 4 : width);
    const int64_t n_vec = n_rows * row_vecs, grid = ceil_div(n_vec, kBlock);
    YITU_REQUIRE(grid < INT32_MAX, "size out of range");
    if (wide)
        fold_rows_bwd_kernel<4><<<(int)grid, kBlock, 0, stream>>>(
            grad_x, grad_out, out, ranges, sources, (int)n_ranges, n_vec, row_vecs);
    else
        fold_rows_bwd_kernel<1><<<(int)grid, kBlock, 0, stream>>>(
            grad_x, grad_out, out, ranges, sources, (int)n_ranges, n_vec, row_vecs);
    YITU_LAUNCH_CHECK();
    return 0;
}
