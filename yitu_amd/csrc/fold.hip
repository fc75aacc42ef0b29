// Sums of row ranges: out[range r, row i] = act_r((sum_k x[source_rk + i]) * factor_r), and its
// backward. The batched form of a heterogeneous model keeps the rows of all its relations in
// one buffer (yitu_amd/xgnn_h/batch.py); what stands between two batched products (the sum
// over the relations that reach a node type, the division by their number, the activation;
// test/common/model.py:137-171, 198-236) is this one pass, and so is the sum of the gradients
// of the places that read one node type.
// Bound by memory at large sizes (each row of x read once, each row of out written once) and by
// the launch at small ones. The range of a row is looked up in a table of a few dozen entries
// that stays in cache; as a chain of dependent loads before the row itself it held large folds at
// 3.4 TB/s. Where a workgroup's rows lie in one range, the lookup is the workgroup's own, and from
// kManyVecs 16-byte vectors on (1,024 workgroups of four each) a thread has kPerThread of them
// under way: 491,520 rows of 256 floats divided 298 -> 156 us (6.4 TB/s), two such ranges added up
// 430 -> 290 us; 7,262 rows of 32 floats in five ranges 3.2 us, where the division and the ReLU
// of each range were ten launches of 2.3.
#include <hip/hip_runtime.h>

#include "../../include/yitu_hip.h"
#include "common.hpp"

namespace yitu {
namespace {

static_assert(sizeof(YituFoldRange) == 32, "the table is read as 32-byte entries");

constexpr int kPerThread = 4;
constexpr int64_t kManyVecs = 1 << 20;

// The range that holds output row `row` (ranges tile the rows in ascending order).
__device__ __forceinline__ int range_of(const YituFoldRange *ranges, int n_ranges, int row) {
    int lo = 0, hi = n_ranges;  // ranges[lo].out_begin <= row < ranges[hi].out_begin
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (ranges[mid].out_begin <= row) lo = mid; else hi = mid;
    }
    return lo;
}

__device__ __forceinline__ float fold_act(const YituFoldRange &r, float v) {
    if (r.factor != 1.0f) v *= r.factor;
    if (r.act == YITU_FOLD_RELU) v = v > 0.0f || v != v ? v : 0.0f;
    if (r.act == YITU_FOLD_ELU) v = v > 0.0f ? v : r.alpha * expm1f(v);
    return v;
}
// ReLU and ELU are differentiated at their own result y (y > 0; alpha e^v = y + alpha).
__device__ __forceinline__ float fold_act_bwd(const YituFoldRange &r, float g, float y) {
    if (r.act == YITU_FOLD_RELU) g = y <= 0.0f ? 0.0f : g;
    if (r.act == YITU_FOLD_ELU) g = y <= 0.0f ? g * (y + r.alpha) : g;
    return r.factor != 1.0f ? g * r.factor : g;
}

// The vectors of a workgroup: PER of each thread, kBlock apart. `one`: they lie in one range, whose
// table entry is then the workgroup's (scalar loads), and a source's vector is the output's at a
// distance: no division and no dependent lookup a thread.
template <int PER>
struct FoldBlock {
    int64_t first, n_vec;
    int row_vecs, index;
    bool one;
    __device__ __forceinline__ FoldBlock(const YituFoldRange *ranges, int n_ranges, int64_t n,
                                         int row_vecs_)
        : first((int64_t)blockIdx.x * (PER * kBlock)), n_vec(n), row_vecs(row_vecs_) {
        const int64_t last = min(first + PER * kBlock, n_vec) - 1;
        index = __builtin_amdgcn_readfirstlane(range_of(ranges, n_ranges, row(first)));
        one = row(last) - ranges[index].out_begin < ranges[index].rows;
    }
    __device__ __forceinline__ int row(int64_t vec) const {
        return n_vec <= UINT32_MAX ? (int)((unsigned)vec / (unsigned)row_vecs) : (int)(vec / row_vecs);
    }
    __device__ __forceinline__ int64_t vec(int u) const { return first + u * kBlock + threadIdx.x; }
    __device__ __forceinline__ int64_t distance(const YituFoldRange &r, const int32_t *sources,
                                                int k) const {
        return (int64_t)(sources[r.first_source + k] - r.out_begin) * row_vecs;
    }
};

template <int VEC, int PER>
__global__ __launch_bounds__(kBlock) void fold_rows_kernel(float *__restrict__ out,
                                                           const float *__restrict__ x,
                                                           const YituFoldRange *__restrict__ ranges,
                                                           const int32_t *__restrict__ sources,
                                                           int n_ranges, int64_t n_vec, int row_vecs) {
    const FoldBlock<PER> b(ranges, n_ranges, n_vec, row_vecs);
    if (b.one) {
        const YituFoldRange r = ranges[b.index];
        float v[PER][VEC] = {};
        int64_t at[PER];
#pragma unroll
        for (int u = 0; u < PER; u++) at[u] = min(b.vec(u), n_vec - 1);
#pragma unroll 2
        for (int k = 0; k < r.n_sources; k++) {
            const int64_t d = b.distance(r, sources, k);
            float t[PER][VEC];
#pragma unroll
            for (int u = 0; u < PER; u++) RowLoad<VEC, float>::ld(x + (at[u] + d) * VEC, t[u]);
#pragma unroll
            for (int u = 0; u < PER; u++)
#pragma unroll
                for (int j = 0; j < VEC; j++) v[u][j] += t[u][j];
        }
#pragma unroll
        for (int u = 0; u < PER; u++) {
#pragma unroll
            for (int j = 0; j < VEC; j++) v[u][j] = fold_act(r, v[u][j]);
            if (b.vec(u) < n_vec) store_row<VEC>(out + b.vec(u) * VEC, v[u]);
        }
        return;
    }
    for (int u = 0; u < PER; u++) {
        const int64_t i = b.vec(u);
        if (i >= n_vec) return;
        const YituFoldRange r = ranges[range_of(ranges, n_ranges, b.row(i))];
        float v[VEC] = {};
        for (int k = 0; k < r.n_sources; k++) {
            float t[VEC];
            RowLoad<VEC, float>::ld(x + (i + b.distance(r, sources, k)) * VEC, t);
#pragma unroll
            for (int j = 0; j < VEC; j++) v[j] += t[j];
        }
#pragma unroll
        for (int j = 0; j < VEC; j++) v[j] = fold_act(r, v[j]);
        store_row<VEC>(out + i * VEC, v);
    }
}

// grad_x of every source of a range = grad_out act'(out) factor.
template <int VEC, int PER>
__global__ __launch_bounds__(kBlock) void fold_rows_bwd_kernel(
    float *__restrict__ grad_x, const float *__restrict__ grad_out, const float *__restrict__ out,
    const YituFoldRange *__restrict__ ranges, const int32_t *__restrict__ sources, int n_ranges,
    int64_t n_vec, int row_vecs) {
    const FoldBlock<PER> b(ranges, n_ranges, n_vec, row_vecs);
    if (b.one) {
        const YituFoldRange r = ranges[b.index];
        float g[PER][VEC], y[PER][VEC] = {};
#pragma unroll
        for (int u = 0; u < PER; u++) {
            const int64_t i = min(b.vec(u), n_vec - 1);
            RowLoad<VEC, float>::ld(grad_out + i * VEC, g[u]);
            if (r.act != YITU_FOLD_NONE) RowLoad<VEC, float>::ld(out + i * VEC, y[u]);
        }
#pragma unroll
        for (int u = 0; u < PER; u++)
#pragma unroll
            for (int j = 0; j < VEC; j++) g[u][j] = fold_act_bwd(r, g[u][j], y[u][j]);
        for (int k = 0; k < r.n_sources; k++) {
            const int64_t d = b.distance(r, sources, k);
#pragma unroll
            for (int u = 0; u < PER; u++)
                if (b.vec(u) < n_vec) store_row<VEC>(grad_x + (b.vec(u) + d) * VEC, g[u]);
        }
        return;
    }
    for (int u = 0; u < PER; u++) {
        const int64_t i = b.vec(u);
        if (i >= n_vec) return;
        const YituFoldRange r = ranges[range_of(ranges, n_ranges, b.row(i))];
        float g[VEC], y[VEC] = {};
        RowLoad<VEC, float>::ld(grad_out + i * VEC, g);
        if (r.act != YITU_FOLD_NONE) RowLoad<VEC, float>::ld(out + i * VEC, y);
#pragma unroll
        for (int j = 0; j < VEC; j++) g[j] = fold_act_bwd(r, g[j], y[j]);
        for (int k = 0; k < r.n_sources; k++)
            store_row<VEC>(grad_x + (i + b.distance(r, sources, k)) * VEC, g);
    }
}

// f(floats of a vector, vectors of a thread): 16-byte vectors where the rows allow it, single floats
// otherwise; several vectors a thread once that leaves every CU a few workgroups.
template <typename F>
void with_form(bool wide, int64_t n_vec, F f) {
    const bool many = n_vec >= kManyVecs;
    const auto per = [&](auto vec) {
        if (many) f(vec, std::integral_constant<int, kPerThread>());
        else f(vec, std::integral_constant<int, 1>());
    };
    if (wide) per(std::integral_constant<int, 4>());
    else per(std::integral_constant<int, 1>());
}

}  // namespace
}  // namespace yitu

using namespace yitu;
#define YITU_API extern "C" __attribute__((visibility("default")))

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
    const int64_t n_vec = n_rows * row_vecs;
    YITU_REQUIRE(ceil_div(n_vec, kBlock) < INT32_MAX, "size out of range");
    with_form(wide, n_vec, [&](auto vec, auto per) {
        constexpr int V = decltype(vec)::value, P = decltype(per)::value;
        fold_rows_kernel<V, P><<<(int)ceil_div(n_vec, kBlock * P), kBlock, 0, stream>>>(
            out, x, ranges, sources, (int)n_ranges, n_vec, row_vecs);
    });
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
    const int64_t n_vec = n_rows * row_vecs;
    YITU_REQUIRE(ceil_div(n_vec, kBlock) < INT32_MAX, "size out of range");
    with_form(wide, n_vec, [&](auto vec, auto per) {
        constexpr int V = decltype(vec)::value, P = decltype(per)::value;
        fold_rows_bwd_kernel<V, P><<<(int)ceil_div(n_vec, kBlock * P), kBlock, 0, stream>>>(
            grad_x, grad_out, out, ranges, sources, (int)n_ranges, n_vec, row_vecs);
    });
    YITU_LAUNCH_CHECK();
    return 0;
}
