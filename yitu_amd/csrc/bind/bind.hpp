// The Python-facing side of the library: argument checks, output and scratch tensors, the
// state kept per graph and the autograd nodes, compiled against torch and linked to
// libyitu_hip.so. A layer call on a small graph is a handful of launches of a few
// microseconds each; the same work done op by op through ctypes and Python autograd nodes cost
// 25-30 us of host time per launch, several times what the kernels take (GCN layer on 3,000
// nodes, forward and backward: 100-200 us by host before, 78-88 us with this; 8 x 8 attention
// layer 320-510 -> 284 us; a two-layer relational model of 124 launches 2.6-3.1 -> 1.6 ms).
#pragma once
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include "../../../include/yitu_hip.h"

namespace yitu_bind {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
using TensorVec = std::vector<Tensor>;

constexpr int kColMask = 0xFFFFFF;
constexpr int kAllBits = 0x7FFFFFFF;
constexpr int64_t kLongRow = 64;  // rows of this many edges use the plan and its workspace
// Graphs of fewer edges and no long row have no plan: their rows fit every L2, and a call is
// its launch (at 124,000 edges in communities dealing the rows to the XCDs made 9.3 us 6.1).
constexpr int64_t kPlanMinEdges = 1 << 15;

// ---- checks ------------------------------------------------------------------------
inline void check_device(const Tensor &t) {
    TORCH_CHECK(t.is_cuda(), "expected a tensor on the GPU (HIP device), got ", t.device());
    TORCH_CHECK(t.is_contiguous(), "expected a contiguous tensor");
}
inline void check(const Tensor &t, at::ScalarType dtype, const char *name, int64_t dim = -1) {
    check_device(t);
    TORCH_CHECK(t.scalar_type() == dtype, name, " must be ", dtype, ", got ", t.scalar_type());
    TORCH_CHECK(dim < 0 || t.dim() == dim, name, " must be ", dim, "-D, got ", t.dim(), "-D");
}
inline void check_f32(const Tensor &t, const char *name, int64_t dim = -1) {
    check(t, at::kFloat, name, dim);
}
inline void check_i32(const Tensor &t, const char *name, int64_t dim = -1) {
    check(t, at::kInt, name, dim);
}
template <typename... Ts>
void same_device(const Tensor &first, const Ts &...rest) {
    const auto one = [&](const Tensor &t) {
        TORCH_CHECK(t.device() == first.device(), "tensors live on different devices: ",
                    first.device(), " vs ", t.device());
    };
    (one(rest), ...);
}

// ---- one call ----------------------------------------------------------------------
// The device made current for the launches and the caller's stream on it.
struct Call {
    c10::DeviceGuard guard;
    c10::Device device;
    void *stream;
    explicit Call(const Tensor &t)
        : guard(t.device()), device(t.device()),
          stream(c10::hip::getCurrentHIPStream(t.device().index()).stream()) {}
    Tensor empty(at::IntArrayRef size, at::ScalarType dtype = at::kFloat) const {
        return Tensor(at::detail::empty_cuda(size, dtype, device, std::nullopt));
    }
    // Scratch for one call, in the allocator's stream order; nothing where nothing is needed.
    struct Scratch {
        Tensor buffer;
        void *data_ptr() const { return buffer.defined() ? buffer.data_ptr() : nullptr; }
        size_t numel() const { return buffer.defined() ? (size_t)buffer.numel() : 0; }
    };
    Scratch scratch(size_t bytes) const {
        return bytes ? Scratch{empty({(int64_t)bytes}, at::kByte)} : Scratch{};
    }
};
inline void ok(int rc, const char *what) {
    TORCH_CHECK(rc == 0, what, " failed (code ", rc, "): ", yitu_last_error());
}

inline float *f32(const Tensor &t) { return static_cast<float *>(t.data_ptr()); }
inline float *f32(const OptTensor &t) { return t.has_value() && t->defined() ? f32(*t) : nullptr; }
inline const int32_t *i32(const Tensor &t) { return static_cast<const int32_t *>(t.data_ptr()); }
inline const void *raw(const OptTensor &t) {
    return t.has_value() && t->defined() ? t->data_ptr() : nullptr;
}
inline bool aligned16(const Tensor &t) {
    return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}
inline bool has(const OptTensor &t) { return t.has_value() && t->defined(); }

// ---- state kept per graph (graph_state.cpp) ------------------------------------------
struct RowState {  // what the row kernels want to know of a CSR
    int64_t max_degree = -1;
    OptTensor plan;
};
struct BySource {  // the transposed structure
    Tensor t_indptr, t_rows, t_perm;
    int64_t max_degree = -1;
    OptTensor plan;
};
RowState row_state(const Tensor &indptr, const Tensor &indices, int64_t n_src, int mask);
BySource by_source(const Tensor &indptr, const Tensor &indices, int64_t n_src);
BySource by_source_of(const py::handle &transposed);  // the same, read off the Python object
OptTensor by_source_values(const Tensor &values, const Tensor &indptr, const Tensor &indices,
                           int64_t n_src, bool force);
void bind_graph_state(py::module_ &m);

// ---- ops (ops.cpp) -------------------------------------------------------------------
Tensor agg(const Tensor &x, const Tensor &rp, const Tensor &ci, const OptTensor &degrees,
           const OptTensor &edge_scale, double alpha, const RowState &rows);
Tensor sgemm(const Tensor &a, const Tensor &b, bool trans_a, bool trans_b, const OptTensor &out,
             bool accumulate = false);  // accumulate: add to `out`
Tensor linear_forward(const Tensor &x, const Tensor &w, const OptTensor &bias);
TensorVec linear_forward_typed(const TensorVec &xs, const TensorVec &ws,
                               const std::vector<OptTensor> &bs,
                               const std::optional<TensorVec> &outs);
TensorVec sgemm_typed(const TensorVec &as, const TensorVec &bs, bool trans_a, bool trans_b,
                      const std::optional<TensorVec> &outs);
// The same over matrices given by address and row count (the caller has checked them):
// y_i [m_i, n] = x_i [m_i, k] . w_i^T + b_i, and dx_i [m_i, k] = g_i [m_i, n] . w_i
struct RowsView {
    std::vector<const float *> x;
    std::vector<int64_t> rows;
};
void linear_forward_at(const Call &c, const std::vector<float *> &y, const RowsView &x,
                       const std::vector<const float *> &w, const std::vector<const float *> &b,
                       int64_t n, int64_t k);
void linear_input_grad_at(const Call &c, const std::vector<float *> &dx, const RowsView &g,
                          const std::vector<const float *> &w, int64_t n, int64_t k);
void linear_weight_grad_at(const Call &c, const std::vector<float *> &dw,
                           const std::vector<float *> &db, const RowsView &g,
                           const std::vector<const float *> &x, int64_t n, int64_t k);
// dw_i = g_i^T . x_i, and db_i = column sums of g_i where want_bias[i]
void linear_weight_grad(const TensorVec &gs, const TensorVec &xs,
                        const std::vector<bool> &want_bias, TensorVec *dws,
                        std::vector<OptTensor> *dbs);
TensorVec b2gemm(const Tensor &x, const Tensor &w_a, const Tensor &w_b);
TensorVec b2gemm_backward(const Tensor &x, const Tensor &w_a, const Tensor &w_b,
                          const Tensor &grad_a, const Tensor &grad_b);
Tensor spmm_forward(const Tensor &values, const Tensor &indptr, const Tensor &indices,
                    const Tensor &features, bool bf16_out, const RowState &rows);
void spmm_backward_check(const Tensor &values, const Tensor &indptr, const Tensor &indices,
                         const Tensor &features, const Tensor &grad_out);
std::pair<OptTensor, OptTensor> spmm_backward(const Tensor &values, const Tensor &indptr,
                                              const Tensor &indices, const Tensor &features,
                                              const Tensor &grad_out, bool need_a, bool need_x,
                                              const RowState &rows, const BySource &t);
Tensor edge_dot(const Tensor &indptr, const Tensor &indices, const Tensor &dst, const Tensor &src,
                const RowState &rows);
Tensor sddmm_forward(const Tensor &indptr, const Tensor &indices, const Tensor &query,
                     const Tensor &key, const RowState &rows);
std::pair<Tensor, Tensor> sddmm_backward(const Tensor &indptr, const Tensor &indices,
                                         const Tensor &query, const Tensor &key, const Tensor &attn,
                                         const Tensor &grad_out, const RowState &rows,
                                         const std::optional<BySource> &t);
bool gat_one_pass_shape(int64_t heads, int64_t width);
bool gat_mean_shape(const Tensor &x);  // of the head-mean backward, x [n_src, H, F]
// whether the backward needs no more of the forward's softmax than its row statistics
bool gat_stats_suffice(const Tensor &x, bool head_mean);
struct GatOut {
    Tensor out;
    OptTensor attn, stats;
};
GatOut gat_forward(const Tensor &indptr, const Tensor &indices, const Tensor &query,
                   const Tensor &key, const Tensor &x, bool stats_only, const RowState &rows);
struct GatGrads {
    Tensor query, key, x;
};
GatGrads gat_backward(const Tensor &indptr, const Tensor &indices, const Tensor &query,
                      const Tensor &key, const Tensor &x, const OptTensor &attn,
                      const Tensor &grad_out, const OptTensor &out, bool head_mean,
                      const OptTensor &stats, const RowState &rows, const BySource &t);
std::pair<Tensor, OptTensor> head_dot(const Tensor &x, const Tensor &a, const OptTensor &b);
std::tuple<Tensor, Tensor, OptTensor> head_dot_backward(const Tensor &x, const Tensor &a,
                                                        const OptTensor &b, const Tensor &grad_a,
                                                        const OptTensor &grad_b,
                                                        const OptTensor &grad_x);
bool skinny_linear_shape(int64_t in_features, int64_t out_features);
// one Linear with a handful of outputs, or two over the same x (w_b given)
std::pair<Tensor, OptTensor> skinny_pair(const Tensor &x, const Tensor &w_a, const OptTensor &w_b,
                                         const OptTensor &bias_a, const OptTensor &bias_b);
struct SkinnyGrads {
    Tensor x, w_a;
    OptTensor w_b, bias_a, bias_b;
};
SkinnyGrads skinny_pair_backward(const Tensor &x, const Tensor &w_a, const OptTensor &w_b,
                                 const Tensor &grad_a, const OptTensor &grad_b,
                                 const OptTensor &grad_x,  // given: added to in place
                                 bool bias_a, bool bias_b);
Tensor column_sum(const Tensor &x);
TensorVec column_sum_typed(const TensorVec &xs);
void bind_ops(py::module_ &m);

void bind_autograd(py::module_ &m);
void bind_batched(py::module_ &m);
void bind_temporal(py::module_ &m);

}  // namespace yitu_bind
