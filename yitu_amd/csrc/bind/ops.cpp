// One function per op of graph_ext / YiTu_GNN_kernel: checks the operands, makes the outputs
// and the scratch, calls the C entry point. What an op means stands in the Python wrapper of
// the same name and at the entry point (include/yitu_hip.h).
#include "bind.hpp"

namespace yitu_bind {
namespace {

template <typename P>
std::vector<P> pointers(const TensorVec &ts) {
    std::vector<P> v;
    v.reserve(ts.size());
    for (const Tensor &t : ts) v.push_back(static_cast<P>(t.numel() ? t.data_ptr() : nullptr));
    return v;
}

// outputs of a grouped product: the caller's tensors, or new [m_i, n] ones
TensorVec outputs(const Call &c, const std::optional<TensorVec> &given,
                  const std::vector<int64_t> &ms, int64_t n, at::ScalarType dtype) {
    TensorVec outs;
    outs.reserve(ms.size());
    if (!given) {
        for (int64_t m : ms) outs.push_back(c.empty({m, n}, dtype));
        return outs;
    }
    TORCH_CHECK(given->size() == ms.size(), "as many outputs as products are needed");
    for (size_t i = 0; i < ms.size(); i++) {
        const Tensor &o = (*given)[i];
        TORCH_CHECK(o.scalar_type() == dtype && o.dim() == 2 && o.size(0) == ms[i] &&
                        o.size(1) == n && o.device() == c.device && o.is_contiguous(),
                    "out must be contiguous [", ms[i], ", ", n, "] ", dtype,
                    " on the operands' device");
        outs.push_back(o);
    }
    return outs;
}

size_t spmm_scratch(int64_t nnz, int64_t row_len, int64_t widest) {
    return widest >= kLongRow ? yitu_spmm_workspace_bytes(nnz, row_len, 1) : 0;
}

}  // namespace

Tensor agg(const Tensor &x, const Tensor &rp, const Tensor &ci, const OptTensor &degrees,
           const OptTensor &edge_scale, double alpha, const RowState &rows) {
    check_i32(rp, "row_pointers");
    check_i32(ci, "column_index");
    check_device(x);
    const bool bf16 = x.scalar_type() == at::kBFloat16;
    TORCH_CHECK(bf16 || x.scalar_type() == at::kFloat, "features must be float32 or bfloat16, got ",
                x.scalar_type());
    TORCH_CHECK(x.dim() == 2, "features must be 2-D [n_nodes, dim]");
    const int64_t n_rows = rp.numel() - 1, n_src = x.size(0), dim = x.size(1), nnz = ci.numel();
    if (has(degrees)) {
        check_f32(*degrees, "degrees");
        TORCH_CHECK(degrees->numel() >= std::max(n_rows, n_src),
                    "degrees is shorter than the number of nodes");
    }
    if (has(edge_scale)) {
        check_f32(*edge_scale, "edge_scale");
        TORCH_CHECK(edge_scale->numel() == nnz, "edge_scale must hold one value per edge");
    }
    Call c(x);
    Tensor out = c.empty({n_rows, dim});
    const size_t need =
        has(rows.plan) && rows.max_degree >= kLongRow ? yitu_spmm_workspace_bytes(nnz, dim, 1) : 0;
    const auto ws = c.scratch(need);
    ok(yitu_agg_csr(f32(out), x.data_ptr(), bf16, i32(rp), i32(ci), f32(degrees), n_rows, n_src, nnz,
                    dim, (float)alpha, rows.max_degree, raw(rows.plan), f32(edge_scale),
                    ws.data_ptr(), ws.numel(), c.stream),
       "yitu_agg_csr");
    return out;
}

Tensor edge_scale(const Tensor &ci, const Tensor &degrees) {
    check_i32(ci, "column_index");
    check_f32(degrees, "degrees");
    same_device(ci, degrees);
    Call c(ci);
    Tensor out = c.empty({ci.numel()});
    ok(yitu_edge_scale(f32(out), i32(ci), f32(degrees), ci.numel(), degrees.numel(), c.stream),
       "yitu_edge_scale");
    return out;
}

// ---- dense products ------------------------------------------------------------------
Tensor sgemm(const Tensor &a, const Tensor &b, bool trans_a, bool trans_b, const OptTensor &out,
             bool accumulate) {
    check_f32(a, "a", 2);
    check_f32(b, "b", 2);
    same_device(a, b);
    const int64_t m = a.size(trans_a ? 1 : 0), k = a.size(trans_a ? 0 : 1);
    const int64_t kb = b.size(trans_b ? 1 : 0), n = b.size(trans_b ? 0 : 1);
    TORCH_CHECK(k == kb, "inner dimensions differ: ", k, " vs ", kb);
    Call call(a);
    Tensor c;
    if (has(out)) {
        check_f32(*out, "out", 2);
        TORCH_CHECK(out->size(0) == m && out->size(1) == n && out->device() == call.device,
                    "out must be [", m, ", ", n, "] on the operands' device");
        c = *out;
    } else {
        c = call.empty({m, n});
    }
    const auto ws = call.scratch(yitu_sgemm_workspace_bytes(m, n, k, 1));
    ok(yitu_sgemm(f32(c), f32(a), f32(b), m, n, k, trans_a, trans_b, a.size(1), b.size(1), n, accumulate,
                  ws.data_ptr(), ws.numel(), call.stream),
       "yitu_sgemm");
    return c;
}

Tensor linear_forward(const Tensor &x, const Tensor &w, const OptTensor &bias) {
    check_f32(x, "x", 2);
    check_f32(w, "weight", 2);
    same_device(x, w);
    const int64_t m = x.size(0), k = x.size(1), n = w.size(0);
    if (has(bias)) {
        check_f32(*bias, "bias", 1);
        same_device(x, *bias);
    }
    TORCH_CHECK(w.size(1) == k && (!has(bias) || bias->numel() == n),
                "linear_forward: x [m, k], weight [n, k], bias [n]");
    Call c(x);
    Tensor y = c.empty({m, n});
    const auto ws = c.scratch(yitu_sgemm_workspace_bytes(m, n, k, 1));
    ok(yitu_linear_forward(f32(y), f32(x), f32(w), f32(bias), m, n, k, ws.data_ptr(), ws.numel(),
                           c.stream),
       "yitu_linear_forward");
    return y;
}

TensorVec linear_forward_typed(const TensorVec &xs, const TensorVec &ws,
                               const std::vector<OptTensor> &bs,
                               const std::optional<TensorVec> &given) {
    const size_t count = xs.size();
    TORCH_CHECK(count > 0 && ws.size() == count && bs.size() == count,
                "linear_forward_typed needs as many weights and biases as inputs");
    check_f32(ws[0], "weight", 2);
    const int64_t n = ws[0].size(0), k = ws[0].size(1);
    std::vector<int64_t> ms;
    std::vector<const float *> biases;
    for (size_t i = 0; i < count; i++) {
        check_f32(xs[i], "x", 2);
        check_f32(ws[i], "weight", 2);
        same_device(xs[0], xs[i], ws[i]);
        TORCH_CHECK(ws[i].size(0) == n && ws[i].size(1) == k && xs[i].size(1) == k,
                    "linear_forward_typed: x_i [m_i, k], weight_i [n, k]");
        if (has(bs[i])) {
            check_f32(*bs[i], "bias", 1);
            same_device(xs[0], *bs[i]);
            TORCH_CHECK(bs[i]->numel() == n, "linear_forward_typed: bias_i [n]");
        }
        ms.push_back(xs[i].size(0));
        biases.push_back(f32(bs[i]));
    }
    Call c(xs[0]);
    TensorVec outs = outputs(c, given, ms, n, at::kFloat);
    linear_forward_at(c, pointers<float *>(outs), {pointers<const float *>(xs), ms},
                      pointers<const float *>(ws), biases, n, k);
    return outs;
}

TensorVec sgemm_typed(const TensorVec &as, const TensorVec &bs, bool trans_a, bool trans_b,
                      const std::optional<TensorVec> &given) {
    const size_t count = as.size();
    TORCH_CHECK(count > 0 && bs.size() == count,
                "sgemm_typed needs as many a as b operands, at least one");
    std::vector<int64_t> ms, ks;
    bool shared = true;
    for (size_t i = 0; i < count; i++) {
        check_f32(as[i], "a", 2);
        check_f32(bs[i], "b", 2);
        same_device(as[0], as[i], bs[i]);
        ms.push_back(as[i].size(trans_a ? 1 : 0));
        ks.push_back(as[i].size(trans_a ? 0 : 1));
        const int64_t kb = bs[i].size(trans_b ? 1 : 0);
        TORCH_CHECK(kb == ks[i], "inner dimensions differ: ", ks[i], " vs ", kb);
        shared = shared && bs[i].size(trans_b ? 0 : 1) == bs[0].size(trans_b ? 0 : 1) &&
                 as[i].size(1) == as[0].size(1) && bs[i].size(1) == bs[0].size(1);
    }
    if (!shared) {  // widths differ between the types: one product at a time
        TensorVec outs;
        for (size_t i = 0; i < count; i++)
            outs.push_back(sgemm(as[i], bs[i], trans_a, trans_b,
                                 given ? OptTensor((*given)[i]) : std::nullopt));
        return outs;
    }
    const int64_t n = bs[0].size(trans_b ? 0 : 1);
    Call c(as[0]);
    TensorVec outs = outputs(c, given, ms, n, at::kFloat);
    const auto ws = c.scratch(yitu_sgemm_workspace_bytes(*std::max_element(ms.begin(), ms.end()), n,
                                                     *std::max_element(ks.begin(), ks.end()),
                                                     (int64_t)count));
    ok(yitu_sgemm_typed(pointers<float *>(outs).data(), pointers<const float *>(as).data(),
                        pointers<const float *>(bs).data(), ms.data(), ks.data(), (int64_t)count, n,
                        trans_a, trans_b, as[0].size(1), bs[0].size(1), n, 0, ws.data_ptr(),
                        ws.numel(), c.stream),
       "yitu_sgemm_typed");
    return outs;
}

void linear_weight_grad(const TensorVec &gs, const TensorVec &xs,
                        const std::vector<bool> &want_bias, TensorVec *dws,
                        std::vector<OptTensor> *dbs) {
    const int64_t count = (int64_t)gs.size(), n = gs[0].size(1), k = xs[0].size(1);
    std::vector<int64_t> rows;
    for (int64_t i = 0; i < count; i++) {
        check_f32(gs[i], "grad", 2);
        check_f32(xs[i], "x", 2);
        same_device(gs[0], gs[i], xs[i]);
        TORCH_CHECK(gs[i].size(1) == n && xs[i].size(1) == k && gs[i].size(0) == xs[i].size(0),
                    "linear_weight_grad: grad_i [m_i, ", n, "], x_i [m_i, ", k, "]");
        rows.push_back(gs[i].size(0));
    }
    Call c(gs[0]);
    *dws = outputs(c, std::nullopt, std::vector<int64_t>(count, n), k, at::kFloat);
    dbs->assign(count, std::nullopt);
    std::vector<float *> db(count, nullptr);
    for (int64_t i = 0; i < count; i++)
        if (want_bias[i]) {
            (*dbs)[i] = c.empty({n});
            db[i] = f32((*dbs)[i]);
        }
    linear_weight_grad_at(c, pointers<float *>(*dws), db, {pointers<const float *>(gs), rows},
                          pointers<const float *>(xs), n, k);
}

void linear_forward_at(const Call &c, const std::vector<float *> &y, const RowsView &x,
                       const std::vector<const float *> &w, const std::vector<const float *> &b,
                       int64_t n, int64_t k) {
    const int64_t count = (int64_t)y.size(), most = *std::max_element(x.rows.begin(), x.rows.end());
    const auto ws = c.scratch(yitu_sgemm_workspace_bytes(most, n, k, count));
    ok(yitu_linear_forward_typed(y.data(), x.x.data(), w.data(), b.data(), x.rows.data(), count, n, k,
                                 ws.data_ptr(), ws.numel(), c.stream),
       "yitu_linear_forward_typed");
}

void linear_input_grad_at(const Call &c, const std::vector<float *> &dx, const RowsView &g,
                          const std::vector<const float *> &w, int64_t n, int64_t k) {
    const int64_t count = (int64_t)dx.size(), most = *std::max_element(g.rows.begin(), g.rows.end());
    const std::vector<int64_t> ks(count, n);
    const auto ws = c.scratch(yitu_sgemm_workspace_bytes(most, k, n, count));
    ok(yitu_sgemm_typed(dx.data(), g.x.data(), w.data(), g.rows.data(), ks.data(), count, k, 0, 0, n,
                        k, k, 0, ws.data_ptr(), ws.numel(), c.stream),
       "yitu_sgemm_typed");
}

void linear_weight_grad_at(const Call &c, const std::vector<float *> &dw,
                           const std::vector<float *> &db, const RowsView &g,
                           const std::vector<const float *> &x, int64_t n, int64_t k) {
    const int64_t count = (int64_t)dw.size(), most = *std::max_element(g.rows.begin(), g.rows.end());
    const auto ws = c.scratch(yitu_linear_weight_grad_workspace_bytes(most, n, k, count));
    ok(yitu_linear_weight_grad_typed(dw.data(), db.data(), g.x.data(), x.data(), g.rows.data(), count,
                                     n, k, ws.data_ptr(), ws.numel(), c.stream),
       "yitu_linear_weight_grad_typed");
}

Tensor gemm_bf16(const Tensor &a, const Tensor &b, bool trans_b, at::ScalarType dtype,
                 const OptTensor &out) {
    check(a, at::kBFloat16, "a", 2);
    check(b, at::kBFloat16, "b", 2);
    same_device(a, b);
    const int64_t m = a.size(0), k = a.size(1), n = b.size(trans_b ? 0 : 1);
    TORCH_CHECK(b.size(trans_b ? 1 : 0) == k, "inner dimensions differ: ", k, " vs ",
                b.size(trans_b ? 1 : 0));
    if (has(out)) dtype = out->scalar_type();
    TORCH_CHECK(dtype == at::kFloat || dtype == at::kBFloat16,
                "out_dtype must be float32 or bfloat16");
    Call call(a);
    Tensor c = outputs(call, has(out) ? std::optional<TensorVec>(TensorVec{*out}) : std::nullopt,
                       {m}, n, dtype)[0];
    const auto ws = call.scratch(yitu_gemm_bf16_workspace_bytes(n, k, trans_b));
    ok(yitu_gemm_bf16(c.data_ptr(), dtype == at::kBFloat16, a.data_ptr(), b.data_ptr(), m, n, k,
                      trans_b, k, b.size(1), n, ws.data_ptr(), ws.numel(), call.stream),
       "yitu_gemm_bf16");
    return c;
}

TensorVec gemm_bf16_typed(const TensorVec &as, const TensorVec &bs, bool trans_b,
                          at::ScalarType dtype, const std::optional<TensorVec> &given) {
    const size_t count = as.size();
    TORCH_CHECK(count > 0 && bs.size() == count,
                "gemm_bf16_typed needs as many a as b operands, at least one");
    check(as[0], at::kBFloat16, "a", 2);
    check(bs[0], at::kBFloat16, "b", 2);
    const int64_t k = as[0].size(1), n = bs[0].size(trans_b ? 0 : 1);
    std::vector<int64_t> ms;
    for (size_t i = 0; i < count; i++) {
        check(as[i], at::kBFloat16, "a", 2);
        check(bs[i], at::kBFloat16, "b", 2);
        same_device(as[0], as[i], bs[i]);
        TORCH_CHECK(as[i].size(1) == k && bs[i].size(trans_b ? 1 : 0) == k &&
                        bs[i].size(trans_b ? 0 : 1) == n,
                    "gemm_bf16_typed: every pair must be [m_i, ", k, "] x ",
                    trans_b ? "[n, k]" : "[k, n]", " with k = ", k, ", n = ", n);
        ms.push_back(as[i].size(0));
    }
    if (given && !given->empty()) dtype = (*given)[0].scalar_type();
    TORCH_CHECK(dtype == at::kFloat || dtype == at::kBFloat16,
                "out_dtype must be float32 or bfloat16");
    Call c(as[0]);
    TensorVec outs = outputs(c, given, ms, n, dtype);
    const auto ws = c.scratch(yitu_gemm_bf16_typed_workspace_bytes((int64_t)count, n, k, trans_b));
    ok(yitu_gemm_bf16_typed(pointers<void *>(outs).data(), dtype == at::kBFloat16,
                            pointers<const void *>(as).data(), pointers<const void *>(bs).data(),
                            ms.data(), (int64_t)count, n, k, trans_b, k, bs[0].size(1), n,
                            ws.data_ptr(), ws.numel(), c.stream),
       "yitu_gemm_bf16_typed");
    return outs;
}

TensorVec gemm_bf16_tn_typed(const TensorVec &as, const TensorVec &bs,
                             const std::optional<TensorVec> &given, bool accumulate) {
    const size_t count = as.size();
    TORCH_CHECK(count > 0 && bs.size() == count,
                "gemm_bf16_tn_typed needs as many a as b operands, at least one");
    for (const TensorVec *v : {&as, &bs})
        for (const Tensor &t : *v)
            TORCH_CHECK(t.scalar_type() == at::kBFloat16 && t.dim() == 2 && t.stride(1) == 1 &&
                            t.is_cuda(),
                        "operands must be 2-D bf16 GPU tensors with contiguous rows");
    const int64_t ki = as[0].size(1), no = bs[0].size(1);
    const int64_t lda = as[0].stride(0), ldb = bs[0].stride(0);
    std::vector<int64_t> ms;
    for (size_t i = 0; i < count; i++) {
        const Tensor &a = as[i], &b = bs[i];
        TORCH_CHECK(a.device() == as[0].device() && b.device() == as[0].device() &&
                        a.size(0) == b.size(0) && a.size(1) == ki && b.size(1) == no &&
                        (a.size(0) <= 1 || a.stride(0) == lda) &&
                        (b.size(0) <= 1 || b.stride(0) == ldb),
                    "gemm_bf16_tn_typed: every pair must be [m_i, ", ki, "], [m_i, ", no,
                    "] with common row strides on one device");
        ms.push_back(a.size(0));
    }
    TORCH_CHECK(!accumulate || given, "accumulate needs outputs to add to");
    Call c(as[0]);
    TensorVec outs = outputs(c, given, std::vector<int64_t>(count, ki), no, at::kFloat);
    const auto ws = c.scratch(yitu_gemm_bf16_tn_typed_workspace_bytes(ms.data(), (int64_t)count, ki, no));
    ok(yitu_gemm_bf16_tn_typed(pointers<float *>(outs).data(), pointers<const void *>(as).data(),
                               pointers<const void *>(bs).data(), ms.data(), (int64_t)count, ki, no,
                               std::max(lda, ki), std::max(ldb, no), no, accumulate, ws.data_ptr(),
                               ws.numel(), c.stream),
       "yitu_gemm_bf16_tn_typed");
    return outs;
}

Tensor gemm_bf16_tn(const Tensor &a, const Tensor &b, const OptTensor &out, bool accumulate) {
    for (const Tensor *t : {&a, &b})
        TORCH_CHECK(t->scalar_type() == at::kBFloat16 && t->dim() == 2 && t->stride(1) == 1 &&
                        t->is_cuda(),
                    "a and b must be 2-D bf16 GPU tensors with contiguous rows");
    TORCH_CHECK(a.device() == b.device() && a.size(0) == b.size(0),
                "a and b must have the same number of rows on one device");
    TORCH_CHECK(!accumulate || has(out), "accumulate needs an output to add to");
    const int64_t m = a.size(0), ki = a.size(1), no = b.size(1);
    Call c(a);
    Tensor o = outputs(c, has(out) ? std::optional<TensorVec>(TensorVec{*out}) : std::nullopt, {ki},
                       no, at::kFloat)[0];
    const auto ws = c.scratch(yitu_gemm_bf16_tn_workspace_bytes(m, ki, no));
    ok(yitu_gemm_bf16_tn(f32(o), a.data_ptr(), b.data_ptr(), m, ki, no, a.stride(0), b.stride(0), no,
                         accumulate, ws.data_ptr(), ws.numel(), c.stream),
       "yitu_gemm_bf16_tn");
    return o;
}

TensorVec b2gemm(const Tensor &x, const Tensor &w_a, const Tensor &w_b) {
    check_f32(x, "x", 2);
    check_f32(w_a, "w_a", 2);
    check_f32(w_b, "w_b", 2);
    same_device(x, w_a, w_b);
    TORCH_CHECK(w_a.sizes() == w_b.sizes() && w_a.size(1) == x.size(1),
                "w_a and w_b must both be [m, k] with k = x.size(1)");
    const int64_t n = x.size(0), k = x.size(1), m = w_a.size(0);
    Call c(x);
    Tensor y_a = c.empty({n, m}), y_b = c.empty({n, m});
    ok(yitu_b2gemm(f32(y_a), f32(y_b), f32(x), f32(w_a), f32(w_b), n, k, m, c.stream),
       "yitu_b2gemm");
    return {y_a, y_b};
}

TensorVec b2gemm_backward(const Tensor &x, const Tensor &w_a, const Tensor &w_b,
                          const Tensor &grad_a, const Tensor &grad_b) {
    check_f32(x, "x", 2);
    check_f32(w_a, "w_a", 2);
    check_f32(w_b, "w_b", 2);
    check_f32(grad_a, "grad_a", 2);
    check_f32(grad_b, "grad_b", 2);
    same_device(x, w_a, w_b, grad_a, grad_b);
    TORCH_CHECK(grad_a.sizes() == grad_b.sizes() && w_a.sizes() == w_b.sizes(),
                "the two halves of the bundle must have equal shapes");
    const int64_t n = x.size(0), k = x.size(1), m = w_a.size(0);
    TORCH_CHECK(grad_a.size(0) == n && grad_a.size(1) == m, "grad_* must be [n, m]");
    Call c(x);
    Tensor dx = c.empty({n, k}), dw_a = c.empty({m, k}), dw_b = c.empty({m, k});
    const auto ws = c.scratch(yitu_sgemm_workspace_bytes(m, k, n, 2));
    ok(yitu_b2gemm_backward(f32(dx), f32(dw_a), f32(dw_b), f32(x), f32(w_a), f32(w_b), f32(grad_a),
                            f32(grad_b), n, k, m, ws.data_ptr(), ws.numel(), c.stream),
       "yitu_b2gemm_backward");
    return {dx, dw_a, dw_b};
}

// ---- SpMM ----------------------------------------------------------------------------
Tensor spmm_forward(const Tensor &values, const Tensor &indptr, const Tensor &indices,
                    const Tensor &features, bool bf16_out, const RowState &rows) {
    check_f32(values, "values", 2);
    check_i32(indptr, "indptr", 1);
    check_i32(indices, "indices", 1);
    const bool bf16 = features.scalar_type() == at::kBFloat16;
    check(features, bf16 ? at::kBFloat16 : at::kFloat, "features", 3);
    same_device(values, indptr, indices, features);
    const int64_t n_dst = indptr.numel() - 1, nnz = indices.numel();
    const int64_t n_src = features.size(0), h = features.size(1), f = features.size(2);
    TORCH_CHECK(values.size(0) == nnz && values.size(1) == h, "values must be [n_edges, n_heads]");
    TORCH_CHECK(!bf16_out || (bf16 && f % 8 == 0),
                "out_dtype is float32, or bfloat16 for bf16 features whose head width is a "
                "multiple of 8");
    Call c(features);
    Tensor out = c.empty({n_dst, h, f}, bf16_out ? at::kBFloat16 : at::kFloat);
    const auto ws = c.scratch(has(rows.plan) ? spmm_scratch(nnz, h * f, rows.max_degree) : 0);
    int rc;
    if (bf16_out)
        rc = yitu_spmm_forward_bf16_rows(out.data_ptr(), f32(values), i32(indptr), i32(indices),
                                         features.data_ptr(), n_dst, n_src, nnz, h, f,
                                         rows.max_degree, raw(rows.plan), ws.data_ptr(), ws.numel(),
                                         c.stream);
    else if (bf16)
        rc = yitu_spmm_forward_bf16(f32(out), f32(values), i32(indptr), i32(indices),
                                    features.data_ptr(), n_dst, n_src, nnz, h, f, rows.max_degree,
                                    raw(rows.plan), ws.data_ptr(), ws.numel(), c.stream);
    else
        rc = yitu_spmm_forward(f32(out), f32(values), i32(indptr), i32(indices), f32(features),
                               n_dst, n_src, nnz, h, f, rows.max_degree, raw(rows.plan),
                               ws.data_ptr(), ws.numel(), c.stream);
    ok(rc, "yitu_spmm_forward");
    return out;
}

// What every form of the backward asks of its operands, before any of them is chosen: each
// kernel reads grad_out by destination and values by edge. Rows of grad_out in bf16 take bf16
// features too (they are not read).
void spmm_backward_check(const Tensor &values, const Tensor &indptr, const Tensor &indices,
                         const Tensor &features, const Tensor &grad_out) {
    check_f32(values, "values", 2);
    check_i32(indptr, "indptr", 1);
    check_i32(indices, "indices", 1);
    const bool bf16 = grad_out.scalar_type() == at::kBFloat16;
    check(features, bf16 && features.scalar_type() == at::kBFloat16 ? at::kBFloat16 : at::kFloat,
          "features", 3);
    check(grad_out, bf16 ? at::kBFloat16 : at::kFloat, "grad_out", 3);
    same_device(values, indptr, indices, features, grad_out);
    TORCH_CHECK(grad_out.size(0) == indptr.numel() - 1 && grad_out.size(1) == features.size(1) &&
                    grad_out.size(2) == features.size(2),
                "grad_out must be [n_dst, n_heads, n_features]");
    TORCH_CHECK(values.size(0) >= indices.numel() && values.size(1) == features.size(1),
                "values must be [n_edges, n_heads]");
}

std::pair<OptTensor, OptTensor> spmm_backward(const Tensor &values, const Tensor &indptr,
                                              const Tensor &indices, const Tensor &features,
                                              const Tensor &grad_out, bool need_a, bool need_x,
                                              const RowState &rows, const BySource &t) {
    check_f32(grad_out, "grad_out", 3);
    spmm_backward_check(values, indptr, indices, features, grad_out);
    const int64_t n_dst = indptr.numel() - 1, nnz = indices.numel();
    const int64_t n_src = features.size(0), h = features.size(1), f = features.size(2);
    Call c(features);
    OptTensor grad_a, grad_x;
    if (need_a) grad_a = c.empty(values.sizes());
    if (need_x) grad_x = c.empty(features.sizes());
    const auto ws = c.scratch(spmm_scratch(nnz, h * f, std::max(rows.max_degree, t.max_degree)));
    ok(yitu_spmm_backward(f32(grad_a), f32(grad_x), f32(values), i32(indptr), i32(indices),
                          f32(features), f32(grad_out), i32(t.t_indptr), i32(t.t_rows),
                          i32(t.t_perm), n_dst, n_src, nnz, h, f, rows.max_degree, t.max_degree,
                          raw(rows.plan), raw(t.plan), ws.data_ptr(), ws.numel(), c.stream),
       "yitu_spmm_backward");
    return {grad_a, grad_x};
}

Tensor edge_dot(const Tensor &indptr, const Tensor &indices, const Tensor &dst, const Tensor &src,
                const RowState &rows) {
    check_i32(indptr, "indptr", 1);
    check_i32(indices, "indices", 1);
    check_f32(dst, "dst_feat", 3);
    check_f32(src, "src_feat", 3);
    same_device(indptr, indices, dst, src);
    const int64_t n_dst = indptr.numel() - 1, nnz = indices.numel();
    const int64_t n_src = src.size(0), h = src.size(1), f = src.size(2);
    TORCH_CHECK(dst.size(0) == n_dst && dst.size(1) == h && dst.size(2) == f,
                "dst_feat must be [n_dst, H, F] matching src_feat's H and F");
    Call c(src);
    Tensor out = c.empty({nnz, h});
    const auto ws = c.scratch(0);
    ok(yitu_spmm_backward(f32(out), nullptr, nullptr, i32(indptr), i32(indices), f32(src), f32(dst),
                          nullptr, nullptr, nullptr, n_dst, n_src, nnz, h, f, rows.max_degree, -1,
                          raw(rows.plan), nullptr, ws.data_ptr(), ws.numel(), c.stream),
       "yitu_spmm_backward");
    return out;
}

// ---- SDDMM + LeakyReLU + edge softmax --------------------------------------------------
namespace {
void sddmm_check(const Tensor &indptr, const Tensor &indices, const Tensor &query,
                 const Tensor &key) {
    check_i32(indptr, "indptr", 1);
    check_i32(indices, "indices", 1);
    check_f32(query, "query", 3);
    check_f32(key, "key", 2);
    same_device(indptr, indices, query, key);
    TORCH_CHECK(query.size(2) == key.size(1), "query and key disagree on the number of heads");
    TORCH_CHECK(query.size(1) == indptr.numel() - 1,
                "query.size(1) must equal the number of destination rows");
    TORCH_CHECK(query.size(0) <= 16, "at most 16 query blocks (the block tag is 4 bits wide)");
}
}  // namespace

Tensor sddmm_forward(const Tensor &indptr, const Tensor &indices, const Tensor &query,
                     const Tensor &key, const RowState &rows) {
    sddmm_check(indptr, indices, query, key);
    const int64_t n_dst = indptr.numel() - 1, nnz = indices.numel();
    const int64_t n_src = key.size(0), h = key.size(1), n_bid = query.size(0);
    Call c(key);
    Tensor attn = c.empty({nnz, h});
    const auto ws = c.scratch(rows.max_degree >= kLongRow
                              ? yitu_sddmm_workspace_bytes(n_dst, nnz, h, n_bid, 1)
                              : 0);
    ok(yitu_sddmm_forward(f32(attn), i32(indptr), i32(indices), f32(query), f32(key), n_dst, n_src,
                          nnz, h, n_bid, rows.max_degree, raw(rows.plan), ws.data_ptr(), ws.numel(),
                          c.stream),
       "yitu_sddmm_forward");
    return attn;
}

std::pair<Tensor, Tensor> sddmm_backward(const Tensor &indptr, const Tensor &indices,
                                         const Tensor &query, const Tensor &key, const Tensor &attn,
                                         const Tensor &grad_out, const RowState &rows,
                                         const std::optional<BySource> &t) {
    sddmm_check(indptr, indices, query, key);
    check_f32(attn, "attn_values", 2);
    check_f32(grad_out, "grad_out", 2);
    same_device(key, attn, grad_out);
    const int64_t n_dst = indptr.numel() - 1, nnz = indices.numel();
    const int64_t n_src = key.size(0), h = key.size(1), n_bid = query.size(0);
    TORCH_CHECK(attn.size(0) == nnz && attn.size(1) == h && grad_out.sizes() == attn.sizes(),
                "attn_values and grad_out must be [n_edges, n_heads]");
    Call c(key);
    Tensor grad_q = c.empty(query.sizes()), grad_k = c.empty(key.sizes());
    OptTensor grad_edge;
    if (t) grad_edge = c.empty({nnz, h});
    const bool wide = rows.max_degree >= kLongRow || (t && t->max_degree >= kLongRow);
    const auto ws = c.scratch(wide ? yitu_sddmm_workspace_bytes(n_dst, nnz, h, n_bid, 1) : 0);
    ok(yitu_sddmm_backward(f32(grad_q), f32(grad_k), f32(grad_edge), i32(indptr), i32(indices),
                           f32(query), f32(key), f32(attn), f32(grad_out),
                           t ? i32(t->t_indptr) : nullptr, t ? i32(t->t_perm) : nullptr, n_dst, n_src,
                           nnz, h, n_bid, rows.max_degree, t ? t->max_degree : -1, raw(rows.plan),
                           t ? raw(t->plan) : nullptr, ws.data_ptr(), ws.numel(), c.stream),
       "yitu_sddmm_backward");
    return {grad_q, grad_k};
}

// ---- fused GAT -------------------------------------------------------------------------
// Rows whose backward is the one by-source pass (and needs only the row statistics).
bool gat_one_pass_shape(int64_t heads, int64_t width) {
    const int64_t row = heads * width, lph = width / 4;
    return width % 4 == 0 && lph >= 8 && lph <= 64 && (lph & (lph - 1)) == 0 &&
           (row == 256 || row == 512 || row == 1024);
}

// Features whose backward takes the gradient of the mean over heads as it is.
bool gat_mean_shape(const Tensor &x) {
    const int64_t heads = x.size(1), width = x.size(2);
    return (heads == 1 || heads == 2 || heads == 4 || heads == 8) && width >= 4 && width <= 256 &&
           width % 4 == 0 && x.size(0) <= (1 << 24) && aligned16(x);
}

bool gat_stats_suffice(const Tensor &x, bool head_mean) {
    return gat_one_pass_shape(x.size(1), x.size(2)) || (head_mean && gat_mean_shape(x));
}

GatOut gat_forward(const Tensor &indptr, const Tensor &indices, const Tensor &query,
                   const Tensor &key, const Tensor &x, bool stats_only, const RowState &rows) {
    check_i32(indptr, "indptr", 1);
    check_i32(indices, "indices", 1);
    check_f32(query, "query", 2);
    check_f32(key, "key", 2);
    check_f32(x, "features", 3);
    same_device(indptr, indices, query, key, x);
    const int64_t n_dst = indptr.numel() - 1, nnz = indices.numel();
    const int64_t n_src = x.size(0), h = x.size(1), f = x.size(2);
    TORCH_CHECK(query.size(0) == n_dst && query.size(1) == h && key.size(0) == n_src &&
                    key.size(1) == h,
                "query must be [n_dst, H] and key [n_src, H]");
    TORCH_CHECK(!stats_only || gat_one_pass_shape(h, f) || gat_mean_shape(x),
                "stats_only needs a one-pass shape (see gat_one_pass_shape)");
    Call c(x);
    GatOut o;
    o.out = c.empty({n_dst, h, f});
    if (stats_only) o.stats = c.empty({n_dst, h, 2});
    else o.attn = c.empty({nnz, h});
    const auto ws = c.scratch(
        rows.max_degree >= kLongRow ? yitu_gat_workspace_bytes(n_dst, nnz, h, f, 1) : 0);
    ok(yitu_gat_forward(f32(o.out), f32(o.attn), f32(o.stats), i32(indptr), i32(indices), f32(query),
                        f32(key), f32(x), n_dst, n_src, nnz, h, f, rows.max_degree, raw(rows.plan),
                        ws.data_ptr(), ws.numel(), c.stream),
       "yitu_gat_forward");
    return o;
}

GatGrads gat_backward(const Tensor &indptr, const Tensor &indices, const Tensor &query,
                      const Tensor &key, const Tensor &x, const OptTensor &attn,
                      const Tensor &grad_out_, const OptTensor &out, bool head_mean,
                      const OptTensor &stats, const RowState &rows, const BySource &t) {
    TORCH_CHECK(has(attn) || (has(stats) && has(out)),
                "without attn the backward needs stats and out");
    if (has(attn)) check_f32(*attn, "attn", 2);
    if (has(stats)) check_f32(*stats, "stats", 3);
    check_device(grad_out_);
    check_f32(x, "features", 3);
    check_f32(query, "query", 2);
    check_f32(key, "key", 2);
    same_device(indptr, indices, query, key, x, grad_out_);
    const int64_t n_dst = indptr.numel() - 1, nnz = indices.numel();
    const int64_t n_src = x.size(0), h = x.size(1), f = x.size(2);
    Tensor grad_out = grad_out_;
    if (head_mean) {
        check_f32(grad_out, "grad_out", 2);
        TORCH_CHECK(grad_out.size(0) == n_dst && grad_out.size(1) == f,
                    "a head-mean grad_out must be [n_dst, n_features]");
        if (!aligned16(grad_out)) grad_out = grad_out.clone();
        if (!((gat_one_pass_shape(h, f) || (gat_mean_shape(x) && has(out))) && n_dst > 0 && nnz > 0)) {
            // shapes outside the head-mean kernels: spell the gradient out per head
            grad_out = (grad_out / (double)h).unsqueeze(1).expand({n_dst, h, f}).contiguous();
            head_mean = false;
        }
    }
    if (!head_mean) check_f32(grad_out, "grad_out", 3);
    if (has(out)) {
        check_f32(*out, "out", 3);
        TORCH_CHECK(out->size(0) == n_dst && out->size(1) == h && out->size(2) == f,
                    "out must be [n_dst, n_heads, n_features]");
    }
    Call c(x);
    GatGrads g{c.empty(query.sizes()), c.empty(key.sizes()), c.empty(x.sizes())};
    Tensor s1 = c.empty({nnz, h});
    Tensor s2 = has(attn) ? c.empty({nnz, h}) : s1;  // unused by the one-pass path
    const bool wide = std::max(rows.max_degree, t.max_degree) >= kLongRow || has(out);
    const auto ws =
        c.scratch(wide ? yitu_gat_workspace_bytes(std::max(n_dst, n_src), nnz, h, f, 1) : 0);
    ok(yitu_gat_backward(f32(g.query), f32(g.key), f32(g.x), f32(s1), f32(s2), i32(indptr),
                         i32(indices), f32(query), f32(key), f32(x), f32(attn), f32(stats), f32(out),
                         f32(grad_out), i32(t.t_indptr), i32(t.t_rows), i32(t.t_perm), n_dst, n_src,
                         nnz, h, f, rows.max_degree, t.max_degree, raw(rows.plan), raw(t.plan),
                         head_mean, ws.data_ptr(), ws.numel(), c.stream),
       "yitu_gat_backward");
    return g;
}

// ---- projections -----------------------------------------------------------------------
std::pair<Tensor, OptTensor> head_dot(const Tensor &x, const Tensor &a, const OptTensor &b) {
    check_f32(x, "x", 3);
    check_f32(a, "vec_a", 2);
    if (has(b)) check_f32(*b, "vec_b", 2);
    same_device(x, a);
    const int64_t n = x.size(0), h = x.size(1), f = x.size(2);
    TORCH_CHECK(a.size(0) == h && a.size(1) == f && (!has(b) || b->sizes() == a.sizes()),
                "attention vectors must be [n_heads, n_features]");
    Call c(x);
    Tensor out_a = c.empty({n, h});
    OptTensor out_b;
    if (has(b)) out_b = c.empty({n, h});
    ok(yitu_head_dot(f32(out_a), f32(out_b), f32(x), f32(a), f32(b), n, h, f, c.stream),
       "yitu_head_dot");
    return {out_a, out_b};
}

std::tuple<Tensor, Tensor, OptTensor> head_dot_backward(const Tensor &x, const Tensor &a,
                                                        const OptTensor &b, const Tensor &grad_a,
                                                        const OptTensor &grad_b,
                                                        const OptTensor &grad_x) {
    check_f32(x, "x", 3);
    check_f32(a, "vec_a", 2);
    check_f32(grad_a, "grad_a", 2);
    same_device(x, a, grad_a);
    const int64_t n = x.size(0), h = x.size(1), f = x.size(2);
    Call c(x);
    Tensor gx;
    if (has(grad_x)) {
        check_f32(*grad_x, "grad_x", 3);
        TORCH_CHECK(grad_x->sizes() == x.sizes(), "grad_x must have the shape of x");
        gx = *grad_x;
    } else {
        gx = c.empty(x.sizes());
    }
    Tensor gva = c.empty(a.sizes());
    OptTensor gvb;
    if (has(b)) gvb = c.empty(b->sizes());
    const auto ws = c.scratch(yitu_head_dot_workspace_bytes(n, h, f));
    ok(yitu_head_dot_backward(f32(gx), has(grad_x), f32(gva), f32(gvb), f32(x), f32(a), f32(b),
                              f32(grad_a), f32(grad_b), n, h, f, ws.data_ptr(), ws.numel(), c.stream),
       "yitu_head_dot_backward");
    return {gx, gva, gvb};
}

bool skinny_linear_shape(int64_t in_features, int64_t out_features) {
    const int64_t tiles = in_features <= 256 ? 1 : (in_features <= 512 ? 2 : 4);
    return in_features % 4 == 0 && in_features > 0 && in_features <= 1024 && out_features > 0 &&
           out_features <= 16 && out_features * tiles <= 16;
}

std::pair<Tensor, OptTensor> skinny_pair(const Tensor &x, const Tensor &w_a, const OptTensor &w_b,
                                         const OptTensor &bias_a, const OptTensor &bias_b) {
    check_f32(x, "x", 2);
    check_f32(w_a, "weight", 2);
    same_device(x, w_a);
    const int64_t n = x.size(0), k = x.size(1), ja = w_a.size(0), jb = has(w_b) ? w_b->size(0) : 0;
    if (has(w_b)) {
        check_f32(*w_b, "weight", 2);
        same_device(x, *w_b);
    }
    if (has(bias_a)) check_f32(*bias_a, "bias", 1);
    if (has(bias_b)) check_f32(*bias_b, "bias", 1);
    TORCH_CHECK(w_a.size(1) == k && (!has(w_b) || w_b->size(1) == k) &&
                    (!has(bias_a) || bias_a->numel() == ja) && (!has(bias_b) || bias_b->numel() == jb),
                "weight must be [out, in] and bias [out]");
    Call c(x);
    Tensor y_a = c.empty({n, ja});
    OptTensor y_b;
    if (jb) y_b = c.empty({n, jb});
    ok(yitu_skinny_pair(f32(y_a), f32(y_b), f32(x), f32(w_a), f32(w_b), f32(bias_a), f32(bias_b), n, k,
                        ja, jb, c.stream),
       "yitu_skinny_pair");
    return {y_a, y_b};
}

SkinnyGrads skinny_pair_backward(const Tensor &x, const Tensor &w_a, const OptTensor &w_b,
                                 const Tensor &grad_a, const OptTensor &grad_b,
                                 const OptTensor &grad_x, bool bias_a, bool bias_b) {
    check_f32(x, "x", 2);
    check_f32(w_a, "weight", 2);
    check_f32(grad_a, "grad_y", 2);
    same_device(x, w_a, grad_a);
    const int64_t n = x.size(0), k = x.size(1), ja = w_a.size(0), jb = has(w_b) ? w_b->size(0) : 0;
    TORCH_CHECK(w_a.size(1) == k && grad_a.size(0) == n && grad_a.size(1) == ja,
                "weight must be [out, in] and grad_y [n, out]");
    if (jb) {
        check_f32(*w_b, "weight", 2);
        check_f32(*grad_b, "grad_y", 2);
        same_device(x, *w_b, *grad_b);
        TORCH_CHECK(w_b->size(1) == k && grad_b->size(0) == n && grad_b->size(1) == jb,
                    "weight must be [out, in] and grad_y [n, out]");
    }
    if (has(grad_x)) {
        check_f32(*grad_x, "grad_x", 2);
        TORCH_CHECK(grad_x->sizes() == x.sizes(), "grad_x must have the shape of x");
    }
    Call c(x);
    SkinnyGrads g{has(grad_x) ? *grad_x : c.empty({n, k}), c.empty({ja, k})};
    if (jb) g.w_b = c.empty({jb, k});
    if (bias_a) g.bias_a = c.empty({ja});
    if (jb && bias_b) g.bias_b = c.empty({jb});
    const auto ws = c.scratch(yitu_skinny_linear_workspace_bytes(n, k, ja + jb));
    ok(yitu_skinny_pair_backward(f32(g.x), has(grad_x), f32(g.w_a), f32(g.w_b), f32(g.bias_a),
                                 f32(g.bias_b), f32(x), f32(w_a), f32(w_b), f32(grad_a), f32(grad_b),
                                 n, k, ja, jb, ws.data_ptr(), ws.numel(), c.stream),
       "yitu_skinny_pair_backward");
    return g;
}

Tensor column_sum(const Tensor &x) {
    check_f32(x, "x", 2);
    const int64_t m = x.size(0), n = x.size(1);
    Call c(x);
    Tensor out = c.empty({n});
    const auto ws = c.scratch(yitu_column_sum_workspace_bytes(m, n));
    ok(yitu_column_sum(f32(out), f32(x), m, n, ws.data_ptr(), ws.numel(), c.stream),
       "yitu_column_sum");
    return out;
}

constexpr int64_t kColumnSumTypedMaxRows = 4096;  // taller matrices take the two-stage form

TensorVec column_sum_typed(const TensorVec &xs) {
    if (xs.empty()) return {};
    const int64_t n = xs[0].size(1);
    const int64_t ld = xs[0].size(0) > 1 ? xs[0].stride(0) : n;
    bool is_short = ld >= n;
    std::vector<int64_t> ms;
    for (const Tensor &x : xs) {
        TORCH_CHECK(x.scalar_type() == at::kFloat && x.dim() == 2 && x.is_cuda() &&
                        x.size(1) == n && (n <= 1 || x.stride(1) == 1),
                    "column_sum_typed takes 2-D fp32 GPU tensors of one width");
        ms.push_back(x.size(0));
        is_short = is_short && x.size(0) <= kColumnSumTypedMaxRows &&
                   (x.size(0) <= 1 || x.stride(0) == ld);
    }
    TensorVec outs;
    outs.reserve(xs.size());
    if (!is_short) {
        for (const Tensor &x : xs) outs.push_back(column_sum(x.contiguous()));
        return outs;
    }
    Call c(xs[0]);
    Tensor out = c.empty({(int64_t)xs.size(), n});
    outs = out.unbind(0);
    ok(yitu_column_sum_typed(pointers<float *>(outs).data(), pointers<const float *>(xs).data(),
                             ms.data(), (int64_t)xs.size(), n, ld, c.stream),
       "yitu_column_sum_typed");
    return outs;
}

// ---- graph preparation -----------------------------------------------------------------
namespace {
// indptr, indices (as many as edges went in), {distinct edges or -1, longest row}
std::tuple<Tensor, Tensor, Tensor> coo_to_csr(const Tensor &rows, const Tensor &cols, int64_t n_rows,
                                              int64_t n_cols) {
    const at::ScalarType ids = rows.scalar_type();
    TORCH_CHECK(ids == at::kInt || ids == at::kLong, "ids must be int32 or int64");
    check(rows, ids, "rows", 1);
    check(cols, ids, "cols", 1);
    same_device(rows, cols);
    const int64_t n_edges = rows.numel();
    TORCH_CHECK(cols.numel() == n_edges, "rows and cols must be equally long");
    Call c(rows);
    Tensor indptr = c.empty({n_rows + 1}, at::kInt);
    Tensor indices = c.empty({std::max<int64_t>(n_edges, 1)}, at::kInt);
    Tensor info = c.empty({2}, at::kLong);
    const auto ws = c.scratch(yitu_coo_to_csr_workspace_bytes(n_edges, n_rows));
    ok(yitu_coo_to_csr_ids(static_cast<int32_t *>(indptr.data_ptr()),
                           static_cast<int32_t *>(indices.data_ptr()),
                           static_cast<long long *>(info.data_ptr()), rows.data_ptr(),
                           cols.data_ptr(), ids == at::kInt ? 4 : 8, n_edges, n_rows, n_cols,
                           ws.data_ptr(), ws.numel(), c.stream),
       "yitu_coo_to_csr_ids");
    return {indptr, indices, info};
}

Tensor longest_row(const Tensor &indptr) {
    check_i32(indptr, "indptr", 1);
    Call c(indptr);
    Tensor out = c.empty({1}, at::kLong);
    ok(yitu_longest_row(static_cast<long long *>(out.data_ptr()), i32(indptr), indptr.numel() - 1,
                        c.stream),
       "yitu_longest_row");
    return out;
}

std::tuple<Tensor, Tensor, Tensor> csr_transpose(const Tensor &indptr, const Tensor &indices,
                                                 int64_t n_src) {
    check_i32(indptr, "indptr", 1);
    check_i32(indices, "indices", 1);
    const int64_t n_rows = indptr.numel() - 1, nnz = indices.numel();
    Call c(indices);
    Tensor t_indptr = c.empty({n_src + 1}, at::kInt), t_rows = c.empty({nnz}, at::kInt),
           t_perm = c.empty({nnz}, at::kInt);
    const auto ws = c.scratch(yitu_csr_transpose_workspace_bytes(nnz, n_src));
    ok(yitu_csr_transpose(static_cast<int32_t *>(t_indptr.data_ptr()),
                          static_cast<int32_t *>(t_rows.data_ptr()),
                          static_cast<int32_t *>(t_perm.data_ptr()), i32(indptr), i32(indices),
                          n_rows, n_src, nnz, kColMask, ws.data_ptr(), ws.numel(), c.stream),
       "yitu_csr_transpose");
    return {t_indptr, t_rows, t_perm};
}

Tensor build_plan(const Tensor &indptr, const Tensor &indices, int64_t n_src, int mask,
                  int64_t max_degree) {
    check_i32(indptr, "indptr", 1);
    check_i32(indices, "indices", 1);
    const int64_t nnz = indices.numel();
    Call c(indices);
    if (max_degree >= 0 && max_degree < kLongRow) {
        Tensor plan = c.empty({(int64_t)yitu_plan_header_bytes()}, at::kByte);
        ok(yitu_plan_build_header(plan.data_ptr(), i32(indptr), i32(indices), indptr.numel() - 1,
                                  n_src, nnz, mask, c.stream),
           "yitu_plan_build_header");
        return plan;
    }
    Tensor plan = c.empty({(int64_t)yitu_plan_bytes(nnz)}, at::kByte);
    const auto ws = c.scratch(yitu_plan_workspace_bytes(nnz));
    ok(yitu_plan_build(plan.data_ptr(), plan.numel(), i32(indptr), i32(indices), indptr.numel() - 1,
                       n_src, nnz, mask, ws.data_ptr(), ws.numel(), c.stream),
       "yitu_plan_build");
    return plan;
}

RowState rows_of(int64_t max_degree, const OptTensor &plan) { return {max_degree, plan}; }
}  // namespace

void bind_ops(py::module_ &m) {
    const auto dtype = [](const py::object &d) {
        return torch::python::detail::py_object_to_dtype(d);
    };
    m.def("agg", [](const Tensor &x, const Tensor &rp, const Tensor &ci, const OptTensor &degrees,
                    const OptTensor &scale, double alpha, int64_t md, const OptTensor &plan) {
        return agg(x, rp, ci, degrees, scale, alpha, rows_of(md, plan));
    });
    m.def("check_inputs", [](const TensorVec &ts) {
        for (const Tensor &t : ts) {
            check_device(t);
            same_device(ts[0], t);
        }
    });
    m.def("edge_scale", &edge_scale);
    m.def("sgemm", [](const Tensor &a, const Tensor &b, bool ta, bool tb, const OptTensor &out) {
        return sgemm(a, b, ta, tb, out);
    });
    m.def("linear_forward", &linear_forward);
    m.def("linear_forward_typed", &linear_forward_typed);
    m.def("sgemm_typed", &sgemm_typed);
    m.def("gemm_bf16", [dtype](const Tensor &a, const Tensor &b, bool tb, const py::object &d,
                               const OptTensor &out) { return gemm_bf16(a, b, tb, dtype(d), out); });
    m.def("gemm_bf16_typed", [dtype](const TensorVec &as, const TensorVec &bs, bool tb,
                                     const py::object &d, const std::optional<TensorVec> &outs) {
        return gemm_bf16_typed(as, bs, tb, dtype(d), outs);
    });
    m.def("gemm_bf16_tn", &gemm_bf16_tn);
    m.def("gemm_bf16_tn_typed", &gemm_bf16_tn_typed);
    m.def("b2gemm", &b2gemm);
    m.def("b2gemm_backward", &b2gemm_backward);
    m.def("spmm_forward", [](const Tensor &v, const Tensor &ip, const Tensor &ix, const Tensor &x,
                             bool bf16_out, int64_t md, const OptTensor &plan) {
        return spmm_forward(v, ip, ix, x, bf16_out, rows_of(md, plan));
    });
    m.def("spmm_backward_check", &spmm_backward_check);
    m.def("spmm_backward", [](const Tensor &v, const Tensor &ip, const Tensor &ix, const Tensor &x,
                              const Tensor &g, bool need_a, bool need_x, int64_t md,
                              const OptTensor &plan, const py::object &t) {
        return spmm_backward(v, ip, ix, x, g, need_a, need_x, rows_of(md, plan), by_source_of(t));
    });
    m.def("edge_dot", [](const Tensor &ip, const Tensor &ix, const Tensor &d, const Tensor &s,
                         int64_t md, const OptTensor &plan) {
        return edge_dot(ip, ix, d, s, rows_of(md, plan));
    });
    m.def("sddmm_forward", [](const Tensor &ip, const Tensor &ix, const Tensor &q, const Tensor &k,
                              int64_t md, const OptTensor &plan) {
        return sddmm_forward(ip, ix, q, k, rows_of(md, plan));
    });
    m.def("sddmm_backward", [](const Tensor &ip, const Tensor &ix, const Tensor &q, const Tensor &k,
                               const Tensor &a, const Tensor &g, int64_t md, const OptTensor &plan,
                               const py::object &t) {
        std::optional<BySource> b;
        if (!t.is_none()) b = by_source_of(t);
        return sddmm_backward(ip, ix, q, k, a, g, rows_of(md, plan), b);
    });
    m.def("gat_one_pass_shape", &gat_one_pass_shape);
    m.def("gat_forward", [](const Tensor &ip, const Tensor &ix, const Tensor &q, const Tensor &k,
                            const Tensor &x, bool stats_only, int64_t md, const OptTensor &plan) {
        GatOut o = gat_forward(ip, ix, q, k, x, stats_only, rows_of(md, plan));
        return std::make_tuple(o.out, o.attn, o.stats);
    });
    m.def("gat_backward", [](const Tensor &ip, const Tensor &ix, const Tensor &q, const Tensor &k,
                             const Tensor &x, const OptTensor &attn, const Tensor &g,
                             const OptTensor &out, bool head_mean, const OptTensor &stats,
                             int64_t md, const OptTensor &plan, const py::object &t) {
        GatGrads r = gat_backward(ip, ix, q, k, x, attn, g, out, head_mean, stats,
                                  rows_of(md, plan), by_source_of(t));
        return std::make_tuple(r.query, r.key, r.x);
    });
    m.def("head_dot", &head_dot);
    m.def("head_dot_backward", &head_dot_backward);
    m.def("skinny_linear_shape", &skinny_linear_shape);
    m.def("skinny_linear", [](const Tensor &x, const Tensor &w, const OptTensor &bias) {
        return skinny_pair(x, w, std::nullopt, bias, std::nullopt).first;
    });
    m.def("skinny_linear_backward", [](const Tensor &x, const Tensor &w, const Tensor &grad_y,
                                       const OptTensor &grad_x, bool need_bias) {
        SkinnyGrads g = skinny_pair_backward(x, w, std::nullopt, grad_y, std::nullopt, grad_x,
                                             need_bias, false);
        return std::make_tuple(g.x, g.w_a, g.bias_a);
    });
    m.def("column_sum", &column_sum);
    m.def("column_sum_typed", &column_sum_typed);
    m.def("coo_to_csr", &coo_to_csr);
    m.def("csr_transpose", &csr_transpose);
    m.def("longest_row", &longest_row);
    m.def("build_plan", &build_plan, py::arg("indptr"), py::arg("indices"), py::arg("n_src"),
          py::arg("mask"), py::arg("max_degree") = -1);
    m.attr("plan_min_edges") = kPlanMinEdges;
}

}  // namespace yitu_bind
