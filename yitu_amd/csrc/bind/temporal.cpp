// The temporal sampler's call and the temporal attention layer's two (yitu_amd/temporal/fused.py
// states the layer): dimensions, buffers and the dozen launches of a pass without the
// interpreter, which took as long as the launches themselves.
#include "bind.hpp"

namespace yitu_bind {
namespace {

// Consecutive fp32 matrices in one buffer, each at a multiple of 64 floats.
struct Carver {
    int64_t room = 0;
    std::vector<int64_t> at;
    int add(int64_t rows, int64_t cols) {
        at.push_back(room);
        room += (rows * cols + 63) / 64 * 64;
        return (int)at.size() - 1;
    }
};

struct Dims {
    int64_t B, E, Dn, De, Dt, O, H, LD;
};

Dims dims_of(const OptTensor &h, const OptTensor &f, const Tensor &dt, const OptTensor &time_w,
             const Tensor &w_k, int64_t n_dst, int64_t heads) {
    Dims d{n_dst, dt.numel(), has(h) ? h->size(1) : 0, has(f) ? f->size(1) : 0,
           has(time_w) ? time_w->size(0) : 0, w_k.size(0), heads, 0};
    d.LD = yitu_tattn_row_length(d.Dn, d.De, d.Dt, d.O);
    return d;
}

// What the forward keeps for the backward, in one buffer.
struct Kept {
    Carver c;
    int x_kv, x_q, x_r, w_kv, w_q2, w_r, kv, q2, attn, pre;
    explicit Kept(const Dims &d)
        : x_kv(c.add(d.E, d.LD)), x_q(c.add(d.B, d.LD)), x_r(c.add(d.B, d.LD)),
          w_kv(c.add(2 * d.O, d.LD)), w_q2(c.add(2 * d.O, d.LD)), w_r(c.add(d.O, d.LD)),
          kv(c.add(d.E, 2 * d.O)), q2(c.add(d.B, 2 * d.O)), attn(c.add(d.E, d.H)),
          pre(c.add(d.B, d.O)) {}
};

void gemm(const Call &c, float *out, const float *a, const float *b, int64_t m, int64_t n, int64_t k,
          bool ta, bool tb, int64_t lda, int64_t ldb, int64_t ldc) {
    ok(yitu_sgemm(out, a, b, m, n, k, ta, tb, lda, ldb, ldc, 0, nullptr, 0, c.stream), "yitu_sgemm");
}

std::pair<Tensor, Tensor> tattn_forward(const Tensor &indptr, int64_t n_dst, int64_t heads, double eps,
                                        const OptTensor &h, const OptTensor &f, const Tensor &dt,
                                        const OptTensor &time_w, const OptTensor &time_b,
                                        const TensorVec &params, const Tensor &ln_w,
                                        const Tensor &ln_b) {
    check_i32(indptr, "indptr", 1);
    check_f32(dt, "dt");
    for (const OptTensor *t : {&h, &f, &time_w, &time_b})
        if (has(*t)) {
            check_f32(**t, "input");
            same_device(dt, **t);
        }
    TORCH_CHECK(params.size() == 8, "the layer has eight projection tensors");
    for (const Tensor &t : params) check_f32(t, "parameter");
    same_device(dt, indptr, params[0], params[1], params[2], params[3], params[4], params[5], params[6],
                params[7], ln_w, ln_b);
    check_f32(ln_w, "ln_w");
    check_f32(ln_b, "ln_b");
    const Dims d = dims_of(h, f, dt, time_w, params[2], n_dst, heads);
    TORCH_CHECK(indptr.numel() == n_dst + 1, "indptr must be [n_dst + 1]");
    TORCH_CHECK(!has(h) || h->size(0) == d.B + d.E, "node features: one row per root and per edge");
    TORCH_CHECK(!has(f) || f->size(0) == d.E, "edge features: one row per edge");
    TORCH_CHECK(!has(time_w) || (time_w->numel() == d.Dt && has(time_b) && time_b->numel() == d.Dt),
                "the time encoder is a Linear(1, dim_time)");
    const int64_t Dkv = d.Dn + d.De + d.Dt, Dq = d.Dn + d.Dt;
    const int64_t want[8] = {d.O * Dq, d.O, d.O * Dkv, d.O, d.O * Dkv, d.O, d.O * (d.O + d.Dn), d.O};
    for (int i = 0; i < 8; i++)
        TORCH_CHECK(params[i].numel() == want[i], "projection tensor ", i, " has the wrong size");
    TORCH_CHECK(ln_w.numel() == d.O && ln_b.numel() == d.O, "layer_norm has the wrong size");
    Call c(dt);
    const Kept k(d);
    Tensor buf = c.empty({std::max<int64_t>(k.c.room, 64)}), out = c.empty({d.B, d.O});
    const auto p = [&](int i) { return f32(buf) + k.c.at[i]; };
    ok(yitu_tattn_prepare(p(k.x_kv), p(k.x_q), p(k.x_r), p(k.w_kv), p(k.w_q2), p(k.w_r), f32(h), f32(f),
                          f32(dt), f32(time_w), f32(time_b), f32(params[0]), f32(params[1]),
                          f32(params[2]), f32(params[3]), f32(params[4]), f32(params[5]),
                          f32(params[6]), f32(params[7]), d.B, d.E, d.Dn, d.De, d.Dt, d.O, d.LD,
                          c.stream),
       "yitu_tattn_prepare");
    if (d.E > 0) {
        float *cs[] = {p(k.kv), p(k.q2)};
        const float *as[] = {p(k.x_kv), p(k.x_q)}, *bs[] = {p(k.w_kv), p(k.w_q2)};
        const int64_t ms[] = {d.E, d.B}, ks[] = {d.LD, d.LD};
        ok(yitu_sgemm_typed(cs, as, bs, ms, ks, 2, 2 * d.O, 0, 1, d.LD, d.LD, 2 * d.O, 0, nullptr, 0,
                            c.stream),
           "yitu_sgemm_typed");
    } else {
        gemm(c, p(k.q2), p(k.x_q), p(k.w_q2), d.B, 2 * d.O, d.LD, false, true, d.LD, d.LD, 2 * d.O);
    }
    ok(yitu_tattn_forward(p(k.x_r), p(k.attn), p(k.q2), p(k.kv), i32(indptr), d.B, d.E, d.O,
                          d.H, d.LD, c.stream),
       "yitu_tattn_forward");
    gemm(c, p(k.pre), p(k.x_r), p(k.w_r), d.B, d.O, d.LD, false, true, d.LD, d.LD, d.O);
    ok(yitu_relu_layernorm_forward(f32(out), p(k.pre), f32(ln_w), f32(ln_b), d.B, d.O, (float)eps,
                                   c.stream),
       "yitu_relu_layernorm_forward");
    return {out, buf};
}

int64_t up4(int64_t n) { return (n + 3) / 4 * 4; }

// grad_h, grad_f (None where not needed), time_w, time_b, w_q, b_q, w_k, b_k, w_v, b_v, w_out,
// b_out, ln_w, ln_b
std::vector<OptTensor> tattn_backward(const Tensor &grad_out, const Tensor &buf, const Tensor &indptr,
                                      const Tensor &dt, const OptTensor &time_w,
                                      const OptTensor &time_b, const Tensor &ln_w,
                                      const std::vector<int64_t> &dim, double eps, bool need_h,
                                      bool need_f) {
    const Dims d{dim.at(0), dim.at(1), dim.at(2), dim.at(3), dim.at(4), dim.at(5), dim.at(6),
                 yitu_tattn_row_length(dim.at(2), dim.at(3), dim.at(4), dim.at(5))};
    const Kept k(d);
    check_f32(grad_out, "grad_out", 2);
    same_device(grad_out, buf, indptr, dt, ln_w);
    TORCH_CHECK(grad_out.size(0) == d.B && grad_out.size(1) == d.O &&
                    buf.numel() >= std::max<int64_t>(k.c.room, 64),
                "temporal attention backward: not the forward's operands");
    const int64_t Dkv = d.Dn + d.De + d.Dt, Dq = d.Dn + d.Dt;
    need_h = need_h && d.Dn > 0;
    need_f = need_f && d.De > 0;
    // Columns of the input gradients that anybody reads: the time encoding's, the features' only
    // where their gradient is asked for. Whole 16-byte pieces, both windows of one width where the
    // two products can then share a launch.
    const int64_t first_kv = (need_h ? 0 : need_f ? d.Dn : d.Dn + d.De) / 4 * 4;
    const int64_t first_q = (need_h ? 0 : d.Dn) / 4 * 4;
    int64_t n_kv = std::max<int64_t>(up4(Dkv - first_kv), 4), n_q = std::max<int64_t>(up4(Dq - first_q), 4);
    const int64_t both = std::max(n_kv, n_q);
    if (first_kv + both <= d.LD && first_q + both <= d.LD) n_kv = n_q = both;
    const bool reads_kv = d.E > 0 && (d.Dt > 0 || need_h || need_f), reads_q = d.Dt > 0 || need_h;
    const int64_t n_r = need_h ? d.LD : up4(d.O);
    const int64_t rows_ln = yitu_tattn_partial_rows(d.B), rows_t = yitu_tattn_partial_rows(d.B + d.E);
    Carver c1;
    const int d_pre2 = c1.add(d.B, 2 * d.O), dx_r = c1.add(d.B, n_r), dq2 = c1.add(d.B, 2 * d.O),
              dkv = c1.add(d.E, 2 * d.O), scratch = c1.add(d.E, 2 * d.H), dx_kv = c1.add(d.E, n_kv),
              dx_q = c1.add(d.B, n_q), part_ln = c1.add(rows_ln, 2 * d.O),
              part_t = c1.add(rows_t, 2 * std::max<int64_t>(d.Dt, 1)), dw_kv = c1.add(2 * d.O, d.LD),
              dw_q = c1.add(d.O, d.LD), dw_r = c1.add(d.O, d.LD);
    Call c(grad_out);
    Tensor work = c.empty({std::max<int64_t>(c1.room, 64)});
    const auto w = [&](int i) { return f32(work) + c1.at[i]; };
    const auto p = [&](int i) { return f32(buf) + k.c.at[i]; };
    std::vector<OptTensor> g(14);
    if (need_h) g[0] = c.empty({d.B + d.E, d.Dn});
    if (need_f) g[1] = c.empty({d.E, d.De});
    Tensor d_time = c.empty({2, std::max<int64_t>(d.Dt, 1)}), d_ln = c.empty({2, d.O});
    const int64_t width[4] = {Dq, Dkv, Dkv, d.O + d.Dn};
    for (int i = 0; i < 4; i++) {
        g[4 + 2 * i] = c.empty({d.O, width[i]});
        g[5 + 2 * i] = c.empty({d.O});
    }
    ok(yitu_relu_layernorm_backward(w(d_pre2), w(part_ln), f32(grad_out), p(k.pre), f32(ln_w), d.B, d.O,
                                    2 * d.O, (float)eps, c.stream),
       "yitu_relu_layernorm_backward");
    gemm(c, w(dx_r), w(d_pre2), p(k.w_r), d.B, n_r, d.O, false, false, 2 * d.O, d.LD, n_r);
    ok(yitu_tattn_backward(w(dq2), w(dkv), w(scratch), w(dx_r), p(k.q2), p(k.kv), p(k.attn),
                           i32(indptr), d.B, d.E, d.O, d.H, n_r, c.stream),
       "yitu_tattn_backward");
    if (reads_kv && reads_q && n_kv == n_q) {
        float *cs[] = {w(dx_kv), w(dx_q)};
        const float *as[] = {w(dkv), w(dq2)}, *bs[] = {p(k.w_kv) + first_kv, p(k.w_q2) + first_q};
        const int64_t ms[] = {d.E, d.B}, ks[] = {2 * d.O, d.O};
        ok(yitu_sgemm_typed(cs, as, bs, ms, ks, 2, n_kv, 0, 0, 2 * d.O, d.LD, n_kv, 0, nullptr, 0,
                            c.stream),
           "yitu_sgemm_typed");
    } else {
        if (reads_kv)
            gemm(c, w(dx_kv), w(dkv), p(k.w_kv) + first_kv, d.E, n_kv, 2 * d.O, false, false, 2 * d.O,
                 d.LD, n_kv);
        if (reads_q)
            gemm(c, w(dx_q), w(dq2), p(k.w_q2) + first_q, d.B, n_q, d.O, false, false, 2 * d.O, d.LD,
                 n_q);
    }
    {
        const auto ws = c.scratch(yitu_sgemm_workspace_bytes(2 * d.O, d.LD, std::max(d.E, d.B), 3));
        float *cs[] = {w(dw_kv), w(dw_q), w(dw_r)};
        const float *as[] = {w(dkv), w(dq2), w(d_pre2)}, *bs[] = {p(k.x_kv), p(k.x_q), p(k.x_r)};
        const int64_t ms[] = {2 * d.O, d.O, d.O}, ks[] = {d.E, d.B, d.B};
        const int from = d.E > 0 ? 0 : 1;
        if (from) work.narrow(0, c1.at[dw_kv], 2 * d.O * d.LD).zero_();
        ok(yitu_sgemm_typed(cs + from, as + from, bs + from, ms + from, ks + from, 3 - from, d.LD, 1, 0,
                            2 * d.O, d.LD, d.LD, 0, ws.data_ptr(), ws.numel(), c.stream),
           "yitu_sgemm_typed");
    }
    ok(yitu_tattn_finalize_windows(f32(g[0]), f32(g[1]), w(part_t), w(dx_kv), n_kv, first_kv, w(dx_q), n_q,
                                   first_q, w(dx_r), n_r, f32(dt), f32(time_w), f32(time_b), d.B, d.E,
                                   d.Dn, d.De, d.Dt, d.O, d.LD, c.stream),
       "yitu_tattn_finalize");
    ok(yitu_tattn_collect(f32(d_ln), f32(d_time), f32(g[4]), f32(g[5]), f32(g[6]), f32(g[7]), f32(g[8]),
                          f32(g[9]), f32(g[10]), f32(g[11]), w(part_ln), rows_ln, w(part_t), rows_t,
                          w(dw_kv), w(dw_q), w(dw_r), d.Dn, d.De, d.Dt, d.O, d.LD, c.stream),
       "yitu_tattn_collect");
    if (d.Dt > 0) {
        g[2] = d_time.select(0, 0).view({d.Dt, 1});
        g[3] = d_time.select(0, 1);
    }
    g[12] = d_ln.select(0, 0);
    g[13] = d_ln.select(0, 1);
    return g;
}

// One layer of most-recent sampling: {row, col, eid, ts, dts, nodes, block indptr}, cut to the
// sampled edges (one wait for their number).
TensorVec tsample_recent(const Tensor &cursor, const Tensor &indptr, const Tensor &indices,
                         const Tensor &eid, const Tensor &ts, const Tensor &roots,
                         const Tensor &root_ts, int64_t fan, bool prop_time) {
    check_i32(cursor, "cursor", 1);
    check_i32(indptr, "indptr", 1);
    check_i32(indices, "indices", 1);
    check_i32(eid, "eid", 1);
    check_f32(ts, "ts", 1);
    check_i32(roots, "roots", 1);
    check_f32(root_ts, "root_ts", 1);
    same_device(cursor, indptr, indices, eid, ts, roots, root_ts);
    const int64_t n = roots.numel(), n_nodes = indptr.numel() - 1;
    TORCH_CHECK(root_ts.numel() == n && cursor.numel() >= n_nodes, "sample: operand too short");
    Call c(roots);
    const auto i32s = [&](int64_t m) { return c.empty({std::max<int64_t>(m, 1)}, at::kInt); };
    const auto f32s = [&](int64_t m) { return c.empty({std::max<int64_t>(m, 1)}); };
    Tensor row = i32s(n * fan), col = i32s(n * fan), e = i32s(n * fan), t = f32s(n * (fan + 1)),
           dts = f32s(n * (fan + 1)), nodes = i32s(n * (fan + 1)), block = i32s(n + 1),
           count = c.empty({1}, at::kLong);
    const auto ws = c.scratch(yitu_tsample_workspace_bytes(n));
    const auto out = [](const Tensor &x) { return static_cast<int32_t *>(x.data_ptr()); };
    ok(yitu_tsample_recent_block(out(block), out(row), out(col), out(e), f32(t), f32(dts), out(nodes),
                                 static_cast<long long *>(count.data_ptr()), out(cursor),
                                 i32(indptr), i32(indices), i32(eid),
                                 f32(ts), n_nodes, i32(roots), f32(root_ts), n, (int)fan,
                                 prop_time, ws.data_ptr(), ws.numel(), c.stream),
       "yitu_tsample_recent");
    const int64_t m = count.item<int64_t>();
    TORCH_CHECK(m >= 0, "sample failed: a root node id is out of range");
    return {row.narrow(0, 0, m), col.narrow(0, 0, m), e.narrow(0, 0, m), t.narrow(0, 0, n + m),
            dts.narrow(0, 0, n + m), nodes.narrow(0, 0, n + m), block};
}

}  // namespace

void bind_temporal(py::module_ &m) {
    using release = py::call_guard<py::gil_scoped_release>;
    m.def("tattn_forward", &tattn_forward, release());
    m.def("tattn_backward", &tattn_backward, release());
    m.def("tsample_recent", &tsample_recent, release());
}

}  // namespace yitu_bind
