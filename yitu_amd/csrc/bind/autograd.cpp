// The differentiable layers and ops as autograd nodes. Forward and backward run without the
// interpreter (on a small graph it cost more than the kernels did); the sparse structure
// takes no gradient, and a gradient that nobody asked for is not computed.
#include "nodes.hpp"

namespace yitu_bind {
namespace {

// ---- GCN / GIN over the reference's module-1 ops -----------------------------------------
Tensor aggregate(const Kept &k, const Tensor &x) {
    const OptTensor degrees = k.degrees.defined() ? OptTensor(k.degrees) : std::nullopt;
    return agg(x, k.indptr, k.indices, degrees, k.edge_scale, k.alpha,
               row_state(k.indptr, k.indices, x.size(0), kAllBits));
}

struct GcnConvFunction : Function<GcnConvFunction> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &w, KeptPtr k) {
        ctx->save_for_backward({x, w});
        keep(ctx, k);
        return aggregate(*k, sgemm(x, w, false, false, std::nullopt));
    }
    // the reference's semantics: the same CSR aggregates the output gradient
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const Tensor g = aggregate(*kept(ctx), dense(grads[0]));
        Tensor dx, dw;
        if (ctx->needs_input_grad(0)) dx = sgemm(g, saved[1], false, true, std::nullopt);
        if (ctx->needs_input_grad(1)) dw = sgemm(saved[0], g, true, false, std::nullopt);
        return {dx, dw, Tensor()};
    }
};

struct GinConvFunction : Function<GinConvFunction> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &w, KeptPtr k) {
        const Tensor a = aggregate(*k, x);
        ctx->save_for_backward({a, w});
        keep(ctx, k);
        return sgemm(a, w, false, false, std::nullopt);
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const Tensor g = dense(grads[0]);
        Tensor dx, dw;
        if (ctx->needs_input_grad(1)) dw = sgemm(saved[0], g, true, false, std::nullopt);
        if (ctx->needs_input_grad(0))
            dx = aggregate(*kept(ctx), sgemm(g, saved[1], false, true, std::nullopt));
        return {dx, dw, Tensor()};
    }
};

// ---- Linears -----------------------------------------------------------------------------
struct MfmaLinearFunction : Function<MfmaLinearFunction> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &w,
                          const OptTensor &bias) {
        ctx->save_for_backward({x, w});
        ctx->saved_data["bias"] = has(bias);
        return linear_forward(x, w, dense(bias));
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const Tensor g = dense(grads[0]);
        Tensor dx, dw, db;
        if (ctx->needs_input_grad(0)) dx = sgemm(g, saved[1], false, false, std::nullopt);
        const bool want_b = ctx->saved_data["bias"].toBool() && ctx->needs_input_grad(2);
        if (ctx->needs_input_grad(1)) {
            TensorVec dws;
            std::vector<OptTensor> dbs;
            linear_weight_grad({g}, {saved[0]}, {want_b}, &dws, &dbs);
            dw = dws[0];
            db = grad_or_none(dbs[0]);
        } else if (want_b) {
            db = column_sum(g);
        }
        return once({dx, dw, db});
    }
};

struct SkinnyLinearFunction : Function<SkinnyLinearFunction> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &w,
                          const OptTensor &bias) {
        ctx->save_for_backward({x, w});
        ctx->saved_data["bias"] = has(bias);
        return skinny_pair(x, w, std::nullopt, dense(bias), std::nullopt).first;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const SkinnyGrads g =
            skinny_pair_backward(saved[0], saved[1], std::nullopt, dense(grads[0]), std::nullopt,
                                 std::nullopt, ctx->saved_data["bias"].toBool(), false);
        return once({g.x, g.w_a, grad_or_none(g.bias_a)});
    }
};

// Two skinny Linears over one x; an undefined bias is one that is not there.
struct SkinnyPairFunction : Function<SkinnyPairFunction> {
    static variable_list forward(AutogradContext *ctx, const Tensor &x, const Tensor &w_a,
                                 const Tensor &w_b, const Tensor &b_a, const Tensor &b_b) {
        ctx->save_for_backward({x, w_a, w_b});
        ctx->saved_data["bias_a"] = b_a.defined();
        ctx->saved_data["bias_b"] = b_b.defined();
        auto [y_a, y_b] = skinny_pair(x, w_a, w_b, given(b_a), given(b_b));
        return {y_a, *y_b};
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto s = ctx->get_saved_variables();
        const SkinnyGrads g = skinny_pair_backward(
            s[0], s[1], s[2], dense(grads[0]), dense(grads[1]), std::nullopt,
            ctx->saved_data["bias_a"].toBool(), ctx->saved_data["bias_b"].toBool());
        return once({g.x, g.w_a, *g.w_b, grad_or_none(g.bias_a), grad_or_none(g.bias_b)});
    }
};

Tensor linear(const Tensor &x, const Tensor &w, const OptTensor &bias) {
    const Tensor xd = dense(x), wd = dense(w);
    if (skinny_linear_shape(w.size(1), w.size(0))) return SkinnyLinearFunction::apply(xd, wd, bias);
    return MfmaLinearFunction::apply(xd, wd, bias);
}

struct GemmBundleFunction : Function<GemmBundleFunction> {
    static variable_list forward(AutogradContext *ctx, const Tensor &x, const Tensor &w_a,
                                 const Tensor &w_b) {
        ctx->save_for_backward({x, w_a, w_b});
        return b2gemm(x, w_a, w_b);
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto s = ctx->get_saved_variables();
        return once(b2gemm_backward(s[0], s[1], s[2], dense(grads[0]), dense(grads[1])));
    }
};

struct LinearPairFunction : Function<LinearPairFunction> {
    static variable_list forward(AutogradContext *ctx, const Tensor &x, const Tensor &w_a,
                                 const Tensor &w_b, const Tensor &b_a, const Tensor &b_b) {
        ctx->save_for_backward({x, w_a, w_b});
        return linear_forward_typed({x, x}, {w_a, w_b}, {given(b_a), given(b_b)}, std::nullopt);
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto s = ctx->get_saved_variables();
        const Tensor g_a = dense(grads[0]), g_b = dense(grads[1]);
        TensorVec dws;
        std::vector<OptTensor> dbs;
        linear_weight_grad({g_a, g_b}, {s[0], s[0]},
                           {ctx->needs_input_grad(3), ctx->needs_input_grad(4)}, &dws, &dbs);
        Tensor dx;
        if (ctx->needs_input_grad(0)) {
            dx = sgemm(g_a, s[1], false, false, std::nullopt);
            sgemm(g_b, s[2], false, false, dx, true);
        }
        return once({dx, dws[0], dws[1], grad_or_none(dbs[0]), grad_or_none(dbs[1])});
    }
};

// The Linears of several node types into one buffer: y[off_i : off_i + m_i] = x_i . W_i^T + b_i
struct TypedLinearFunction : Function<TypedLinearFunction> {
    static Tensor forward(AutogradContext *ctx, int64_t count, at::TensorList xs, at::TensorList ws,
                          at::TensorList bs, std::vector<bool> has_bias) {
        variable_list saved;
        TensorVec dx, dw, parts;
        std::vector<OptTensor> db;
        int64_t total = 0;
        bool one_shape = true;
        for (int64_t i = 0, b = 0; i < count; i++) {
            total += xs[i].size(0);
            dx.push_back(dense(xs[i]));
            dw.push_back(dense(ws[i]));
            db.push_back(has_bias[i] ? OptTensor(dense(bs[b++])) : std::nullopt);
            one_shape = one_shape && ws[i].sizes() == ws[0].sizes();
        }
        const int64_t n = ws[0].size(0);
        Tensor y = Call(xs[0]).empty({total, n});
        int64_t off = 0;
        for (int64_t i = 0; i < count; i++) {
            parts.push_back(y.narrow(0, off, xs[i].size(0)));
            off += xs[i].size(0);
        }
        if (one_shape) {
            linear_forward_typed(dx, dw, db, parts);
        } else {
            sgemm_typed(dx, dw, false, true, parts);
            for (int64_t i = 0; i < count; i++)
                if (has(db[i])) parts[i].add_(*db[i]);
        }
        for (auto *v : {&xs, &ws})
            for (const Tensor &t : *v) saved.push_back(t);
        ctx->save_for_backward(std::move(saved));
        ctx->saved_data["count"] = count;
        std::vector<int64_t> bias_at;
        for (int64_t i = 0; i < count; i++)
            if (has_bias[i]) bias_at.push_back(i);
        ctx->saved_data["bias_at"] = std::move(bias_at);
        return y;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const int64_t count = ctx->saved_data["count"].toInt();
        const auto bias_at = ctx->saved_data["bias_at"].toIntVector();
        const auto saved = ctx->get_saved_variables();
        const Tensor g = dense(grads[0]);
        TensorVec parts;
        int64_t off = 0;
        for (int64_t i = 0; i < count; i++) {
            parts.push_back(g.narrow(0, off, saved[i].size(0)));
            off += saved[i].size(0);
        }
        // one entry per argument: the count, xs, ws, the biases that are there, the flags
        variable_list out(1 + 2 * count + bias_at.size() + 1);
        TensorVec a, b;
        std::vector<size_t> at;
        const auto take = [&](TensorVec &&made) {
            for (size_t i = 0; i < at.size(); i++) out[at[i]] = made[i];
            a.clear(), b.clear(), at.clear();
        };
        for (int64_t i = 0; i < count; i++)
            if (ctx->needs_input_grad(i)) {
                at.push_back(1 + i);
                a.push_back(parts[i]);
                b.push_back(dense(saved[count + i]));
            }
        if (!at.empty()) take(sgemm_typed(a, b, false, false, std::nullopt));
        // weight gradients, each with the bias gradient that belongs to it
        std::vector<bool> want;
        std::vector<int64_t> bias_slot(count, -1);
        for (size_t j = 0; j < bias_at.size(); j++)
            if (ctx->needs_input_grad(2 * count + j)) bias_slot[bias_at[j]] = 1 + 2 * count + j;
        const bool one_shape = std::all_of(saved.begin() + count, saved.end(), [&](const Tensor &w) {
            return w.sizes() == saved[count].sizes();
        });
        for (int64_t i = 0; i < count; i++) {
            if (one_shape && ctx->needs_input_grad(count + i)) {
                at.push_back(1 + count + i);
                a.push_back(parts[i]);
                b.push_back(dense(saved[i]));
                want.push_back(bias_slot[i] >= 0);
            } else {
                if (ctx->needs_input_grad(count + i))
                    out[1 + count + i] = sgemm(parts[i], dense(saved[i]), true, false, std::nullopt);
                if (bias_slot[i] >= 0) out[bias_slot[i]] = column_sum(dense(parts[i]));
            }
        }
        if (!at.empty()) {
            TensorVec dws;
            std::vector<OptTensor> dbs;
            linear_weight_grad(a, b, want, &dws, &dbs);
            for (size_t i = 0; i < at.size(); i++) {
                out[at[i]] = dws[i];
                if (want[i]) out[bias_slot[at[i] - 1 - count]] = *dbs[i];
            }
        }
        return out;
    }
};

Tensor typed_linear(const TensorVec &xs, const TensorVec &ws, const std::vector<OptTensor> &bs) {
    TensorVec biases;
    std::vector<bool> has_bias;
    for (const OptTensor &b : bs) {
        has_bias.push_back(has(b));
        if (has(b)) biases.push_back(*b);
    }
    TORCH_CHECK(!xs.empty() && xs.size() == ws.size() && xs.size() == bs.size(),
                "typed_linear needs as many weights and biases as inputs, at least one");
    return TypedLinearFunction::apply((int64_t)xs.size(), at::TensorList(xs), at::TensorList(ws),
                                      at::TensorList(biases), has_bias);
}

// ---- sparse ops over a block -------------------------------------------------------------
struct SpmmFunction : Function<SpmmFunction> {
    static Tensor forward(AutogradContext *ctx, const Tensor &values, const Tensor &x, KeptPtr k) {
        ctx->save_for_backward({values, x});
        keep(ctx, k);
        return spmm_forward(values, k->indptr, k->indices, x, false, k->rows());
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const auto k = kept(ctx);
        const Tensor g = dense(grads[0]);
        const bool need_a = ctx->needs_input_grad(0), need_x = ctx->needs_input_grad(1);
        spmm_backward_check(saved[0], k->indptr, k->indices, saved[1], g);
        if (!need_a && !need_x) return {Tensor(), Tensor(), Tensor()};
        const int64_t n_dst = k->indptr.numel() - 1;
        if (!need_a && k->indices.numel() > 0 && n_dst <= kColMask) {
            const OptTensor by = by_source_values(saved[0], k->indptr, k->indices, k->n_src, false);
            if (has(by)) {
                // constant edge weights, seen before: grad_x is a forward product over the
                // by-source structure, its weights already in that order
                const BySource t = by_source(k->indptr, k->indices, k->n_src);
                return once({Tensor(),
                             spmm_forward(*by, t.t_indptr, t.t_rows, g, false,
                                          row_state(t.t_indptr, t.t_rows, n_dst, kColMask)),
                             Tensor()});
            }
        }
        auto [da, dx] = spmm_backward(saved[0], k->indptr, k->indices, saved[1], g, need_a, need_x,
                                      k->rows(), by_source(k->indptr, k->indices, k->n_src));
        return once({grad_or_none(da), grad_or_none(dx), Tensor()});
    }
};

struct SddmmFunction : Function<SddmmFunction> {
    static Tensor forward(AutogradContext *ctx, const Tensor &query, const Tensor &key, KeptPtr k) {
        const Tensor attn =
            sddmm_forward(k->indptr, k->indices, query, key,
                          query.size(0) == 1 ? k->rows()
                                             : RowState{k->rows().max_degree, std::nullopt});
        ctx->save_for_backward({query, key, attn});
        keep(ctx, k);
        return attn;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        // like the reference, both projections are expected to train
        TORCH_CHECK(ctx->needs_input_grad(0) && ctx->needs_input_grad(1),
                    "query and key must both take gradients");
        const auto s = ctx->get_saved_variables();
        const auto k = kept(ctx);
        RowState rows = k->rows();
        if (s[0].size(0) != 1) rows.plan = std::nullopt;
        auto [dq, dk] = sddmm_backward(k->indptr, k->indices, s[0], s[1], s[2], dense(grads[0]), rows,
                                       by_source(k->indptr, k->indices, k->n_src));
        return once({dq, dk, Tensor()});
    }
};

// ---- fused attention -----------------------------------------------------------------------
struct FusedGatFunction : Function<FusedGatFunction> {
    static Tensor forward(AutogradContext *ctx, const Tensor &query, const Tensor &key,
                          const Tensor &x, bool head_mean, KeptPtr k) {
        // one-pass shapes: each row's softmax statistics are kept instead of the probabilities
        k->flag = gat_stats_suffice(x, head_mean) && k->indices.numel() > 0;
        k->flag2 = head_mean;
        const GatOut o = gat_forward(k->indptr, k->indices, query, key, x, k->flag, k->rows());
        ctx->save_for_backward({query, key, x, k->flag ? *o.stats : *o.attn, o.out});
        keep(ctx, k);
        return head_mean ? o.out.mean(1) : o.out;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto s = ctx->get_saved_variables();
        const auto k = kept(ctx);
        const OptTensor attn = k->flag ? std::nullopt : OptTensor(s[3]);
        const OptTensor stats = k->flag ? OptTensor(s[3]) : std::nullopt;
        const GatGrads g = gat_backward(k->indptr, k->indices, s[0], s[1], s[2], attn,
                                        dense(grads[0]), s[4], k->flag2, stats, k->rows(),
                                        by_source(k->indptr, k->indices, k->n_src));
        return {g.query, g.key, g.x, Tensor(), Tensor()};
    }
};

struct GatHeadsFunction : Function<GatHeadsFunction> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x_src, const OptTensor &x_dst,
                          const Tensor &a_src, const Tensor &a_dst, bool head_mean, KeptPtr k) {
        Tensor query, key;
        if (has(x_dst)) {
            query = head_dot(*x_dst, a_dst, std::nullopt).first;
            key = head_dot(x_src, a_src, std::nullopt).first;
        } else {
            auto both = head_dot(x_src, a_dst, a_src);
            query = both.first;
            key = *both.second;
        }
        k->flag = gat_stats_suffice(x_src, head_mean) && k->indices.numel() > 0;
        k->flag2 = head_mean;
        const GatOut o = gat_forward(k->indptr, k->indices, query, key, x_src, k->flag, k->rows());
        variable_list saved = {x_src, a_src, a_dst, query, key, k->flag ? *o.stats : *o.attn, o.out};
        if (has(x_dst)) saved.push_back(*x_dst);
        ctx->save_for_backward(std::move(saved));
        keep(ctx, k);
        return head_mean ? o.out.mean(1) : o.out;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto s = ctx->get_saved_variables();
        const auto k = kept(ctx);
        const OptTensor attn = k->flag ? std::nullopt : OptTensor(s[5]);
        const OptTensor stats = k->flag ? OptTensor(s[5]) : std::nullopt;
        const GatGrads g = gat_backward(k->indptr, k->indices, s[3], s[4], s[0], attn,
                                        dense(grads[0]), s[6], k->flag2, stats, k->rows(),
                                        by_source(k->indptr, k->indices, k->n_src));
        if (s.size() == 7) {
            auto [dx, d_dst, d_src] = head_dot_backward(s[0], s[2], s[1], g.query, g.key, g.x);
            return once({dx, Tensor(), *d_src, d_dst, Tensor(), Tensor()});
        }
        auto [dx, d_src, none] = head_dot_backward(s[0], s[1], std::nullopt, g.key, std::nullopt, g.x);
        auto [dxd, d_dst, none2] =
            head_dot_backward(s[7], s[2], std::nullopt, g.query, std::nullopt, std::nullopt);
        return once({dx, dxd, d_src, d_dst, Tensor(), Tensor()});
    }
};

// The attention layer whose logit terms are Linears of the projected features (reference
// test/common/model.py:61-106) as one node: h = x W_v^T + b_v, q = h W_q^T + b_q,
// k = h W_k^T + b_k, attention, mean over heads. As separate nodes the two gradients of h met
// in an addition pass over [n, H F], beside concatenations and copies of the two projections
// (140 us of elementwise passes at 2^18 nodes x 4 x 64); here the projections' backward adds
// to the attention's gradient in place.
struct GatLayerFunction : Function<GatLayerFunction> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &w_v, const Tensor &b_v,
                          const Tensor &w_q, const Tensor &b_q, const Tensor &w_k, const Tensor &b_k,
                          KeptPtr k) {
        const int64_t heads = w_q.size(0);
        const Tensor h = linear_forward(x, w_v, given(b_v));
        auto [q, key] = skinny_pair(h, w_q, w_k, given(b_q), given(b_k));
        const Tensor h3 = h.view({h.size(0), heads, -1});
        k->flag = gat_stats_suffice(h3, true) && k->indices.numel() > 0;
        const GatOut o = gat_forward(k->indptr, k->indices, q, *key, h3, k->flag, k->rows());
        ctx->save_for_backward({x, w_v, w_q, w_k, h, q, *key, k->flag ? *o.stats : *o.attn, o.out});
        ctx->saved_data["bias_v"] = b_v.defined();
        ctx->saved_data["bias_q"] = b_q.defined();
        ctx->saved_data["bias_k"] = b_k.defined();
        keep(ctx, k);
        return o.out.mean(1);
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto s = ctx->get_saved_variables();
        const auto k = kept(ctx);
        const OptTensor attn = k->flag ? std::nullopt : OptTensor(s[7]);
        const OptTensor stats = k->flag ? OptTensor(s[7]) : std::nullopt;
        const Tensor &h = s[4];
        const GatGrads g = gat_backward(k->indptr, k->indices, s[5], s[6],
                                        h.view({h.size(0), s[2].size(0), -1}), attn, dense(grads[0]),
                                        s[8], true, stats, k->rows(),
                                        by_source(k->indptr, k->indices, k->n_src));
        const SkinnyGrads p = skinny_pair_backward(
            h, s[2], s[3], g.query, g.key, g.x.view(h.sizes()), ctx->saved_data["bias_q"].toBool(),
            ctx->saved_data["bias_k"].toBool());
        const bool bias_v = ctx->saved_data["bias_v"].toBool();
        TensorVec dws;
        std::vector<OptTensor> dbs{std::nullopt};
        if (ctx->needs_input_grad(1)) linear_weight_grad({p.x}, {s[0]}, {bias_v}, &dws, &dbs);
        else if (bias_v) dbs[0] = column_sum(p.x);
        Tensor dx;
        if (ctx->needs_input_grad(0)) dx = sgemm(p.x, s[1], false, false, std::nullopt);
        return once({dx, dws.empty() ? Tensor() : dws[0], grad_or_none(dbs[0]), p.w_a,
                     grad_or_none(p.bias_a), *p.w_b, grad_or_none(p.bias_b), Tensor()});
    }
};

}  // namespace

void bind_autograd(py::module_ &m) {
    const auto conv = [](const Tensor &x, const Tensor &w, const Tensor &rp, const Tensor &ci,
                         const Tensor &pp, const Tensor &p2n) {
        for (const Tensor *t : {&x, &w, &rp, &ci, &pp, &p2n}) {
            check_device(*t);
            same_device(x, *t);
        }
        return graph_of(rp, ci, x.size(0));
    };
    m.def("gcn_conv",
          [conv](const Tensor &x, const Tensor &w, const Tensor &rp, const Tensor &ci,
                 const Tensor &degrees, const Tensor &pp, const Tensor &p2n, const OptTensor &scale) {
              const auto k = conv(x, w, rp, ci, pp, p2n);
              check_device(degrees);
              same_device(x, degrees);
              k->degrees = degrees;
              k->edge_scale = scale;
              return GcnConvFunction::apply(x, w, k);
          });
    m.def("gin_conv", [conv](const Tensor &x, const Tensor &w, const Tensor &rp, const Tensor &ci,
                             double eps, const Tensor &pp, const Tensor &p2n) {
        const auto k = conv(x, w, rp, ci, pp, p2n);
        k->alpha = eps;
        return GinConvFunction::apply(x, w, k);
    });
    m.def("linear", &linear);
    m.def("skinny_linear_fn", [](const Tensor &x, const Tensor &w, const OptTensor &b) {
        return SkinnyLinearFunction::apply(x, w, b);
    });
    m.def("gemm_bundle", [](const Tensor &x, const Tensor &a, const Tensor &b) {
        return GemmBundleFunction::apply(x, a, b);
    });
    m.def("linear_pair", [](const Tensor &x, const Tensor &w_a, const Tensor &w_b, const OptTensor &b_a,
                            const OptTensor &b_b) {
        return LinearPairFunction::apply(x, w_a, w_b, grad_or_none(b_a), grad_or_none(b_b));
    });
    m.def("skinny_pair", [](const Tensor &x, const Tensor &w_a, const Tensor &w_b, const OptTensor &b_a,
                            const OptTensor &b_b) {
        return SkinnyPairFunction::apply(dense(x), dense(w_a), dense(w_b), grad_or_none(b_a),
                                         grad_or_none(b_b));
    });
    m.def("typed_linear", &typed_linear);
    m.def("gspmm", [](const Tensor &ip, const Tensor &ix, const Tensor &values, const Tensor &x) {
        return SpmmFunction::apply(values, x, graph_of(ip, ix, x.size(0)));
    });
    m.def("gsddmm", [](const Tensor &ip, const Tensor &ix, const Tensor &q, const Tensor &k) {
        return SddmmFunction::apply(q, k, graph_of(ip, ix, k.size(0)));
    });
    m.def("fused_gat", [](const Tensor &ip, const Tensor &ix, const Tensor &q, const Tensor &k,
                          const Tensor &x, bool head_mean) {
        return FusedGatFunction::apply(q, k, x, head_mean, graph_of(ip, ix, x.size(0)));
    });
    m.def("gat_heads", [](const Tensor &ip, const Tensor &ix, const Tensor &x_src,
                          const OptTensor &x_dst, const Tensor &a_src, const Tensor &a_dst,
                          bool head_mean) {
        return GatHeadsFunction::apply(x_src, x_dst, a_src, a_dst, head_mean,
                                       graph_of(ip, ix, x_src.size(0)));
    });
    m.def("gat_layer", [](const Tensor &ip, const Tensor &ix, const Tensor &x, const Tensor &w_v,
                          const OptTensor &b_v, const Tensor &w_q, const OptTensor &b_q,
                          const Tensor &w_k, const OptTensor &b_k) -> OptTensor {
        // shapes it does not take (the caller composes those): a projection too wide for the
        // skinny product, values so narrow that they are one themselves, no rows
        const bool takes = x.dim() == 2 && x.is_cuda() && x.size(0) > 0 &&
                           x.scalar_type() == at::kFloat && w_v.scalar_type() == at::kFloat &&
                           w_q.scalar_type() == at::kFloat && w_q.sizes() == w_k.sizes() &&
                           skinny_linear_shape(w_q.size(1), 2 * w_q.size(0)) &&
                           !skinny_linear_shape(w_v.size(1), w_v.size(0));
        if (!takes) return std::nullopt;
        return GatLayerFunction::apply(dense(x), dense(w_v), grad_or_none(b_v), dense(w_q),
                                       grad_or_none(b_q), dense(w_k), grad_or_none(b_k),
                                       graph_of(ip, ix, x.size(0)));
    });
}

}  // namespace yitu_bind

PYBIND11_MODULE(_ops, m) {
    yitu_bind::bind_graph_state(m);
    yitu_bind::bind_ops(m);
    yitu_bind::bind_autograd(m);
    yitu_bind::bind_batched(m);
    yitu_bind::bind_temporal(m);
}
