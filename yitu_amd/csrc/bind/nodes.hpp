// What the autograd nodes share: what a node keeps beside its saved tensors, and the refusal
// of a second differentiation.
#pragma once
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>

#include "bind.hpp"

namespace yitu_bind {

using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

// What a node keeps besides its saved tensors.
struct Kept : torch::CustomClassHolder {
    Tensor indptr, indices, degrees;
    OptTensor edge_scale;
    int64_t n_src = 0;
    int mask = kColMask;
    double alpha = 1.0;
    bool flag = false, flag2 = false;
    RowState rows() const { return row_state(indptr, indices, n_src, mask); }
};
using KeptPtr = c10::intrusive_ptr<Kept>;

inline void keep(AutogradContext *ctx, const KeptPtr &k) {
    ctx->saved_data["kept"] = c10::IValue::make_capsule(k);
}
inline KeptPtr kept(AutogradContext *ctx) {
    return c10::static_intrusive_pointer_cast<Kept>(ctx->saved_data["kept"].toCapsule());
}
inline KeptPtr graph_of(const Tensor &indptr, const Tensor &indices, int64_t n_src) {
    auto k = c10::make_intrusive<Kept>();
    k->indptr = indptr;
    k->indices = indices;
    k->n_src = n_src;
    return k;
}

// The gradients of ops whose backward is not differentiable itself: a second differentiation
// raises instead of silently giving nothing.
inline variable_list once(variable_list grads) {
    if (!at::GradMode::is_enabled()) return grads;
    std::vector<size_t> at;
    variable_list live;
    for (size_t i = 0; i < grads.size(); i++)
        if (grads[i].defined()) {
            at.push_back(i);
            live.push_back(grads[i].detach().requires_grad_());
        }
    torch::autograd::DelayedError error(
        "trying to differentiate twice a function that was marked with @once_differentiable",
        (int64_t)live.size());
    live = error(std::move(live));
    for (size_t i = 0; i < at.size(); i++) grads[at[i]] = live[i];
    return grads;
}

inline Tensor dense(const Tensor &t) { return t.is_contiguous() ? t : t.contiguous(); }
inline OptTensor dense(const OptTensor &t) { return has(t) ? OptTensor(dense(*t)) : std::nullopt; }
inline Tensor grad_or_none(const OptTensor &t) { return has(t) ? *t : Tensor(); }
inline OptTensor given(const Tensor &t) { return t.defined() ? OptTensor(dense(t)) : std::nullopt; }

}  // namespace yitu_bind
