"""The temporal attention layer (YiTu_GNN/YiTu_T/layers.py:75-142) as one autograd node
of a dozen launches: input assembly, Q | K | V as one grouped product, attention per root,
output product, ReLU + LayerNorm; the backward mirrors it. Biases ride as one more column
of every weight matrix against a column of ones, so no launch adds a bias or sums a bias
gradient. The launches of a direction are one native call (csrc/bind/temporal.cpp)."""
import torch

from .. import _lib

MAX_OUT, MAX_HEADS = 256, 8


def supported(dim_node, dim_edge, dim_time, dim_out, num_head):
    """Shapes the fused kernels take: a query made of node or time features, rows of at
    most 256 floats, at most 8 heads."""
    return (dim_node + dim_time > 0 and 1 <= dim_out <= MAX_OUT and dim_time <= MAX_OUT
            and 1 <= num_head <= MAX_HEADS and dim_out % num_head == 0)


def _dense(t):
    return None if t is None else t.contiguous()


class TemporalAttentionFunction(torch.autograd.Function):
    """apply(indptr, n_dst, num_head, eps, h, f, dt, time_w, time_b, w_q, b_q, w_k, b_k, w_v,
    b_v, w_out, b_out, ln_w, ln_b) -> [n_dst, dim_out]. ``h`` [n_dst + E, dim_node] or None,
    ``f`` [E, dim_edge] or None, ``time_w`` [dim_time, 1] / ``time_b`` or None."""

    @staticmethod
    def forward(ctx, indptr, n_dst, num_head, eps, h, f, dt, time_w, time_b, w_q, b_q, w_k, b_k,
                w_v, b_v, w_out, b_out, ln_w, ln_b):
        h, f, dt, time_w, time_b = _dense(h), _dense(f), _dense(dt), _dense(time_w), _dense(time_b)
        ln_w = _dense(ln_w)
        params = [_dense(t) for t in (w_q, b_q, w_k, b_k, w_v, b_v, w_out, b_out)]
        out, buf = _lib.ops().tattn_forward(indptr, n_dst, num_head, eps, h, f, dt, time_w, time_b,
                                            params, ln_w, _dense(ln_b))
        ctx.dims = (n_dst, dt.numel(), 0 if h is None else h.size(1), 0 if f is None else f.size(1),
                    0 if time_w is None else time_w.size(0), w_k.size(0), num_head)
        ctx.eps = eps
        ctx.buf = buf
        ctx.save_for_backward(indptr, dt, time_w, time_b, ln_w)
        return out

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, grad_out):
        indptr, dt, time_w, time_b, ln_w = ctx.saved_tensors
        grads = _lib.ops().tattn_backward(grad_out.contiguous(), ctx.buf, indptr, dt, time_w, time_b,
                                          ln_w, ctx.dims, ctx.eps, ctx.needs_input_grad[4],
                                          ctx.needs_input_grad[5])
        return (None, None, None, None, grads[0], grads[1], None, *grads[2:])
