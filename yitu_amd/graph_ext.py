"""Drop-in for the reference's ``graph_ext`` extension module
(YiTu_GNN/YiTu_H/src/entry.cpp:184-193): ``spmm_forward/backward``,
``sddmm_forward/backward``, ``hfused_forward/backward``, ``b2gemm`` and
``b2gemm_backward`` with the reference's argument order, dtype checks
(CHECK_INPUT: device + contiguous + exact dtype, common.h:6-12) and return
arity, backed by libyitu_hip.so.

Observable differences from the reference:
  * any number of destination rows works (the reference launches
    ``dim3(n_heads, n_nodes)`` and silently returns zeros above 65,535 rows,
    spmm_cuda.cu:57);
  * the edge softmax subtracts the row maximum (the reference does not,
    sddmm_cuda.cu:15-21); equal within tolerance wherever the reference does
    not overflow;
  * backward scatters are gathers over a transposed structure that is built on
    the device once per graph and cached on the ``indices`` tensor: results are
    bitwise reproducible, unlike the reference's float atomics;
  * ``hfused_backward`` returns ``[grad_a, grad_x, grad_query, grad_key]``; the
    reference version drops the first two and mis-indexes heads
    (hfused_cuda.cu:59,186) and is unreachable from its Python side.
"""
import torch

from . import _lib
from ._lib import c_i64, c_int, c_size, check, ptr, stream_ptr

COL_MASK = 0xFFFFFF


def _check(t, dtype, name, dim=None):
    # CHECK_INPUT(x, dtype) of the reference (common.h:6-12)
    _lib.require_device(t)
    _lib.require_dtype(t, dtype, name)
    if dim is not None and t.dim() != dim:
        raise RuntimeError("%s must be %d-D, got %d-D" % (name, dim, t.dim()))


def _size_fn(name):
    fn = getattr(_lib.lib(), name)
    fn.restype = c_size
    return fn


# --------------------------------------------------------------------------- #
# transposed structure, cached per (indptr, indices) pair
# --------------------------------------------------------------------------- #
class _Transposed:
    __slots__ = ("t_indptr", "t_rows", "t_perm", "max_degree_t", "n_src", "plan_t")


def transposed(indptr, indices, n_src):
    """By-source view (t_indptr, t_rows, t_perm) of a packed CSR, built on the
    device on first use and kept for as long as ``indices`` is alive."""
    native = _lib.ops()
    t = native.find_by_source(indptr, indices, int(n_src))
    if t is None:
        t = _Transposed()
        t.n_src = int(n_src)
        t.t_indptr, t.t_rows, t.t_perm = native.csr_transpose(indptr, indices, int(n_src))
        t.max_degree_t = _lib.max_degree(t.t_indptr)
        t.plan_t = _lib.row_plan(t.t_indptr, t.t_rows, indptr.numel() - 1, 0x7FFFFFFF)
        native.put_by_source(indptr, indices, int(n_src), _lib._Built(t, indices.device))
        _lib.watch(indices)
    return t


def forget(*tensors):
    """Drops everything derived from the given index / weight tensors: widest row, row
    plan, by-source view, by-source weight copies. Needed after a tensor was refilled in
    place through its raw pointer (kernels of this library, DLPack consumers): torch's
    version counter, which the caches key on, does not see such writes."""
    _lib.forget(*tensors)


# --------------------------------------------------------------------------- #
# SpMM
# --------------------------------------------------------------------------- #
def spmm_forward(values, indptr, indices, features, out_dtype=torch.float32):
    """out[r,h,k] = sum_i values[i,h] * features[col_i,h,k] (entry.cpp:80-90).
    ``features`` fp32 like the reference, or bf16 (fp32 accumulate; fp32 out, or bf16 rows
    with ``out_dtype=torch.bfloat16``: one rounding per output)."""
    if out_dtype not in (torch.float32, torch.bfloat16):
        raise RuntimeError("out_dtype is float32 or bfloat16")
    return _lib.ops().spmm_forward(values, indptr, indices, features, out_dtype == torch.bfloat16,
                                   _lib.max_degree(indptr),
                                   _lib.row_plan(indptr, indices, features.size(0), COL_MASK))


def spmm_backward(values, indptr, indices, features, grad_out, need_grad_a=True,
                  need_grad_x=True, grad_x_dtype=torch.float32):
    """Returns [grad_a [E,H], grad_x [Ns,H,F]] (entry.cpp:92-104). A gradient
    that the caller does not need is skipped and returned as None. ``grad_x_dtype``:
    bfloat16 with bf16 ``grad_out`` rows writes grad_x as bf16 rows (fp32 sums)."""
    n_src, n_dst = features.size(0), indptr.numel() - 1
    native = _lib.ops()
    if grad_out.dtype == torch.bfloat16:
        # bf16 pipeline: gradient rows in bf16, fp32 sums and fp32 grad_x out. The edge
        # weights of such a pipeline are constants of the graph (norms): grad_a is not
        # offered, and the forward's features are not read at all.
        if need_grad_a:
            raise RuntimeError("spmm_backward with bf16 rows computes grad_x only "
                               "(need_grad_a=False): the reference's op is fp32")
        native.spmm_backward_check(values, indptr, indices, features, grad_out)
        if not need_grad_x:
            return [None, None]
        if n_dst > COL_MASK:
            raise RuntimeError("bf16 spmm_backward needs at most 2**24 destination rows")
        # grad_x[c] = sum over the edges of source c of values[e] * grad_out[row_e]: the
        # forward product over the by-source structure, weights copied into that order
        tr = transposed(indptr, indices, n_src)
        values_t = native.by_source_values(values, indptr, indices, n_src, True)
        return [None, spmm_forward(values_t, tr.t_indptr, tr.t_rows, grad_out,
                                   out_dtype=grad_x_dtype)]
    # before anything reads them: the by-source branch below hands grad_out to a forward
    # product that cannot know how many rows or columns it should have
    native.spmm_backward_check(values, indptr, indices, features, grad_out)
    if not (need_grad_a or need_grad_x):
        return [None, None]
    if grad_x_dtype != torch.float32:
        raise RuntimeError("grad_x_dtype other than float32 needs bf16 grad_out rows")
    tr = transposed(indptr, indices, n_src)
    if not need_grad_a and indices.numel() > 0 and n_dst <= COL_MASK:
        values_t = native.by_source_values(values, indptr, indices, n_src, False)
        if values_t is not None:
            # constant edge weights, seen before: grad_x is a forward product over the
            # by-source structure, its weights already in that order
            return [None, spmm_forward(values_t, tr.t_indptr, tr.t_rows, grad_out)]
    return list(native.spmm_backward(values, indptr, indices, features, grad_out, need_grad_a,
                                     need_grad_x, _lib.max_degree(indptr),
                                     _lib.row_plan(indptr, indices, n_src, COL_MASK), tr))


def edge_dot(indptr, indices, dst_feat, src_feat):
    """e[i,h] = <dst_feat[row_i,h,:], src_feat[col_i,h,:]> for every edge i: the
    SDDMM-dot inside spmm_backward (spmm_cuda.cu:33-35) as an op of its own."""
    return _lib.ops().edge_dot(indptr, indices, dst_feat, src_feat, _lib.max_degree(indptr),
                               _lib.row_plan(indptr, indices, src_feat.size(0), COL_MASK))


# --------------------------------------------------------------------------- #
# SDDMM + LeakyReLU + edge softmax
# --------------------------------------------------------------------------- #
def _sddmm_shapes(indptr, indices, query, key):
    _check(indptr, torch.int32, "indptr", 1)
    _check(indices, torch.int32, "indices", 1)
    _check(query, torch.float32, "query", 3)
    _check(key, torch.float32, "key", 2)
    if query.size(-1) != key.size(-1):
        raise RuntimeError("query and key disagree on the number of heads")
    if query.size(1) != indptr.numel() - 1:
        raise RuntimeError("query.size(1) must equal the number of destination rows")
    if query.size(0) > 16:
        raise RuntimeError("at most 16 query blocks (the block tag is 4 bits wide)")
    return indptr.numel() - 1, key.size(0), indices.numel(), key.size(1), query.size(0)


def sddmm_forward(indptr, indices, query, key):
    """attn[i,h] = softmax_{row, bid}(leaky_relu(query[bid,r,h] + key[col,h], 0.2)) (entry.cpp:106-116)."""
    plan = _lib.row_plan(indptr, indices, key.size(0), COL_MASK) if query.size(0) == 1 else None
    return _lib.ops().sddmm_forward(indptr, indices, query, key, _lib.max_degree(indptr), plan)


def sddmm_backward(indptr, indices, query, key, attn_values, grad_out, deterministic=True):
    """Returns [grad_query, grad_key] (entry.cpp:118-134). ``deterministic=False``
    selects the float-atomic scatter for grad_key (the reference's form)."""
    n_src = key.size(0)
    tr = transposed(indptr, indices, n_src) if deterministic else None
    plan = _lib.row_plan(indptr, indices, n_src, COL_MASK) \
        if query.size(0) == 1 and deterministic else None
    return list(_lib.ops().sddmm_backward(indptr, indices, query, key, attn_values, grad_out,
                                          _lib.max_degree(indptr), plan, tr))


# --------------------------------------------------------------------------- #
# horizontally fused SpMM || SDDMM
# --------------------------------------------------------------------------- #
def hfused_forward(spmm_values, spmm_indptr, spmm_indices, spmm_features, sddmm_indptr,
                   sddmm_indices, sddmm_query, sddmm_key):
    """An SpMM on graph A and an SDDMM+softmax on graph B with equal row counts
    (entry.cpp:136-155; hfused_cuda.cu:96-137) as one launch whose workgroups are split
    between the two ops (when neither graph has long rows; otherwise the two ops one
    after the other). Returns [spmm_out, attn]."""
    if spmm_indptr.numel() != sddmm_indptr.numel():
        raise RuntimeError("the two graphs must have the same number of rows")
    _check(spmm_values, torch.float32, "spmm_values", 2)
    _check(spmm_features, torch.float32, "spmm_features", 3)
    _check(sddmm_key, torch.float32, "sddmm_key", 2)
    if sddmm_query.dtype != torch.float32 or sddmm_query.dim() not in (2, 3):
        raise RuntimeError("sddmm_query must be float32 [n_dst, H] or [n_bid, n_dst, H]")
    for t, name in ((spmm_indptr, "spmm_indptr"), (spmm_indices, "spmm_indices"),
                    (sddmm_indptr, "sddmm_indptr"), (sddmm_indices, "sddmm_indices")):
        _check(t, torch.int32, name, 1)
    dev = _lib.require_device(spmm_values, spmm_indptr, spmm_indices, spmm_features, sddmm_indptr,
                              sddmm_indices, sddmm_query, sddmm_key)
    query = sddmm_query if sddmm_query.dim() == 3 else sddmm_query.unsqueeze(0)
    n_rows = spmm_indptr.numel() - 1
    n_src_a, h, f = spmm_features.shape
    n_bid = query.size(0)
    n_src_b = sddmm_key.size(0)
    nnz_a, nnz_b = spmm_indices.numel(), sddmm_indices.numel()
    if spmm_values.shape != (nnz_a, h):
        raise RuntimeError("spmm_values must be [n_edges, n_heads]")
    if query.size(1) != n_rows or query.size(2) != h or sddmm_key.size(1) != h:
        raise RuntimeError("query must be [n_bid, n_dst, H] and key [n_src, H] with the SpMM's H")
    if not 1 <= n_bid <= 16:
        raise RuntimeError("at most 16 query blocks (4-bit block tag)")
    out = torch.empty((n_rows, h, f), dtype=torch.float32, device=dev)
    attn = torch.zeros((nnz_b, h), dtype=torch.float32, device=dev)
    ws = _lib.workspace(_size_fn("yitu_hfused_forward_workspace_bytes")(
        c_i64(n_rows), c_i64(nnz_a), c_i64(h * f), c_i64(nnz_b), c_i64(h), c_i64(n_bid)), dev)
    with torch.cuda.device(dev):
        rc = _lib.lib().yitu_hfused_forward(
            ptr(out), ptr(attn), ptr(spmm_values), ptr(spmm_indptr), ptr(spmm_indices),
            ptr(spmm_features), ptr(sddmm_indptr), ptr(sddmm_indices), ptr(query), ptr(sddmm_key),
            c_i64(n_rows), c_i64(n_src_a), c_i64(nnz_a), c_i64(h), c_i64(f), c_i64(n_src_b),
            c_i64(nnz_b), c_i64(n_bid), c_i64(_lib.max_degree(spmm_indptr)),
            c_i64(_lib.max_degree(sddmm_indptr)), ptr(ws), c_size(ws.numel()), stream_ptr(dev))
    check(rc, "yitu_hfused_forward")
    return [out, attn]


def hfused_backward(spmm_values, spmm_indptr, spmm_indices, spmm_features, spmm_grad, sddmm_indptr,
                    sddmm_indices, sddmm_query, sddmm_key, sddmm_attn, sddmm_grad):
    """The two backward ops (entry.cpp:157-182) with the correct arithmetic, returning
    [grad_a, grad_x, grad_query, grad_key], in two launches shared by the two graphs: the
    per-row passes of both, then both by-source gathers (no atomics). Graphs with long rows
    run the two ops one after the other. The reference's fused backward kernel is
    unreachable (sparse.py:109-110) and indexes heads by threadIdx.x although they lie on
    threadIdx.y (hfused_cuda.cu:59,186)."""
    if spmm_indptr.numel() != sddmm_indptr.numel():
        raise RuntimeError("the two graphs must have the same number of rows")
    _check(spmm_values, torch.float32, "spmm_values", 2)
    _check(spmm_features, torch.float32, "spmm_features", 3)
    _check(spmm_grad, torch.float32, "spmm_grad", 3)
    _check(sddmm_attn, torch.float32, "sddmm_attn", 2)
    _check(sddmm_grad, torch.float32, "sddmm_grad", 2)
    n_rows, n_src_b, nnz_b, h, n_bid = _sddmm_shapes(sddmm_indptr, sddmm_indices, sddmm_query,
                                                     sddmm_key)
    dev = _lib.require_device(spmm_values, spmm_indptr, spmm_indices, spmm_features, spmm_grad,
                              sddmm_indptr, sddmm_indices, sddmm_query, sddmm_key, sddmm_attn,
                              sddmm_grad)
    n_src_a, h_a, f = spmm_features.shape
    nnz_a = spmm_indices.numel()
    if h_a != h or spmm_values.shape != (nnz_a, h) or spmm_grad.shape != (n_rows, h, f):
        raise RuntimeError("spmm_values must be [n_edges, H], spmm_grad [n_rows, H, F], with the "
                           "SDDMM's H")
    if sddmm_attn.shape != (nnz_b, h) or sddmm_grad.shape != (nnz_b, h):
        raise RuntimeError("sddmm_attn and sddmm_grad must be [n_edges, H]")
    ta = transposed(spmm_indptr, spmm_indices, n_src_a)
    tb = transposed(sddmm_indptr, sddmm_indices, n_src_b)
    grad_a = torch.empty_like(spmm_values)
    grad_x = torch.empty_like(spmm_features)
    grad_q = torch.empty_like(sddmm_query)
    grad_k = torch.empty_like(sddmm_key)
    grad_e = torch.empty_like(sddmm_attn)
    ws = _lib.workspace(_size_fn("yitu_hfused_backward_workspace_bytes")(
        c_i64(n_rows), c_i64(n_src_a), c_i64(nnz_a), c_i64(h * f), c_i64(n_src_b), c_i64(nnz_b),
        c_i64(h), c_i64(n_bid)), dev)
    with torch.cuda.device(dev):
        rc = _lib.lib().yitu_hfused_backward(
            ptr(grad_a), ptr(grad_x), ptr(grad_q), ptr(grad_k), ptr(grad_e), ptr(spmm_values),
            ptr(spmm_indptr), ptr(spmm_indices), ptr(spmm_features), ptr(spmm_grad.contiguous()),
            ptr(ta.t_indptr), ptr(ta.t_rows), ptr(ta.t_perm), ptr(sddmm_indptr), ptr(sddmm_indices),
            ptr(sddmm_query), ptr(sddmm_key), ptr(sddmm_attn), ptr(sddmm_grad.contiguous()),
            ptr(tb.t_indptr), ptr(tb.t_perm), c_i64(n_rows), c_i64(n_src_a), c_i64(nnz_a), c_i64(h),
            c_i64(f), c_i64(n_src_b), c_i64(nnz_b), c_i64(n_bid),
            c_i64(_lib.max_degree(spmm_indptr)), c_i64(ta.max_degree_t),
            c_i64(_lib.max_degree(sddmm_indptr)), c_i64(tb.max_degree_t), ptr(ws),
            c_size(ws.numel()), stream_ptr(dev))
    check(rc, "yitu_hfused_backward")
    return [grad_a, grad_x, grad_q, grad_k]


# --------------------------------------------------------------------------- #
# two Linear layers sharing one input
# --------------------------------------------------------------------------- #
def b2gemm(x, w_a, w_b):
    """Returns [y_a, y_b] = [x . w_a^T, x . w_b^T] (entry.cpp:56-64) on the matrix cores."""
    return _lib.ops().b2gemm(x, w_a, w_b)


def b2gemm_backward(x, w_a, w_b, grad_a, grad_b):
    """Returns [dx, dw_a, dw_b] (entry.cpp:66-78)."""
    return _lib.ops().b2gemm_backward(x, w_a, w_b, grad_a, grad_b)


def linear_forward(x, weight, bias=None):
    """x . weight^T + bias in fp32 on the matrix cores (``weight`` [n, k] as nn.Linear keeps
    it, ``bias`` [n] or None), the bias added inside the product where the kernel allows."""
    return _lib.ops().linear_forward(x, weight, bias)


def linear_forward_typed(x_list, weight_list, bias_list, out_list=None):
    """[x_i . weight_i^T + bias_i] for Linear layers that share both widths (the per-type
    layers of a heterogeneous model), up to 32 layers per launch. ``bias_list`` entries may be
    None. ``out_list``: contiguous [m_i, n] tensors to write (e.g. row slices of one buffer)."""
    return _lib.ops().linear_forward_typed(list(x_list), list(weight_list), list(bias_list), out_list)


def sgemm(a, b, trans_a=False, trans_b=False, out=None):
    """op(a) . op(b) in fp32 on the matrix cores; a, b contiguous 2-D. ``out``:
    a contiguous [m, n] tensor (e.g. a row slice of a larger buffer) to write."""
    return _lib.ops().sgemm(a, b, trans_a, trans_b, out)


def sgemm_typed(a_list, b_list, trans_a=False, trans_b=False, out_list=None):
    """[op(a_i) . op(b_i)] for operand pairs that share the output width, the
    transposes and the row strides (the per-type Linear layers of a heterogeneous
    model and their gradient products), up to 32 products per launch so that the
    row tiles of all types fill the chip together. ``out_list``: contiguous
    [m_i, n] tensors to write (e.g. row slices of one buffer)."""
    return _lib.ops().sgemm_typed(list(a_list), list(b_list), trans_a, trans_b, out_list)


def gemm_bf16(a, b, trans_b=False, out_dtype=torch.float32, out=None):
    """a . op(b) with bf16 operands and fp32 accumulation on the matrix cores.
    ``a`` [m, k]; ``b`` [k, n], or [n, k] with ``trans_b`` (a Linear weight).
    ``out``: a contiguous [m, n] fp32 or bf16 tensor to write (sets ``out_dtype``)."""
    return _lib.ops().gemm_bf16(a, b, trans_b, out_dtype, out)


def gemm_bf16_typed(a_list, b_list, trans_b=False, out_dtype=torch.float32, out_list=None):
    """[a_i . op(b_i)] with bf16 operands for pairs that share the widths (the per-type
    Linear layers of a heterogeneous model in bf16), eight products per launch.
    ``out_list``: contiguous [m_i, n] fp32 or bf16 tensors to write (e.g. row slices of
    one buffer; sets ``out_dtype``)."""
    return _lib.ops().gemm_bf16_typed(list(a_list), list(b_list), trans_b, out_dtype, out_list)


def gemm_bf16_tn(a, b, out=None, accumulate=False):
    """a^T . b for bf16 ``a`` [m, ki] and ``b`` [m, no] (rows may be strided slices of a
    wider buffer), fp32 accumulation on the matrix cores, fp32 [ki, no] out: the weight
    gradient X^T . dY of a bf16 layer. ``accumulate`` adds to ``out``."""
    return _lib.ops().gemm_bf16_tn(a, b, out, accumulate)


def gemm_bf16_tn_typed(a_list, b_list, out_list=None, accumulate=False):
    """[a_i^T . b_i] for bf16 pairs [m_i, ki], [m_i, no] of one shape (rows may be strided
    slices of wider buffers with a common row stride): the weight gradients of a
    heterogeneous bf16 layer, eight products per launch. fp32 [ki, no] outputs."""
    return _lib.ops().gemm_bf16_tn_typed(list(a_list), list(b_list), out_list, accumulate)


# --------------------------------------------------------------------------- #
# fused GAT attention (extension: the composition sddmm_forward -> spmm_forward)
# --------------------------------------------------------------------------- #
def gat_forward(indptr, indices, query, key, features, stats_only=False):
    """Returns [out [Nd,H,F], attn [E,H]] = the reference's two-op GAT lowering
    (sddmm_forward then spmm_forward, n_bid = 1) in one pass per destination row.
    ``stats_only``: returns [out, None, stats] instead, stats [Nd,H,2] = each row's
    softmax (max, 1 / sum): all that ``gat_backward`` needs of the attention for the
    one-pass shapes (``gat_one_pass_shape``); the probabilities are then never stored."""
    out, attn, stats = _lib.ops().gat_forward(
        indptr, indices, query, key, features, stats_only, _lib.max_degree(indptr),
        _lib.row_plan(indptr, indices, features.size(0), COL_MASK))
    return [out, None, stats] if stats_only else [out, attn]


def gat_one_pass_shape(n_heads, n_features, with_out=True):
    """Whether ``yitu_gat_backward`` takes its one-pass path for [*, H, F] rows (the
    shapes for which a head-mean gradient can be passed as it is)."""
    return _lib.ops().gat_one_pass_shape(n_heads, n_features)


def gat_backward(indptr, indices, query, key, features, attn, grad_out, out=None,
                 head_mean=False, stats=None):
    """Returns [grad_query, grad_key, grad_features] of gat_forward's ``out``.
    Passing the forward output ``out`` [n_dst, H, F] lets the softmax backward use
    sum_e a d_attn = <grad_out[row], out[row]> and finish in the same pass over
    the edges that computes grad_features (rows of 256, 512, 1024 floats); without
    it the attention gradient takes passes of its own.
    ``head_mean``: ``grad_out`` is [n_dst, F], the gradient of ``out.mean(dim=1)``
    (the layer's result, model.py:106); the pass then gathers F floats per edge.
    ``stats``: the row statistics of ``gat_forward(stats_only=True)``; ``attn`` may then
    be None (needs ``out`` and a one-pass shape)."""
    n_src = features.size(0)
    return list(_lib.ops().gat_backward(
        indptr, indices, query, key, features, attn, grad_out, out, head_mean, stats,
        _lib.max_degree(indptr), _lib.row_plan(indptr, indices, n_src, COL_MASK),
        transposed(indptr, indices, n_src)))


# --------------------------------------------------------------------------- #
# per-head projections (attention vectors)
# --------------------------------------------------------------------------- #
def head_dot_shape(n_heads, n_features):
    """Shapes the projection kernels take: head width 4 * a power of two up to 256,
    rows of at most 1024 floats."""
    lph = n_features // 4
    return (n_features % 4 == 0 and 1 <= lph <= 64 and lph & (lph - 1) == 0 and
            n_heads * n_features <= 1024)


def head_dot(x, vec_a, vec_b=None):
    """out_a[n,h] = <vec_a[h,:], x[n,h,:]> (and out_b with ``vec_b``): x [n,H,F],
    vec_* [H,F]. Returns (out_a, out_b or None)."""
    return _lib.ops().head_dot(x, vec_a, vec_b)


def head_dot_backward(x, vec_a, vec_b, grad_a, grad_b, grad_x=None):
    """Returns (grad_x, grad_vec_a, grad_vec_b). ``grad_x`` given: the projections'
    share is added to it in place (it holds the gradient that reached x by other
    paths); otherwise a new tensor is written."""
    return _lib.ops().head_dot_backward(x, vec_a, vec_b, grad_a, grad_b, grad_x)


# --------------------------------------------------------------------------- #
# Linear layers with few outputs
# --------------------------------------------------------------------------- #
def skinny_linear_shape(in_features, out_features):
    """Shapes the skinny product takes: at most 16 outputs, fewer for wide inputs."""
    return _lib.ops().skinny_linear_shape(in_features, out_features)


def skinny_linear(x, weight, bias=None):
    """x [n, K] . weight [J, K]^T + bias [J] for a handful of outputs J."""
    return _lib.ops().skinny_linear(x, weight, bias)


def skinny_linear_backward(x, weight, grad_y, grad_x=None, need_bias=True):
    """Returns (grad_x, grad_weight, grad_bias or None); a given ``grad_x`` is added to in place."""
    return _lib.ops().skinny_linear_backward(x, weight, grad_y, grad_x, need_bias)


def column_sum(x):
    """Sum over the rows of a 2-D fp32 tensor (a Linear's bias gradient), in a fixed order and
    without a cleared accumulator: safe to record into a HIP graph."""
    return _lib.ops().column_sum(x)


def column_sum_typed(x_list):
    """``[x_i.sum(0)]`` for 2-D fp32 tensors of one width whose rows are one common stride
    apart (row slices of one buffer): one launch per 32 of them when they are short (the bias
    gradients of the per-relation Linears of a small heterogeneous graph), otherwise
    ``column_sum`` each. Fixed summation order, no cleared accumulator."""
    return _lib.ops().column_sum_typed(list(x_list))
