"""Edge list -> canonical CSR on the GPU through the C ABI (yitu_coo_to_csr):
rows ascending, columns ascending inside a row, duplicates merged, int32 -- what
``scipy.sparse.coo_matrix(...).tocsr()`` gives the reference
(YiTu_GNN/data/dataset.py:116-129)."""
import torch

from .. import _lib


def coo_to_csr(rows, cols, n_rows, n_cols=None):
    """``rows``, ``cols``: integer device tensors [E]. Returns (indptr int32
    [n_rows + 1], indices int32 [nnz]) on the same device."""
    n_cols = n_rows if n_cols is None else n_cols
    _lib.require_device(rows, cols)
    if rows.shape != cols.shape or rows.dim() != 1:
        raise RuntimeError("rows and cols must be 1-D and equally long")
    if rows.dtype != cols.dtype or rows.dtype not in (torch.int32, torch.int64):
        rows, cols = rows.to(torch.int64), cols.to(torch.int64)
    indptr, indices, info = _lib.ops().coo_to_csr(rows, cols, n_rows, n_cols)
    count, longest = info.tolist()
    if count < 0:
        raise RuntimeError("edge list holds a node id outside [0, n_rows) x [0, n_cols)")
    _lib.put_max_degree(indptr, longest)
    return indptr, indices[:count].clone()
