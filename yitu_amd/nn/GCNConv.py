"""GCN layer over ``YiTu_GNN_kernel.forward / backward`` (the role of
YiTu_GNN/nn/GCNConv.py:13-76)."""
from .. import _lib
from ._common import DenseWeight


class GNNAFunction:
    """``apply(X, weight, inputInfo)`` -> normalised aggregation of ``X . weight``, one
    autograd node (csrc/bind/autograd.cpp). ``inputInfo`` carries row_pointers, column_index,
    degrees, partPtr, part2Node, partSize, dimWorker, warpPerBlock (GCNConv.py:27-34) and,
    when ``prepare_edge_scale`` was called, the per-edge column scales."""

    @staticmethod
    def apply(X, weight, inputInfo):
        return _lib.ops().gcn_conv(X, weight, inputInfo.row_pointers, inputInfo.column_index,
                                   inputInfo.degrees, inputInfo.partPtr, inputInfo.part2Node,
                                   getattr(inputInfo, "edge_scale", None))


class GCNConv(DenseWeight):
    """``forward(X, inputInfo)`` with ``weights`` [input_dim, output_dim]."""

    def forward(self, X, inputInfo):
        return GNNAFunction.apply(X, self.weights, inputInfo)
