"""GIN layer over ``YiTu_GNN_kernel.forward_gin / backward_gin`` (the role of
YiTu_GNN/nn/GINConv.py)."""
from .. import _lib
from ._common import DenseWeight


class GNNAFunction_GIN:
    """``apply(X, weight, inputInfo, eplison)`` -> ``(eplison * sum of neighbours) . weight``,
    one autograd node (csrc/bind/autograd.cpp). The aggregate that ``forward_gin`` returns
    beside the output is what the backward needs in place of X (GINConv.py:24), so X itself
    is not kept."""

    @staticmethod
    def apply(X, weight, inputInfo, eplison):
        return _lib.ops().gin_conv(X, weight, inputInfo.row_pointers, inputInfo.column_index,
                                   eplison, inputInfo.partPtr, inputInfo.part2Node)


class GINConv(DenseWeight):
    """``forward(X, inputInfo)``; the neighbour sum is scaled by ``eplison`` = 0.5,
    a constant of the layer as in the reference (GINConv.py:62)."""

    def __init__(self, input_dim, output_dim):
        super().__init__(input_dim, output_dim)
        self.eplison = 0.5

    def forward(self, X, inputInfo):
        return GNNAFunction_GIN.apply(X, self.weights, inputInfo, self.eplison)
