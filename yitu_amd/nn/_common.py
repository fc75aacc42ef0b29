"""What the two conv layers share: the weight and its initialisation."""
import math

import torch

class DenseWeight(torch.nn.Module):
    """A [input_dim, output_dim] parameter named ``weights`` drawn from
    U(-1/sqrt(output_dim), 1/sqrt(output_dim)) (GCNConv.py:58-66, GINConv.py:58-67)."""

    def __init__(self, input_dim, output_dim):
        super().__init__()
        # drawn, then redrawn by reset_parameters, like the reference: a seeded run
        # consumes the generator the same way
        self.weights = torch.nn.Parameter(torch.randn(input_dim, output_dim))
        self.reset_parameters()

    def reset_parameters(self):
        bound = 1.0 / math.sqrt(self.weights.size(1))
        with torch.no_grad():
            self.weights.uniform_(-bound, bound)
