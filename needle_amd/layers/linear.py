"""nn.Linear whose few-row calls (a decode step) run ops.linear's weight-streaming kernel.

Parameters, names, state dict and results up to the order of the fp32 sums are nn.Linear's
(the reference's projections, needle/layers/attention.py:84-96, needle/model/llama.py:36-37).
"""
from __future__ import annotations

import torch
import torch.nn as nn

from .. import ops


class Linear(nn.Linear):
    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return ops.linear(x, self.weight, self.bias)
