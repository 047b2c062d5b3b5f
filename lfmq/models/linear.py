"""Dense projections of the GPU models."""
from __future__ import annotations

import torch.nn as nn

from ..ops import functional as F


class Linear(nn.Linear):
    """nn.Linear without a bias whose decode steps run on the kernel for a
    few rows."""

    def __init__(self, n_in: int, n_out: int, dtype):
        super().__init__(n_in, n_out, bias=False, dtype=dtype)

    def forward(self, x):
        if self.bias is not None:
            return super().forward(x)
        return F.linear(x, self.weight)


def hooked(*modules) -> bool:
    """Whether anyone watches calls of these modules, or has put a forward of
    an instance's own in their way."""
    m = nn.modules.module
    return bool(m._global_forward_hooks or m._global_forward_pre_hooks
                or any(p._forward_hooks or p._forward_pre_hooks
                       or "forward" in p.__dict__ for p in modules))
