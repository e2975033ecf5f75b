"""RMSNorm with the arithmetic of nanoquantization/layers/norm.py:10-35: normalise in fp32, cast back
to the input dtype, then multiply by the weight in that dtype.  One kernel where no gradient is wanted,
torch operations otherwise."""
from __future__ import annotations

import torch
from torch import nn

from .. import _lib
from .inference import keeps, plain, shipped


@shipped("forward", "rms_norm")
class RMSNorm(nn.Module):
    def __init__(self, norm_size: int, eps: float = 1e-6) -> None:
        super().__init__()
        self.norm_size = norm_size
        self.eps = eps
        self.weight = nn.Parameter(torch.ones(norm_size))

    def rms_norm(self, x: torch.Tensor) -> torch.Tensor:
        xf = x.float()
        xf = xf * torch.rsqrt(xf.pow(2).mean(dim=-1, keepdim=True) + self.eps)
        return xf.to(x.dtype) * self.weight

    def _one_kernel(self, x: torch.Tensor) -> bool:
        # a workgroup per row: rows of a few hundred elements (the heads') leave most of it idle
        return (type(self) is RMSNorm and plain(x, self.weight) and keeps(self, RMSNorm, "rms_norm") and 512 <= self.weight.numel() <= 8192
                and self.weight.numel() % 8 == 0 and x.shape[-1:] == self.weight.shape)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        if not torch.jit.is_scripting():
            if self._one_kernel(x):
                return _lib.torch_ops().rms_norm(x, self.weight, self.eps)
        return self.rms_norm(x)
