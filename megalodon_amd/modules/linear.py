"""`nn.Linear` on the attention operator's product kernels where they are expected to be ahead of the library GEMMs.

With model-parallel world size 1 the reference's Column/RowParallelLinear are
`F.linear` (megalodon/modules/model_parallel/layers.py:222-235,321-341).  Weight gradients, and the
forward products and input gradients that an estimate by sizes (csrc/linear_plan.hpp) finds faster there, run on these kernels,
layers of one input together; the other products are library GEMMs.  Those of `dx = dy @ W` with W (out, in) read along its rows are
13-24 % faster on MI355X when both operands run along the reduction axis (`dy @ Wt^T` with Wt = W^T contiguous, the
layout the forward `x @ W^T` uses), and the tiled transpose of W costs 5-30 us, so the backward makes that copy where the
product is large enough to win it back.  The autograd nodes are C++ (csrc/host/ops.cpp).
Values are those of `F.linear`; parameters keep the names and shapes of
`nn.Linear`, so state dicts are interchangeable."""
from typing import Optional, Tuple

import torch
import torch.nn.functional as F
from torch import nn

from .. import _lib


def linear_group(x: torch.Tensor, layers) -> Tuple[torch.Tensor, ...]:
    """`tuple(layer(x) for layer in layers)` for `Linear` layers that read the same input; on the GPU in
    16 bits their products are one launch where that is the faster form, and with gradients their backward
    shares one input-gradient accumulation.  Without gradients only for layers whose call is nothing but
    `Linear.forward`: no hooks of their own or for all modules."""
    layers = list(layers)
    fused = (x.is_cuda and x.dtype in (torch.bfloat16, torch.float16)
             and all(l.weight.dtype == x.dtype for l in layers))
    if fused and not (torch.is_grad_enabled() and (x.requires_grad or any(l.weight.requires_grad for l in layers))):
        fused = all(type(l) is Linear and "forward" not in l.__dict__ and not l._forward_hooks and not l._forward_pre_hooks for l in layers) \
            and not torch.nn.modules.module._global_forward_hooks and not torch.nn.modules.module._global_forward_pre_hooks
    if not fused or len(layers) < 2:
        return tuple(l(x) for l in layers)
    params, has_bias = [], []
    for l in layers:
        params.append(l.weight)
        has_bias.append(l.bias is not None)
        if l.bias is not None:
            params.append(l.bias)
    return tuple(_lib.host().linear_group(x, params, has_bias))


class Linear(nn.Linear):
    """Drop-in for `nn.Linear` (same parameters, same values); `residual`, for
    layers without bias, is added inside the GEMM."""

    def forward(self, x: torch.Tensor, residual: Optional[torch.Tensor] = None) -> torch.Tensor:
        fused = (x.is_cuda and x.dtype in (torch.bfloat16, torch.float16) and self.weight.dtype == x.dtype)
        if residual is not None and (self.bias is not None or not fused or residual.dtype != x.dtype):
            return F.linear(x, self.weight, self.bias) + residual
        if fused:
            return _lib.host().linear(x, self.weight, self.bias, residual)
        return F.linear(x, self.weight, self.bias)
