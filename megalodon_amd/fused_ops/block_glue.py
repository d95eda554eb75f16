"""The block's memory-bound glue as differentiable operators.

The reference writes these steps as plain PyTorch expressions
(megalodon/modules/moving_average_gated_attention.py:299-300,314,319-336,
megalodon/modules/normalized_feedforward_network.py:82,
megalodon/modules/layer_norm.py:30-33,62-65,
megalodon/modules/rotary_positional_embedding.py:53-77); here each is one
streaming kernel forward and one backward, and the autograd nodes are C++
(csrc/host/ops.cpp)."""
from typing import Optional, Tuple

import torch

from .. import _lib


def transpose_last2(x: torch.Tensor) -> torch.Tensor:
    """`x.transpose(-2, -1).contiguous()`; the gradient is the same move back."""
    return _lib.host().transpose_last2(x)


def silu_mul(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """`F.silu(a) * b`; keeps (a, b) for the backward."""
    return _lib.host().silu_mul(a, b)


def layer_norm_plus_one(x: torch.Tensor, weight: Optional[torch.Tensor], bias: Optional[torch.Tensor],
                        eps: float = 1e-5, rms: bool = False) -> torch.Tensor:
    """LayerNorm / RMSNorm over the last axis whose stored weight is gamma - 1."""
    return _lib.host().layer_norm_plus_one(x, weight, bias, eps, rms)


def qk_norm_rotary(z: torch.Tensor, gamma: torch.Tensor, beta: torch.Tensor, freqs_cis: Optional[torch.Tensor],
                   head_dim: int, eps: float) -> Tuple[torch.Tensor, torch.Tensor]:
    """z -> (q, k) in one pass: per-head norm, both affine maps, the rotary product."""
    return _lib.host().qk_norm_rotary(z, gamma, beta, freqs_cis, head_dim, eps)
