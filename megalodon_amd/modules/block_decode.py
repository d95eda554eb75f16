"""One new token through a block on a cache: the fused step of csrc/block_decode.hip where the
block has the standard structure, else None and the block goes operator by operator."""
from typing import Optional

import torch
from torch import Tensor
from torch.nn.modules import module as nn_module

from .. import _lib
from ..fused_ops import swift_efficient_attention
from .chunk_attention import _InnerAttention
from .complex_exponential_moving_average import MultiHeadComplexEMA
from .layer_norm import FusedLayerNorm, FusedRMSNorm
from .linear import Linear
from .normalized_feedforward_network import NormalizedFeedForwardNetwork
from .timestep_norm import TimestepNorm


def _unheard(module) -> bool:
    """Nobody listens to the module's forward or has put another in its place."""
    return not module._forward_hooks and not module._forward_pre_hooks and "forward" not in module.__dict__


def _plain(module, kind) -> bool:
    """`module` is exactly a `kind` whose own forward runs."""
    return type(module) is kind and _unheard(module)


def decode_step(block, x: Tensor, freqs_cis: Optional[Tensor], cache):
    """(out, cache) of `block(x, freqs_cis, None, cache)` for x (B, 1, D) without gradients in
    evaluation mode, or None.  The cache has to be a continued one: its first token goes
    through the operators."""
    cache_attn, cache_norm, hx = cache
    if cache_attn is None or hx is None or cache_norm[0] is None or cache_norm[1] is None or cache_norm[2] is None:
        return None
    keys, values, length = cache_attn
    mods = block._modules
    mega, nffn = mods["mega"], mods["nffn"]
    # (a cache is an unfinished chunk: what is longer is refused by the operators)
    if length < 1 or length >= mega.chunk_size or keys.shape[1] != length or not x.is_cuda:
        return None
    m, f = mega._modules, nffn._modules
    tsn, cema, rms, znorm, attn = m["timenorm"], m["cema"], m["rmsnorm"], m["znorm"], m["inner_attention"]
    wz, wr, wh1, wv, wh2 = m["wz"], m["wr"], m["wh1"], m["wv"], m["wh2"]
    ln, fc1, fc2, fc3 = f["norm"], f["fc1"], f["fc2"], f["fc3"]
    # (a submodule that is in training mode by itself has its dropouts, which the step does not)
    if (mega.training or nffn.training or attn.training or not _unheard(mega) or nn_module._global_forward_hooks
            or nn_module._global_forward_pre_hooks or not _plain(nffn, NormalizedFeedForwardNetwork)
            or nffn._parameters.get("alpha") is not None or fc3 is None
            or not _plain(tsn, TimestepNorm) or not _plain(cema, MultiHeadComplexEMA)
            or not _plain(rms, FusedRMSNorm) or not _plain(znorm, FusedRMSNorm) or znorm.elementwise_affine
            or not _plain(attn, _InnerAttention) or attn.attn_fn is not swift_efficient_attention or not _plain(ln, FusedLayerNorm)
            or any(not _plain(w, Linear) for w in (wz, wr, wh1, wv, wh2, fc1, fc2, fc3))
            or any(w._parameters["bias"] is not None for w in (wh2, fc1, fc2, fc3))):
        return None
    p, q, gamma = cema.coeffs()
    own = mega._parameters

    def weight(module):
        return module._parameters["weight"]

    def bias(module):
        return module._parameters["bias"]

    params = [weight(tsn), bias(tsn), cema._parameters["omega"], weight(rms), weight(wz), bias(wz), weight(wr), bias(wr),
              weight(wh1), bias(wh1), weight(wv), bias(wv), weight(wh2), own["gamma"], own["beta"],
              weight(ln), bias(ln), weight(fc1), weight(fc2), weight(fc3)]
    return _lib.host().block_decode_step(
        x, keys, values, *cache_norm, hx, freqs_cis, params, p, q, gamma, mega.num_heads, tsn.groups_per_partition,
        mega.chunk_size, tsn.eps, rms.eps, znorm.eps, ln.eps)
