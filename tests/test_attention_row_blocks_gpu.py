"""Few (batch, head) pairs and many of them take different kernels (scores in row blocks of 32 with the keys shared out
over a workgroup's waves, products in tiles of 128): every pair of a large batch of copies has to give what
one pair alone gives, at the edges of blocks, tiles, pieces of keys and of what a wave holds, and one alone what
float32 gives."""
import math

import pytest
import torch

from conftest import rel_err
from megalodon_amd.fused_ops import swift_efficient_attention
from test_attention_any_length_gpu import _reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L1,L2,NH,H1,H2,causal,dtype", [
    (31, 31, 1, 64, 64, True, torch.bfloat16),
    (129, 129, 2, 128, 136, True, torch.float16),        # one row behind a tile of 128
    (256, 256, 1, 256, 128, True, torch.bfloat16),
    (384, 384, 2, 64, 64, True, torch.bfloat16),         # an odd number of tiles of 128
    (300, 333, 1, 128, 200, True, torch.bfloat16),       # keys in front, both lengths off the slabs
    (1024, 1024, 1, 256, 256, True, torch.bfloat16),     # four blocks of keys per wave
    (1025, 1025, 1, 256, 264, True, torch.float16),      # one key more
    (2048, 2048, 1, 128, 64, True, torch.bfloat16),      # eight
    (2049, 2049, 1, 256, 128, True, torch.bfloat16),     # a second piece of one key
    (64, 4096, 1, 64, 512, True, torch.bfloat16),        # two whole pieces, keys in front
    (33, 2100, 2, 256, 64, False, torch.float16),        # two pieces, every key for every query
    (4096, 4096, 1, 64, 64, True, torch.bfloat16),
    (70, 5000, 1, 64, 128, True, torch.bfloat16),        # three pieces
])
def test_one_pair_alone_and_among_many(L1, L2, NH, H1, H2, causal, dtype):
    g = torch.Generator().manual_seed(L1 + L2)
    q, dy = torch.randn(1, L1, NH, H1, generator=g).to(dtype), torch.randn(1, L1, NH, H2, generator=g).to(dtype)
    k, v = torch.randn(1, L2, NH, H1, generator=g).to(dtype), torch.randn(1, L2, NH, H2, generator=g).to(dtype)
    scale = 1.5 / math.sqrt(H1)

    def run(copies):
        leaves = [t.cuda().repeat(copies, 1, 1, 1).requires_grad_(True) for t in (q, k, v)]
        y = swift_efficient_attention(*leaves, scale, 0.0, causal, True)
        y.backward(dy.cuda().repeat(copies, 1, 1, 1))
        return [y.detach()] + [t.grad for t in leaves]

    alone = run(1)
    for got, want in zip(alone, _reference(q, k, v, dy, scale, causal)):
        assert rel_err(got, want) <= 2e-2
    many = run(min(200, -(-900 // (NH * -(-L1 // 32)))))
    for a, m in zip(alone, many):
        assert torch.equal(m[:1].expand_as(m), m)
        # the same operands and sums in float32 in another order; probabilities, dP and dS each rounded to 16 bits
        # once, so a rounding may fall the other way: half a unit of the last place, 2^-9, of single terms
        assert (m[:1].float() - a.float()).norm() <= 2 ** -9 * a.float().norm()
