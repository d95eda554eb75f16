"""Both sides of the lines between the two scores kernels (blocks of 32 rows a compute unit, by head width, keys and mask): a pair
among as many copies as the line allows and among one more gives what it gives alone, up to single roundings, and alone
what float32 gives."""
import math

import pytest
import torch

from conftest import rel_err
from megalodon_amd.fused_ops import swift_efficient_attention
from test_attention_any_length_gpu import _reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H1,R,L,eighths,causal,dtype", [
    (64, 384, 384, 32, True, torch.bfloat16), (64, 416, 416, 44, True, torch.float16), (64, 1025, 1025, 44, True, torch.bfloat16),
    (128, 100, 100, 24, True, torch.bfloat16), (128, 513, 513, 32, True, torch.bfloat16), (128, 200, 200, 16, False, torch.float16),
    (256, 128, 128, 10, True, torch.float16), (256, 256, 256, 16, True, torch.bfloat16), (256, 700, 700, 24, True, torch.float16),
    (256, 1280, 1280, 24, True, torch.bfloat16), (256, 2049, 2049, 26, True, torch.bfloat16),
    # more keys than rows, and without a mask
    (64, 100, 1100, 44, True, torch.bfloat16), (64, 200, 600, 40, True, torch.bfloat16), (128, 200, 333, 24, True, torch.float16), (256, 700, 1100, 24, True, torch.bfloat16),
    (64, 512, 512, 26, False, torch.bfloat16), (64, 300, 1000, 40, False, torch.float16), (128, 500, 700, 24, False, torch.bfloat16),
    (256, 200, 200, 8, False, torch.bfloat16), (256, 999, 400, 16, False, torch.float16),
])
def test_both_sides_of_a_line(H1, R, L, eighths, causal, dtype):
    g = torch.Generator().manual_seed(L + H1)
    q, k = (torch.randn(1, n, 1, H1, generator=g).to(dtype) for n in (R, L))
    v, dy = (torch.randn(1, n, 1, 64, generator=g).to(dtype) for n in (L, R))
    scale = 1.5 / math.sqrt(H1)

    def run(copies):
        leaves = [t.cuda().repeat(copies, 1, 1, 1).requires_grad_(True) for t in (q, k, v)]
        y = swift_efficient_attention(*leaves, scale, 0.0, causal, True)
        y.backward(dy.cuda().repeat(copies, 1, 1, 1))
        return [y.detach()] + [t.grad for t in leaves]

    alone = run(1)
    for got, want in zip(alone, _reference(q, k, v, dy, scale, causal)):
        assert rel_err(got, want) <= 2e-2
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    last = eighths * cus // 8 // -(-R // 32)
    for copies in (last, last + 1):
        for a, m in zip(alone, run(copies)):
            assert torch.equal(m[:1].expand_as(m), m)
            # probabilities, dP and dS are rounded to 16 bits once, from float32 sums in another order: 2^-9 of single terms
            assert (m[:1].float() - a.float()).norm() <= 2 ** -9 * a.float().norm()
