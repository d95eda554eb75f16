"""The lines between the two scores kernels where the one for few row blocks reads its keys by whole cache lines: both sides of each,
as test_attention_scores_rule_gpu checks them."""
import pytest
import torch

import test_attention_scores_rule_gpu as rule

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H1,R,L,eighths,causal,dtype", [
    (64, 384, 384, 42, True, torch.bfloat16), (64, 385, 385, 48, True, torch.float16),
    (128, 72, 72, 14, True, torch.bfloat16), (128, 544, 544, 32, True, torch.float16), (128, 768, 768, 28, True, torch.bfloat16),
    (128, 769, 769, 36, True, torch.bfloat16),
    (256, 64, 64, 8, True, torch.bfloat16), (256, 128, 128, 16, True, torch.float16), (256, 384, 384, 19, True, torch.bfloat16),
    (256, 768, 768, 22, True, torch.bfloat16), (256, 1152, 1152, 28, True, torch.bfloat16), (256, 2049, 2049, 34, True, torch.float16),
    (64, 100, 2049, 27, True, torch.bfloat16), (64, 128, 300, 47, True, torch.bfloat16), (128, 600, 1100, 32, True, torch.float16),
    (128, 300, 600, 25, True, torch.bfloat16), (256, 600, 1100, 33, True, torch.bfloat16), (256, 300, 600, 22, True, torch.bfloat16),
    (64, 100, 512, 47, False, torch.bfloat16), (64, 700, 700, 33, False, torch.float16), (64, 200, 1100, 41, False, torch.bfloat16),
    (64, 300, 1200, 32, False, torch.bfloat16), (128, 700, 700, 22, False, torch.bfloat16), (128, 200, 800, 27, False, torch.float16),
    (256, 300, 384, 16, False, torch.bfloat16), (256, 500, 768, 20, False, torch.bfloat16), (256, 300, 1500, 24, False, torch.float16),
    (256, 100, 1600, 20, False, torch.bfloat16),
])
def test_both_sides_of_a_line(H1, R, L, eighths, causal, dtype):
    rule.test_both_sides_of_a_line(H1, R, L, eighths, causal, dtype)
