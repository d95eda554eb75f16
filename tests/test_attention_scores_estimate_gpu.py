"""Both sides of where the estimate puts the line between the two scores kernels, and rows with fewer keys than the short-row kernel has
waves or one block for each, as test_attention_scores_rule_gpu checks them."""
import pytest
import torch

import test_attention_scores_rule_gpu as rule

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H1,R,L,eighths,causal,dtype", [
    (64, 200, 200, 74, False, torch.bfloat16), (64, 512, 512, 43, False, torch.float16), (64, 600, 3000, 44, False, torch.bfloat16),
    (128, 160, 160, 37, True, torch.bfloat16), (128, 435, 2471, 38, True, torch.float16), (128, 1025, 1025, 59, True, torch.bfloat16),
    (256, 33, 33, 8, True, torch.bfloat16), (256, 160, 160, 21, True, torch.float16), (256, 512, 512, 21, False, torch.bfloat16),
    (64, 33, 33, 20, True, torch.bfloat16), (64, 32, 160, 24, False, torch.float16), (128, 1, 17, 12, False, torch.bfloat16),
    (128, 40, 255, 12, True, torch.bfloat16), (256, 5, 257, 8, False, torch.bfloat16), (256, 1, 1, 8, True, torch.float16),
])
def test_both_sides_of_a_line(H1, R, L, eighths, causal, dtype):
    rule.test_both_sides_of_a_line(H1, R, L, eighths, causal, dtype)
