"""Which norms of the one-token step come on the products' way and which ahead of them (csrc/block_decode.hip: run): both sides of
each line, with row counts that a workgroup's four or sixteen rows divide just so.  Against the step in 64 bits; bars as in
test_block_decode_gpu."""
import pytest
import torch

from test_block_decode_rows_gpu import test_step_against_float64 as step_against_float64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,D,S,E,F,heads,groups,dtype", [
    (1, 4096, 64, 64, 96, 1, 8, torch.bfloat16),        # both ahead
    (1, 4064, 64, 128, 32, 1, 127, torch.float16),
    (1, 3104, 64, 64, 32, 1, 97, torch.bfloat16),       # the first width with both ahead
    (1, 3072, 64, 128, 32, 1, 8, torch.float16),        # the second alone
    (2, 4096, 64, 64, 32, 1, 8, torch.bfloat16),
    (4, 3104, 64, 64, 32, 1, 97, torch.float16),        # the shortest row of four pieces a wave
    (4, 2080, 128, 128, 160, 2, 65, torch.bfloat16),    # the first width with the second ahead
    (4, 2048, 128, 128, 160, 2, 8, torch.float16),      # the last without
])
def test_step_against_float64(B, D, S, E, F, heads, groups, dtype):
    step_against_float64(B, D, S, E, F, heads, groups, dtype)
