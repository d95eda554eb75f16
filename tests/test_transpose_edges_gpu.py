"""16-bit transposes in large tiles whose last pieces of eight are cut: every remainder of both sides, bit for bit."""
import pytest
import torch

from megalodon_amd.fused_ops import transpose_last2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,C", [(2048 + i, 2176 - j) for i, j in ((0, 1), (1, 2), (2, 3), (3, 4), (4, 5), (5, 6), (6, 7), (7, 0), (1, 127))])
def test_cut_pieces(R, C):
    x = torch.randint(-2 ** 15, 2 ** 15, (1, R, C), dtype=torch.int16, device="cuda").view(torch.bfloat16)
    y = transpose_last2(x)
    assert torch.equal(y.view(torch.int16), x.view(torch.int16).transpose(1, 2))
