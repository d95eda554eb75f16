"""Column sums of 16-bit rows behind a linear layer's bias gradient: one row, fewer rows than a workgroup
takes at a time, slices of unequal length, columns off the workgroup's 256, and layers whose
shapes leave the kernel (columns that are no multiple of 8)."""
import pytest
import torch

from megalodon_amd.modules.linear import Linear

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,cols", [(1, 8), (7, 256), (8, 264), (9, 2048), (1021, 1000), (4084, 520), (16391, 8), (3000, 4096),
                                       (5, 12)])
def test_bias_gradient(rows, cols, dtype):
    """Bar: the rounding of the result (8 or 11 significant bits: 2^-8 or 2^-11 of it) and float32 sums, `rows` half units in the
    last place of the sum of magnitudes."""
    torch.manual_seed(rows)
    layer = Linear(16, cols).cuda().to(dtype)
    x = torch.randn(rows, 16, device="cuda").to(dtype)
    dy = (torch.randn(rows, cols, device="cuda") + 0.25).to(dtype)
    layer(x).backward(dy)
    want, size = dy.double().sum(0), dy.double().abs().sum(0)
    step = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert bool(((layer.bias.grad.double() - want).abs() <= 1.01 * step * want.abs() + rows * 2.0 ** -24 * size).all())
