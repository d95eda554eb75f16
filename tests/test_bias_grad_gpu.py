"""Column sums of 16-bit rows behind a linear layer's bias gradient: one row, fewer rows than a workgroup
takes at a time, slices of unequal length, columns off the workgroup's 256, and layers whose
shapes leave the kernel (columns that are no multiple of 8).  Both routes of the input's gradient."""
import pytest
import torch

from megalodon_amd.modules.linear import Linear, linear_group

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


@pytest.mark.parametrize("tokens,n_in,n_out", [(4096, 2048, 4096), (4097, 2048, 4096), (33, 64, 40)])  # 2^35 products and above
def test_input_gradient(tokens, n_in, n_out):
    """Bar: two roundings to bfloat16 of a value of the result's size, 2^-8 in the 2-norm."""
    torch.manual_seed(tokens)
    layers = [Linear(n_in, n_out).cuda().bfloat16(), Linear(n_in, n_out, bias=False).cuda().bfloat16()]
    x = torch.randn(tokens, n_in, device="cuda").bfloat16()
    dy = [torch.randn(tokens, n_out, device="cuda").bfloat16() for _ in layers]
    one, two = x.clone().requires_grad_(True), x.clone().requires_grad_(True)
    layers[0](one).backward(dy[0])
    outs = linear_group(two, layers)
    torch.autograd.backward(outs, dy)
    first = dy[0].float() @ layers[0].weight.float()
    both = first + dy[1].float() @ layers[1].weight.float()
    for got, want in ((one.grad, first), (two.grad, both)):
        assert (got.float() - want).norm() <= 2.0 ** -8 * want.norm()
