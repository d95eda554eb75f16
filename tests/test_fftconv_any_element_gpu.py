"""Rows of the convolution operator that lie at any element: odd lengths, and tensors off the 8-byte boundary of their
storage.  Everything around them is NaN, so a value taken from outside a row shows in it."""
import pytest
import torch

from megalodon_amd.fused_ops import fftconv

pytestmark = pytest.mark.gpu


def _inside(shape, dtype, offset, seed):
    n = 1
    for s in shape:
        n *= s
    store = torch.full((n + 64,), float("nan"), dtype=dtype, device="cuda")
    gen = torch.Generator("cuda").manual_seed(seed)
    view = store[32 + offset:32 + offset + n].view(shape)
    view.copy_(torch.randn(shape, generator=gen, device="cuda"))
    return view


def _conv(a, b):
    n = 2 * a.shape[-1]
    return torch.fft.irfft(torch.fft.rfft(a, n) * torch.fft.rfft(b, n), n)[..., :a.shape[-1]]


# float32: 1e-5, the engine's bar at every length (measured below 1e-6); 16 bits: an element's rounding, 2^-9 and 2^-12
@pytest.mark.parametrize("dtype,bar", [(torch.float32, 1e-5), (torch.bfloat16, 4e-3), (torch.float16, 5e-4)])
@pytest.mark.parametrize("B,D,L,offset", [(1, 2, 2049, 0), (2, 3, 2050, 1), (3, 2, 4095, 3), (2, 2, 4097, 0), (5, 1, 8191, 2),
                                          (2, 2, 8194, 1), (1, 3, 16385, 1), (3, 1, 32767, 0), (2, 1, 32768, 3)])
def test_rows_at_any_element(B, D, L, offset, dtype, bar):
    x = _inside((B, D, L), dtype, offset, L).requires_grad_(True)
    k = _inside((D, L), torch.float32, offset, L + 1).mul_(L ** -0.5).requires_grad_(True)
    dy = _inside((B, D, L), dtype, offset, L + 2)
    y = fftconv(x, k)
    y.backward(dy)
    xd, kd, gd = x.detach().double(), k.detach().double(), dy.double()
    want = (_conv(xd, kd), _conv(gd.flip(-1), kd).flip(-1), _conv(gd.flip(-1), xd).sum(0).flip(-1))
    for got, ref, lim in zip((y.detach(), x.grad, k.grad), want, (bar, bar, 1e-5)):
        assert torch.isfinite(got).all()
        assert ((got.double() - ref).norm() / ref.norm()).item() <= lim
