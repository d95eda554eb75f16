"""The transform path takes a channel's rows in pairs, and shares them out over workgroups where there are few channels:
batches of one, of pairs and an odd rest, channels with one, several and all of their rows in a workgroup, against
64 bits; tolerance of the float32 transforms, 2e-6, behind the rounding of 16-bit rows, 2^-8 (float16 2^-11)."""
import pytest
import torch

from megalodon_amd.fused_ops import fftconv

pytestmark = pytest.mark.gpu


def _conv(a, b):
    n = 2 * a.shape[-1]
    return torch.fft.irfft(torch.fft.rfft(a, n) * torch.fft.rfft(b, n), n)[..., :a.shape[-1]]


@pytest.mark.parametrize("B,D,L,dtype", [
    (1, 3, 2049, torch.float32), (2, 5, 4096, torch.float32), (3, 1100, 2050, torch.bfloat16),
    (7, 130, 4097, torch.float32), (5, 400, 6000, torch.float16), (9, 256, 8192, torch.bfloat16),
    (4, 1030, 5001, torch.bfloat16), (6, 100, 16384, torch.float32), (3, 300, 9999, torch.bfloat16),
    (5, 64, 32768, torch.float32), (2, 257, 20001, torch.bfloat16), (3, 700, 5001, torch.float16), (5, 420, 8191, torch.float32),
])
def test_against_64_bits(B, D, L, dtype):
    g = torch.Generator("cuda").manual_seed(B * D + L)
    x = torch.randn(B, D, L, generator=g, device="cuda").to(dtype).requires_grad_(True)
    dy = torch.randn(B, D, L, generator=g, device="cuda").to(dtype)
    t = torch.arange(L, device="cuda")
    k = (torch.randn(D, L, generator=g, device="cuda") * torch.exp(-0.01 * t)).requires_grad_(True)
    y = fftconv(x, k)
    y.backward(dy)
    x64, k64, dy64 = x.detach().double(), k.detach().double(), dy.double().flip(-1)
    step = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for got, want, tol in ((y, _conv(x64, k64), step + 2e-6), (x.grad, _conv(dy64, k64).flip(-1), step + 2e-6),
                           (k.grad, sum(_conv(dy64[b], x64[b]) for b in range(B)).flip(-1), 2e-6)):
        assert (got.double() - want).norm() <= tol * want.norm()
    # every row by itself gives the same outputs but for what the compiler contracts, and the same each time
    with torch.no_grad():
        assert torch.equal(fftconv(x, k), y)
        alone = torch.cat([fftconv(x[b:b + 1].detach(), k) for b in range(B)])
    assert (alone.double() - y.double()).norm() <= (step + 1e-6) * y.double().norm()
