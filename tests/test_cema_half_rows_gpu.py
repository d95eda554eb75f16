"""The EMA layer's backward on float16 rows as they are: x and dy near the type's two ends, and lags of k whose largest is
far from one or none at all.

Bars: dx is rounded once (2^-12 of its norm, below 2^-14 2^-25 of each value: 5e-4 of the norm and 2^-25 of the root of the
count); the parameters' gradients are float32 sums of products with 22 bits
(measured 1e-7 .. 4e-6 relative to 64 bits, 1e-5 with the float32 coefficients)."""
import pytest
import torch

from megalodon_amd.modules import MultiHeadComplexEMA
from oracle import cema as ocema, fftconv as offt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,gamma,omega,up", [(1.0, 1.0, 1.0, 1.0), (2.0 ** -18, 1.0, 1.0, 1.0), (1000.0, 1.0, 1.0, 1.0),
                                                 (1.0, 2.0 ** -14, 0.0, 1.0), (1.0, 0.0, 1.0, 1.0), (1.0, 0.0, 0.0, 1.0),
                                                 (2.0 ** -8, 500.0, 0.1, 1.0), (2.0 ** -8, 1.0, 1000.0, 1.0),
                                                 (1.0, 1.0, 1.0, 2.0 ** -18), (2.0 ** -18, 30.0, 100.0, 2.0 ** -18),
                                                 (1.0, 0.1, 0.1, 2.0 ** 12), (8000.0, 0.05, 0.5, 2.0 ** 13)])
@pytest.mark.parametrize("B,D,L", [(2, 3, 2056), (3, 4, 777), (1, 8, 8193)])
def test_backward_matches_float64(B, D, L, rows, gamma, omega, up):
    torch.manual_seed(L)
    layer = MultiHeadComplexEMA(D, 16).cuda().train()
    with torch.no_grad():
        layer.gamma.mul_(gamma)
        layer.omega.copy_(omega * torch.randn_like(layer.omega))
    x0, dy0 = (rows * torch.randn(B, D, L)).half(), (up * torch.randn(B, D, L)).half()
    x = x0.cuda().requires_grad_(True)
    layer(x)[0].backward(dy0.cuda())
    pr = {n: p.detach().cpu().double().requires_grad_(True) for n, p in layer.named_parameters()}
    xo = x0.double().requires_grad_(True)
    p, q, g = ocema.calc_coeffs(pr["alpha"], pr["delta"], pr["theta"], pr["gamma"], 16)
    want = offt.fftconv_fwd(xo, ocema.ema_weight_fwd(p, q.log(), g, L)) + xo * pr["omega"]
    want.backward(dy0.double())

    def err(got, ref):
        norm = ref.norm()
        return ((got.detach().cpu().double() - ref).norm() / (norm if norm > 0 else 1.0)).item()

    assert x.grad.dtype == torch.float16
    assert (x.grad.cpu().double() - xo.grad).norm() <= 5e-4 * xo.grad.norm() + 2.0 ** -25 * xo.grad.numel() ** 0.5
    for n, prm in layer.named_parameters():
        assert err(prm.grad, pr[n].grad) <= 1e-5, n
