"""The EMA layer's backward on float16 rows where omega is 2^29 times the lags of k beside it: a step of dy in front of which
dy is zero shows the lags alone.

Bar: dx is rounded once (2^-12 of its norm, in the subnormals 2^-25 of each value at most); the lags' 17 bits or more
are far below that."""
import pytest
import torch

from megalodon_amd.modules import MultiHeadComplexEMA
from oracle import cema as ocema

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,D,L", [(2, 3, 2056), (3, 4, 777), (1, 8, 8193)])
def test_lags_beside_a_large_omega(B, D, L):
    torch.manual_seed(L)
    layer = MultiHeadComplexEMA(D, 16).cuda().train()

    def lags():
        prm = {n: p.detach().cpu().double() for n, p in layer.named_parameters()}
        p, q, g = ocema.calc_coeffs(prm["alpha"], prm["delta"], prm["theta"], prm["gamma"], 16)
        return ocema.ema_weight_fwd(p, q.log(), g, L)

    with torch.no_grad():
        layer.omega.fill_(2.0 ** 15)
        layer.gamma.mul_(2.0 ** -14 / lags()[:, 1:64].square().mean().sqrt().item())
    k = lags()
    x = torch.randn(B, D, L).half().cuda().requires_grad_(True)
    dy = torch.zeros(B, D, L).half()
    ends = {(b, d): L - 1 - 11 * (b * D + d) for b in range(B) for d in range(D)}
    for (b, d), t in ends.items():
        dy[b, d, t] = 1.0
    layer(x)[0].backward(dy.cuda())
    dx = x.grad.cpu().double()
    for (b, d), t in ends.items():
        assert dx[b, d, t] == 2.0 ** 15 and not dx[b, d, t + 1:].any()
        got, want = dx[b, d, t - 200:t], k[d, 1:201].flip(0)
        assert (got - want).norm() <= 2.0 ** -12 * want.norm() + 2.0 ** -25 * want.numel() ** 0.5
