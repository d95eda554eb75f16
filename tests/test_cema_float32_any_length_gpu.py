"""The EMA layer on float32 rows whose length no piece of the kernels divides, against the float64 oracle: outputs, gradients,
last state.  Rows, matrices and the state between chunks enter with 24 bits, sums are float32, powers come from float32
coefficients: y, dx and the state up to 6e-7 in the 2-norm at the initial decays, gradients up to 2e-6 (theta, a sum of cancelling
terms).  Bars: three times that."""
import math

import pytest
import torch

from megalodon_amd import _lib, extension as megalodon_ops
from megalodon_amd.modules import MultiHeadComplexEMA
from oracle import cema as ocema, fftconv as offt
from test_cema_any_length_gpu import NAMES, _picked, _rows

pytestmark = pytest.mark.gpu


def _err(got, ref):
    got, ref = (torch.view_as_real(t) if t.is_complex() else t for t in (got.detach().cpu(), ref.detach()))
    return ((got.double() - ref).norm() / ref.norm()).item()


# rows taken from the boundary in front where B D L is a multiple of 8, by accesses at any element elsewhere; one item and several,
# several rows of a channel in one workgroup; one step, a piece, a chunk and a tile cut on either side
@pytest.mark.parametrize("B,D,L,offset", [(1, 8, 1, 0), (2, 8, 7, 0), (1, 3, 9, 0), (1, 8, 63, 1), (3, 8, 65, 0), (1, 5, 1021, 0),
                                          (2, 16, 2047, 0), (1, 16, 2049, 2), (1, 3, 8191, 0), (2, 8, 8195, 0), (1, 8, 20003, 0),
                                          (5, 304, 130, 0), (5, 520, 2049, 0)])
def test_layer_matches_oracle(B, D, L, offset):
    torch.manual_seed(L)
    layer = MultiHeadComplexEMA(D, 16).cuda().train()
    x0, x = _rows(B, D, L, torch.float32, L, offset)
    dy0, dy = _rows(B, D, L, torch.float32, L + 1, offset)
    x.requires_grad_(True)
    out, _ = layer(x)
    out.backward(dy)
    with torch.no_grad():
        layer.eval()
        again = layer(x)[0]
    grads = {n: getattr(layer, n).grad for n in NAMES}
    dx = x.grad
    if D > 64:  # every 50th channel is checked
        pick = slice(0, None, 50)
        out, again, dx, x0, dy0 = (t[:, pick] for t in (out, again, dx, x0, dy0))
        grads = {n: g[pick] for n, g in grads.items()}
        layer = _picked(layer, pick)
    pr = {n: getattr(layer, n).detach().cpu().double().requires_grad_(True) for n in NAMES}
    xo = x0.double().requires_grad_(True)
    p, q, g = ocema.calc_coeffs(pr["alpha"], pr["delta"], pr["theta"], pr["gamma"], 16)
    want = offt.fftconv_fwd(xo, ocema.ema_weight_fwd(p, q.log(), g, L)) + xo * pr["omega"]
    want.backward(dy0.double())
    assert out.dtype == dx.dtype == torch.float32
    assert max(_err(out, want), _err(again, want), _err(dx, xo.grad)) <= 2e-6
    for n in NAMES:
        if L > 1 or n in ("alpha", "gamma", "omega"):  # (one step: no power of q, those gradients are rounding alone)
            assert _err(grads[n], pr[n].grad) <= 6e-6, n


@pytest.mark.parametrize("carried", [False, True])
@pytest.mark.parametrize("B,D,L", [(2, 8, 1), (1, 3, 5), (2, 8, 63), (2, 8, 1531), (1, 3, 8201), (7, 400, 2113)])
def test_last_state(B, D, L, carried):
    """With a carried state these lengths stay with the float32 convolution, whose outputs are 3e-6 off: bar three times that."""
    N = 16
    torch.manual_seed(L)
    layer = MultiHeadComplexEMA(D, N).cuda().eval()
    x0, x = _rows(B, D, L, torch.float32, L, 0)
    h0 = torch.randn(B, D, N, dtype=torch.complex64, generator=torch.Generator().manual_seed(2)) if carried else None
    with torch.no_grad():
        out, last = layer(x, h0.cuda() if carried else None, True)
    if D > 64:
        pick = slice(0, None, 50)
        out, last, x0, h0 = out[:, pick], last[:, pick], x0[:, pick], h0[:, pick] if carried else None
        layer = _picked(layer, pick)
    pr = {n: getattr(layer, n).detach().cpu().double() for n in NAMES}
    p, q, g = ocema.calc_coeffs(pr["alpha"], pr["delta"], pr["theta"], pr["gamma"], N)
    want = offt.fftconv_fwd(x0.double(), ocema.ema_weight_fwd(p, q.log(), g, L)) + x0.double() * pr["omega"]
    if carried:
        want = want + ocema.ema_bias_fwd(q.log(), g, h0, L)
    assert _err(out, want) <= (9e-6 if carried else 2e-6)
    assert last.dtype == torch.complex64 and _err(last, ocema.ema_hidden_fwd(x0, p, q.log(), h0)) <= 2e-6


def _worst(got, ref):
    """The largest over channels of a channel's error in the 2-norm."""
    got, ref = (t.detach().cpu().double().transpose(0, 1).flatten(1) for t in (got, ref))
    return ((got - ref).norm(dim=1) / ref.norm(dim=1)).max().item()


@pytest.mark.parametrize("L", [121, 4097])
@pytest.mark.parametrize("mean", [0.0, 1.0])
@pytest.mark.parametrize("slower", [1, 10, 100])
def test_long_memories(monkeypatch, slower, mean, L):
    """Decays 1 - |q| ten and a hundred times slower than the initial ones, rows with a mean, the channel that is furthest off.
    Against 64 bits on the layer's own float32 coefficients: float32 operands and sums leave some 10 * 2^-24 of a channel whose modes
    do not cancel, up to ten times that where they do (a state of 16 bits: 3e-5).  Against 64 bits throughout: no
    further off than the convolution, where the coefficients decide for both up to a tenth."""
    D, N = 64, 16
    torch.manual_seed(L)
    layer = MultiHeadComplexEMA(D, N)
    with torch.no_grad():
        layer.delta.copy_(torch.logit(torch.sigmoid(layer.delta.double()) / slower))
    layer = layer.cuda().train()
    gen = torch.Generator().manual_seed(L + 1)
    x0, dy = torch.randn(2, D, L, generator=gen) + mean, torch.randn(2, D, L, generator=gen) + mean

    def both():
        x = x0.cuda().requires_grad_(True)
        out, _ = layer(x)
        out.backward(dy.cuda())
        return out, x.grad

    def oracle(p, log_q, g):
        xo = x0.double().requires_grad_(True)
        want = offt.fftconv_fwd(xo, ocema.ema_weight_fwd(p, log_q, g, L)) + xo * layer.omega.detach().cpu().double()
        want.backward(dy.double())
        return want, xo.grad

    got = both()
    monkeypatch.setenv("MEGA_CEMA_FFT", "1")
    convolved = both()
    pr = {n: getattr(layer, n).detach() for n in NAMES}
    p, log_q, g = (t.cpu() for t in megalodon_ops.cema_coeffs_fwd(pr["alpha"], pr["delta"], pr["theta"], pr["gamma"]))
    for a, b in zip(got, oracle(p.double(), log_q.to(torch.complex128), g.to(torch.complex128))):
        assert _err(a, b) <= 1e-6 and _worst(a, b) <= 6e-6
    pr = {n: t.cpu().double() for n, t in pr.items()}
    a, angle = torch.sigmoid(pr["alpha"]), torch.sigmoid(pr["theta"]) * (2 * math.pi / N) * torch.arange(1, N + 1, dtype=torch.float64).view(1, N, 1)
    exact = oracle(a, torch.complex(torch.log1p(-a * torch.sigmoid(pr["delta"])), angle.expand_as(a)),
                   torch.view_as_complex(pr["gamma"].contiguous()) * math.sqrt(1.0 / N))
    for ours, theirs, b in zip(got, convolved, exact):
        assert _err(ours, b) <= 1.1 * _err(theirs, b) and _worst(ours, b) <= 1.1 * _worst(theirs, b)


@pytest.mark.parametrize("B,D,L", [(2, 8, 1), (1, 3, 5), (2, 8, 63), (1, 3, 65), (2, 8, 1531), (1, 3, 8201), (7, 400, 130), (7, 400, 2113)])
def test_entry_point_takes_a_carried_state(B, D, L):
    """mega_cema_layer_scan_fwd with a state in front of such rows (the layer itself takes the convolution there): outputs and
    last state to the bars of rows without one, on the float32 coefficients that the call is given."""
    N = 16
    torch.manual_seed(L)
    layer = MultiHeadComplexEMA(D, N).cuda()
    x0, x = _rows(B, D, L, torch.float32, L, 0)
    h0 = torch.randn(B, D, N, dtype=torch.complex64, generator=torch.Generator().manual_seed(2))
    with torch.no_grad():
        p, log_q, g = megalodon_ops.cema_coeffs_fwd(layer.alpha, layer.delta, layer.theta, layer.gamma)
        omega, h = layer.omega.reshape(-1).contiguous(), h0.cuda()
        out, last = torch.empty_like(x), torch.empty(B, D, N, dtype=torch.complex64, device="cuda")
        _lib.call("mega_cema_layer_scan_fwd", _lib.ptr(x), _lib.i32(_lib.dtype_code(x.dtype)), _lib.ptr(p), _lib.ptr(log_q), _lib.ptr(g),
                  _lib.ptr(omega), _lib.ptr(h), _lib.i64(B), _lib.i64(D), _lib.i64(N), _lib.i64(L), _lib.ptr(out), _lib.ptr(last),
                  _lib.stream_ptr(x.device))
    pick = slice(0, None, 50 if D > 64 else 1)
    p, log_q, g, omega = p[pick].cpu().double(), log_q[pick].cpu().to(torch.complex128), g[pick].cpu().to(torch.complex128), omega[pick].cpu().double()
    x0, h0 = x0[:, pick].double(), h0[:, pick]
    want = offt.fftconv_fwd(x0, ocema.ema_weight_fwd(p, log_q, g, L)) + x0 * omega.view(-1, 1) + ocema.ema_bias_fwd(log_q, g, h0, L)
    assert _err(out[:, pick], want) <= 2e-6
    assert _err(last[:, pick], ocema.ema_hidden_fwd(x0, p.view(-1, N, 1), log_q.view(-1, N, 1), h0)) <= 2e-6


@pytest.mark.parametrize("B,D,L,forward,backward", [
    (8, 256, 9, True, True), (9, 256, 9, True, False), (1, 520, 9, True, False), (16, 64, 129, True, True), (16, 64, 127, True, False),
    (64, 104, 9, False, False), (64, 96, 9, True, False), (4, 1664, 289, True, False), (5, 1232, 287, False, False),
    (4, 520, 737, True, True), (4, 520, 735, True, False), (1, 520, 1025, True, False), (1, 520, 1401, True, True),
    (4, 264, 2303, True, True), (3, 512, 2051, True, False), (1, 513, 5001, True, False), (1, 520, 8191, True, False), (1, 520, 8193, True, True),
])
def test_shorter_way(monkeypatch, B, D, L, forward, backward):
    """Rows for which the convolution is ahead of the recurrence (many short ones: up to seventeen times) take it, bit for bit;
    the others do not."""
    torch.manual_seed(L)
    layer = MultiHeadComplexEMA(D, 16).cuda().train()
    x = _rows(B, D, L, torch.float32, L, 0)[1]

    def both():
        with torch.no_grad():
            y = layer(x)[0]
        xg = x.detach().requires_grad_(True)
        return y, torch.autograd.grad(layer(xg)[0].square().sum(), xg)[0]

    got = both()
    monkeypatch.setenv("MEGA_CEMA_FFT", "1")
    convolved = both()
    assert [torch.equal(a, b) for a, b in zip(got, convolved)] == [not forward, not backward]
    assert all(_err(a, b.double().cpu()) <= 1e-5 for a, b in zip(got, convolved))
