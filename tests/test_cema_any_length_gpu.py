"""The EMA layer on 16-bit rows whose length no piece of the kernels divides (and on rows that start off
16-byte boundaries) against the float64 oracle: outputs, all gradients, the carried state and the last one.
Bars: 2e-2 for 16-bit tensors, 1e-4 for float32 ones; parameters cast to bfloat16 give bfloat16 gradients."""
import pytest
import torch

from conftest import rel_err
from megalodon_amd.modules import MultiHeadComplexEMA
from oracle import cema as ocema, fftconv as offt

pytestmark = pytest.mark.gpu
NAMES = ("alpha", "delta", "theta", "gamma", "omega")


def _rows(B, D, L, dtype, seed, offset):
    """(B, D, L) rows on the GPU, `offset` elements behind a 16-byte boundary."""
    v = torch.randn(B, D, L, generator=torch.Generator().manual_seed(seed)).to(dtype)
    t = torch.empty(v.numel() + 8, dtype=dtype, device="cuda")[offset:offset + v.numel()].view(B, D, L)
    return v, t.copy_(v)


class _picked:
    """The parameters of some channels of a layer."""

    def __init__(self, layer, pick):
        for n in NAMES:
            setattr(self, n, getattr(layer, n)[pick])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,D,L,offset", [(1, 2, 1, 0), (2, 3, 7, 0), (2, 2, 9, 1), (1, 3, 65, 0), (2, 3, 1021, 0),
                                          (1, 2, 2047, 0), (1, 3, 4096, 3), (2, 2, 8193, 0), (1, 2, 20003, 5),
                                          # whole tensors of 16-byte pieces, rows taken from the boundary in front
                                          (8, 1, 1, 0), (1, 8, 57, 0), (1, 8, 65, 0), (2, 8, 2043, 0), (1, 8, 20003, 0),
                                          # several rows of a channel in one workgroup: two, two and one; five, of two tiles each
                                          (5, 300, 130, 0), (5, 520, 2049, 1)])
def test_layer_matches_oracle(B, D, L, offset, dtype):
    torch.manual_seed(L)
    layer = MultiHeadComplexEMA(D, 16).cuda().train()
    x0, x = _rows(B, D, L, dtype, L, offset)
    dy0, dy = _rows(B, D, L, dtype, L + 1, offset)
    x.requires_grad_(True)
    out, _ = layer(x)
    out.backward(dy)
    grads = {n: getattr(layer, n).grad for n in NAMES}
    dx = x.grad
    if D > 64:  # every 50th channel is checked
        pick = slice(0, None, 50)
        out, dx, x0, dy0 = out[:, pick], dx[:, pick], x0[:, pick], dy0[:, pick]
        grads = {n: g[pick] for n, g in grads.items()}
        layer = _picked(layer, pick)
    pr = {n: getattr(layer, n).detach().cpu().double().requires_grad_(True) for n in NAMES}
    xo = x0.double().requires_grad_(True)
    p, q, g = ocema.calc_coeffs(pr["alpha"], pr["delta"], pr["theta"], pr["gamma"], 16)
    want = offt.fftconv_fwd(xo, ocema.ema_weight_fwd(p, q.log(), g, L)) + xo * pr["omega"]
    want.backward(dy0.double())
    assert out.dtype == dtype and rel_err(out, want.detach()) <= 2e-2
    assert dx.dtype == dtype and rel_err(dx, xo.grad) <= 2e-2
    for n in NAMES:
        assert rel_err(grads[n], pr[n].grad) <= 1e-4, n


@pytest.mark.parametrize("B,D,L,offset", [(2, 3, 1, 0), (2, 3, 5, 0), (2, 3, 63, 1), (2, 3, 1531, 0), (2, 3, 8200, 1),
                                          (2, 3, 8201, 0), (5, 400, 70, 0), (7, 400, 2112, 0)])
def test_carried_and_last_state(B, D, L, offset):
    N = 16
    torch.manual_seed(L)
    layer = MultiHeadComplexEMA(D, N).cuda().eval()
    x0, x = _rows(B, D, L, torch.bfloat16, L, offset)
    h0 = torch.randn(B, D, N, dtype=torch.complex64, generator=torch.Generator().manual_seed(2))
    with torch.no_grad():
        out, last = layer(x, h0.cuda(), True)
    if D > 64:  # every 50th channel is checked
        pick = slice(0, None, 50)
        out, last, x0, h0 = out[:, pick], last[:, pick], x0[:, pick], h0[:, pick]
        layer = _picked(layer, pick)
    pr = {n: getattr(layer, n).detach().cpu().double() for n in NAMES}
    p, q, g = ocema.calc_coeffs(pr["alpha"], pr["delta"], pr["theta"], pr["gamma"], N)
    want = offt.fftconv_fwd(x0.double(), ocema.ema_weight_fwd(p, q.log(), g, L)) + x0.double() * pr["omega"]
    want = want + ocema.ema_bias_fwd(q.log(), g, h0, L)
    assert rel_err(out, want) <= 2e-2
    assert last.dtype == torch.complex64 and rel_err(last, ocema.ema_hidden_fwd(x0, p, q.log(), h0)) <= 1e-4


def test_parameters_in_bfloat16():
    B, D, L = 3, 4, 100
    torch.manual_seed(0)
    layer = MultiHeadComplexEMA(D, 16).cuda().bfloat16().train()
    x0, x = _rows(B, D, L, torch.bfloat16, 1, 0)
    dy0, dy = _rows(B, D, L, torch.bfloat16, 2, 0)
    x.requires_grad_(True)
    out, _ = layer(x)
    out.backward(dy)
    pr = {n: getattr(layer, n).detach().cpu().double().requires_grad_(True) for n in NAMES}
    p, q, g = ocema.calc_coeffs(pr["alpha"], pr["delta"], pr["theta"], pr["gamma"], 16)
    want = offt.fftconv_fwd(x0.double(), ocema.ema_weight_fwd(p, q.log(), g, L)) + x0.double() * pr["omega"]
    want.backward(dy0.double())
    assert rel_err(out, want.detach()) <= 2e-2
    for n in NAMES:
        got = getattr(layer, n).grad
        assert got.dtype == torch.bfloat16 and rel_err(got, pr[n].grad) <= 2e-2, n


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,D,L", [(3, 64, 121), (2, 64, 201), (2, 64, 513), (2, 64, 777)])
def test_float32_results_keep_float32_precision(B, D, L, dtype):
    """The last state and the parameter gradients are float32 results: a float32 convolution has them to some four
    units of 2^-24 in the 2-norm, rows and powers of 16 bits to twice that and more.  Bar: six."""
    torch.manual_seed(L)
    layer = MultiHeadComplexEMA(D, 16).cuda().train()
    x0, x = _rows(B, D, L, dtype, L, 0)
    dy0, dy = _rows(B, D, L, dtype, L + 1, 0)
    x.requires_grad_(True)
    layer(x)[0].backward(dy)
    with torch.no_grad():
        last = layer(x, None, True)[1]
    pr = {n: getattr(layer, n).detach().cpu().double().requires_grad_(True) for n in NAMES}
    p, q, g = ocema.calc_coeffs(pr["alpha"], pr["delta"], pr["theta"], pr["gamma"], 16)
    want = offt.fftconv_fwd(x0.double(), ocema.ema_weight_fwd(p, q.log(), g, L)) + x0.double() * pr["omega"]
    want.backward(dy0.double())

    def err(got, ref):
        got, ref = (torch.view_as_real(t) if t.is_complex() else t for t in (got.detach().cpu(), ref.detach()))
        return ((got.double() - ref).norm() / ref.norm()).item()

    errors = {n: err(getattr(layer, n).grad, pr[n].grad) for n in ("alpha", "gamma", "omega")}
    errors["last"] = err(last, ocema.ema_hidden_fwd(x0, p, q.log(), None))
    assert max(errors.values()) <= 6 * 2 ** -24, errors


@pytest.mark.parametrize("channels", [32, 128])
@pytest.mark.parametrize("L", [40, 41])
def test_rows_of_another_width_are_refused(channels, L):
    layer = MultiHeadComplexEMA(64, 16).cuda().eval()
    x = torch.randn(2, channels, L, device="cuda").bfloat16()
    with torch.no_grad(), pytest.raises(RuntimeError):
        layer(x, None, True)
    with torch.no_grad(), pytest.raises(RuntimeError):
        layer(x, torch.zeros(2, channels, 16, dtype=torch.complex64, device="cuda"), False)
