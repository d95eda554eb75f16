"""The EMA layer's forward where a workgroup takes one item (at most four tiles of 2048 steps): other tables, no loads
ahead, coefficients formed in the same launch without gradients.  The arithmetic is that of the other form, so
the bits have to be: of the same channels in longer rows, in batches of any size, with and without gradients."""
import pytest
import torch

from conftest import rel_err
from megalodon_amd.modules import MultiHeadComplexEMA
from oracle import cema as ocema

pytestmark = pytest.mark.gpu


def _layer(D, N, dtype):
    torch.manual_seed(D + N)
    layer = MultiHeadComplexEMA(D, N).cuda().to(dtype)
    return layer.eval()


def _rows(B, D, L, dtype):
    return torch.randn(B, D, L, generator=torch.Generator().manual_seed(L)).to(dtype).cuda()


@pytest.mark.parametrize("params", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N", [16, 5, 1])
@pytest.mark.parametrize("L,more,dtype", [
    (8, 8200, torch.float32), (2048, 6200, torch.float32), (8192, 64, torch.float32),
    (8192, 64, torch.bfloat16), (8128, 8192, torch.float16),
    (1, 8256, torch.bfloat16), (8185, 64, torch.bfloat16), (2041, 6400, torch.float16),  # rows off the 16-byte pieces
])
def test_longer_rows_start_with_the_same_outputs(L, more, dtype, N, params):
    layer, x = _layer(8, N, params), _rows(1, 8, L + more, dtype)
    with torch.no_grad():
        whole = layer(x)[0]
        assert torch.equal(layer(x[..., :L].contiguous())[0], whole[..., :L])


@pytest.mark.parametrize("L,dtype", [(200, torch.float32), (200, torch.bfloat16), (1531, torch.bfloat16), (77, torch.float16)])
def test_rows_of_a_batch_and_alone(L, dtype):
    """1024 channels: one row alone, four or more of a channel in a workgroup's item, and many in one's walk."""
    layer, x = _layer(1024, 16, torch.float32), _rows(24, 1024, L, dtype)
    with torch.no_grad():
        alone = torch.cat([layer(x[b:b + 1])[0] for b in range(4)])
        for B in (3, 4, 8, 24):
            assert torch.equal(layer(x[:B])[0][:4], alone[:B])


@pytest.mark.parametrize("params", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("L,dtype", [(2048, torch.float32), (2000, torch.bfloat16), (1021, torch.float16), (9000, torch.bfloat16)])
def test_with_and_without_gradients(L, dtype, params):
    layer, x = _layer(16, 16, params), _rows(2, 16, L, dtype)
    with torch.no_grad():
        want = layer(x)[0]
        y, h = layer(x, None, True)  # the branch with a last state: coefficients from their own launch
    assert torch.equal(y, want) and torch.isfinite(torch.view_as_real(h)).all()
    assert torch.equal(layer(x.requires_grad_(True))[0].detach(), want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("L", [8, 64, 72, 1984, 2040, 2048, 2056, 4088])
def test_state_behind_the_last_step(L, dtype):
    """The lanes hand each other the steps of the last chunk: full, of one step, and of most; the last chunk of a tile, the
    first, and rows that leave waves without a tile.  Rows alone and in a batch: the same bits; the 16-bit rows of a length
    that is one step shorter likewise.  Bar against float64: the operands' two bf16 pieces, 2^-16, over a sum of terms of
    either sign, which cost some digits (1e-4, as for every state)."""
    lengths = [L] if dtype == torch.float32 else [L, L - 1]
    for steps in lengths:
        layer, x = _layer(256, 16, torch.float32), _rows(20, 256, steps, dtype)
        with torch.no_grad():
            batch = layer(x, None, True)[1]
            alone = torch.cat([layer(x[b:b + 1], None, True)[1] for b in range(4)])
        assert torch.equal(torch.view_as_real(batch[:4]), torch.view_as_real(alone))
        pick = slice(0, None, 51)
        pr = {n: getattr(layer, n).detach().cpu().double()[pick] for n in ("alpha", "delta", "theta", "gamma")}
        p, q, _ = ocema.calc_coeffs(pr["alpha"], pr["delta"], pr["theta"], pr["gamma"], 16)
        want = ocema.ema_hidden_fwd(x[:4, pick].cpu().double(), p, q.log(), None)
        assert rel_err(alone[:, pick], want) <= 1e-4
