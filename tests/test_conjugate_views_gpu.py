"""`t.conj()` of a contiguous complex tensor is a view that shares its memory and keeps the sign in a bit: operators
that read memory have to resolve it.  Every complex operand that a caller hands in, against the resolved one:
the same kernels on the same numbers, so equal bits."""
import pytest
import torch

from megalodon_amd import extension as ops
from megalodon_amd.fused_ops import qk_norm_rotary
from megalodon_amd.modules import MegaBlock, MultiHeadComplexEMA, RotaryEmbedding

pytestmark = pytest.mark.gpu


def _randn(*shape, dtype=torch.float32, seed=1):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed), dtype=torch.float32).to(dtype).cuda()


def _complex(*shape, seed=2):
    return torch.view_as_complex(_randn(*shape, 2, seed=seed))


def test_rotary_factors():
    z = _randn(2, 7, 128, dtype=torch.bfloat16).requires_grad_(True)
    gamma, beta = _randn(2, 128, dtype=torch.bfloat16), _randn(2, 128, dtype=torch.bfloat16)
    f = RotaryEmbedding(64, 16).cuda().get_freqs_cis(0, 7)
    lazy, resolved = f.conj(), f.conj().resolve_conj()
    assert lazy.is_conj() and not resolved.is_conj()
    grads = []
    for factors in (lazy, resolved):
        q, k = qk_norm_rotary(z, gamma, beta, factors, 64, 1e-5)
        z.grad = None
        (q.float() * 2 + k.float()).sum().backward()
        grads.append((q, k, z.grad))
    assert all(torch.equal(a, b) for a, b in zip(*grads))
    plain, _ = qk_norm_rotary(z, gamma, beta, f, 64, 1e-5)
    assert not torch.equal(plain, grads[0][0])
    direct = [ops.qk_norm_rotary_fwd(z.detach(), gamma, beta, factors, 64, 1e-5)[0] for factors in (lazy, resolved)]
    assert torch.equal(*direct)


@pytest.mark.parametrize("dtype,L", [(torch.bfloat16, 100), (torch.float32, 100), (torch.float32, 64)])
def test_carried_state(dtype, L):
    layer = MultiHeadComplexEMA(64, 16).cuda().eval()
    x, h = _randn(2, 64, L, dtype=dtype), _complex(2, 64, 16)
    with torch.no_grad():
        outs = [layer(x, state, True) for state in (h.conj(), h.conj().resolve_conj())]
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    layer.train()
    outs = [layer(x, state, True) for state in (h.conj(), h.conj().resolve_conj())]
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("tokens", [1, 3])
def test_block_on_a_cache(tokens):
    torch.manual_seed(3)
    blk = MegaBlock(model_dim=256, z_dim=128, value_dim=512, num_heads=2, cema_ndim=16, chunk_size=64,
                    ffn_hidden_dim=512, norm_num_groups=2, init_std=0.05).cuda().bfloat16().eval()
    rotary = RotaryEmbedding(64, 64).cuda()
    empty = ((torch.empty(2, 0, 2, 64, dtype=torch.bfloat16, device="cuda"),
              torch.empty(2, 0, 2, 256, dtype=torch.bfloat16, device="cuda"), 0), (None, None, None), None)
    x = _randn(2, tokens, 256, dtype=torch.bfloat16)
    f = rotary.get_freqs_cis(9, 9 + tokens)
    with torch.no_grad():
        _, (attn, norm, h) = blk(_randn(2, 9, 256, dtype=torch.bfloat16, seed=5), rotary.get_freqs_cis(0, 9), None, empty)
        wanted, _ = blk(x, f.conj().resolve_conj(), None, (attn, norm, h.conj().resolve_conj()))
        plain, _ = blk(x, f, None, (attn, norm, h))
        for factors, state in ((f.conj(), h.conj().resolve_conj()), (f.conj().resolve_conj(), h.conj()), (f.conj(), h.conj())):
            got, _ = blk(x, factors, None, (attn, norm, state))
            # (the one-token step goes operator by operator here: the 16-bit bar)
            err = (got.float() - wanted.float()).abs().max() / wanted.float().abs().max()
            assert err <= 2e-2 and (plain.float() - wanted.float()).abs().max() / wanted.float().abs().max() > 5e-2
