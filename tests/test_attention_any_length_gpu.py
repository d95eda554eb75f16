"""Attention through autograd at lengths off the products' slabs (32 queries, 64 keys) and at their
edges, where the probabilities are kept with rows and columns of zeros behind the real ones, against a
float32 reference; values next to the last row are poisoned in the tensor behind to show that
nothing of it is used.  Infinities in the last real row reach what reads it, and nothing else.
Tolerance: the 16-bit bar, 2e-2."""
import pytest
import torch

from conftest import rel_err
from megalodon_amd.fused_ops import swift_efficient_attention

pytestmark = pytest.mark.gpu


def _reference(q, k, v, dy, scale, causal):
    q, k, v = (t.detach().float().cpu().requires_grad_(True) for t in (q, k, v))
    s = scale * torch.matmul(q.transpose(1, 2), k.permute(0, 2, 3, 1).contiguous())
    if causal:
        L1, L2 = s.shape[-2:]
        s = s.masked_fill(torch.ones(L1, L2).triu(1 + L2 - L1).bool(), float("-inf"))
    y = torch.matmul(torch.softmax(s, -1), v.transpose(1, 2)).transpose(1, 2)
    y.backward(dy.float().cpu())
    return y.detach(), q.grad, k.grad, v.grad


@pytest.mark.parametrize("B,L1,L2,NH,H1,H2,causal,dtype", [
    (2, 1, 1, 2, 64, 64, True, torch.bfloat16),          # a single key
    (2, 33, 33, 1, 128, 72, True, torch.bfloat16),       # one row behind a slab
    (1, 255, 255, 2, 64, 128, True, torch.float16),      # one row short of a tile
    (2, 257, 257, 1, 256, 512, True, torch.bfloat16),    # one row behind a tile
    (2, 1021, 1021, 2, 256, 256, True, torch.bfloat16),
    (1, 1000, 1000, 2, 128, 64, True, torch.float16),    # rows of whole 16-byte pieces, but not of whole slabs
    (2, 45, 300, 2, 64, 64, True, torch.bfloat16),       # keys in front of the queries
    (1, 64, 77, 1, 128, 128, True, torch.bfloat16),
    (2, 50, 77, 2, 64, 128, False, torch.bfloat16),      # every key for every query
    (1, 4095, 4095, 1, 64, 64, True, torch.bfloat16),    # the widest padded row
    (1, 4097, 4097, 1, 64, 64, True, torch.bfloat16),    # beyond it
])
def test_forward_and_gradients(B, L1, L2, NH, H1, H2, causal, dtype):
    g = torch.Generator().manual_seed(L1 + L2)

    def rows(L, H):
        return torch.randn(B, L, NH, H, generator=g).to(dtype)

    q, k, v, dy = rows(L1, H1), rows(L2, H1), rows(L2, H2), rows(L1, H2)

    def on_gpu(t):  # NaN right behind the tensor's last element
        buf = torch.full((t.numel() + 4096,), float("nan"), dtype=dtype, device="cuda")
        return buf[:t.numel()].view(t.shape).copy_(t)

    qc, kc, vc = (on_gpu(t).requires_grad_(True) for t in (q, k, v))
    scale = H1 ** -0.5
    y = swift_efficient_attention(qc, kc, vc, scale, 0.0, causal, True)
    y.backward(on_gpu(dy))
    want = _reference(q, k, v, dy, scale, causal)
    for got, ref in zip((y, qc.grad, kc.grad, vc.grad), want):
        assert torch.isfinite(got.float()).all()
        # a single key: its gradients to q and k are zero up to rounding
        assert rel_err(got, ref) <= 2e-2 or (got.float().cpu() - ref).abs().max() <= 2e-2
    with torch.no_grad():
        assert torch.equal(swift_efficient_attention(qc, kc, vc, scale, 0.0, causal, True), y)


@pytest.mark.parametrize("B,L,NH,H1,H2,causal,dtype", [
    (1, 33, 2, 64, 64, True, torch.bfloat16),
    (2, 77, 1, 128, 72, False, torch.float16),
    (1, 300, 2, 256, 256, False, torch.bfloat16),
    (1, 1021, 1, 64, 320, True, torch.bfloat16),
])
def test_infinite_last_rows(B, L, NH, H1, H2, causal, dtype):
    """An infinite value row makes the outputs that see it infinite, an infinite row of the output's gradient the
    value gradients; rows of zeros behind them must not turn that into NaN."""
    g = torch.Generator().manual_seed(L)
    q, k = (torch.randn(B, L, NH, H1, generator=g).to(dtype).cuda() for _ in range(2))
    v, dy = (torch.randn(B, L, NH, H2, generator=g).to(dtype).cuda() for _ in range(2))
    v_inf, dy_inf = v.clone(), dy.clone()
    v_inf[:, -1] = float("inf")
    dy_inf[:, -1] = float("inf")
    scale = 0.1 * H1 ** -0.5  # every key has a probability that 16 bits hold
    with torch.no_grad():
        y = swift_efficient_attention(q, k, v_inf, scale, 0.0, causal, True)
        finite = swift_efficient_attention(q, k, v, scale, 0.0, causal, True)
    assert torch.isposinf(y[:, -1]).all()
    if not causal:
        assert torch.isposinf(y).all()
    else:  # (rows that share a tile with the last one multiply it by a zero probability)
        clear = (L - 1) // 256 * 256
        assert torch.equal(y[:, :clear], finite[:, :clear])
    leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
    swift_efficient_attention(*leaves, scale, 0.0, causal, True).backward(dy_inf)
    assert torch.isposinf(leaves[2].grad).all()


@pytest.mark.parametrize("L", [64, 77])
def test_scale_beyond_the_scores_kernel(L):
    """Scales from 1e30 take the separate product and softmax, at every length: a row picks its largest score."""
    g = torch.Generator().manual_seed(L)
    q, k, v, dy = (torch.randn(1, L, 2, 64, generator=g).bfloat16() for _ in range(4))
    leaves = [t.cuda().requires_grad_(True) for t in (q, k, v)]
    y = swift_efficient_attention(*leaves, 1e30, 0.0, True, True)
    y.backward(dy.cuda())
    s = torch.matmul(q.float().transpose(1, 2), k.float().permute(0, 2, 3, 1))
    s = s.masked_fill(torch.ones(L, L).triu(1).bool(), float("-inf"))
    top, at = s.topk(2, dim=-1) if L > 1 else (None, None)
    clear = (top[..., 0] - top[..., 1]) > 2 ** -7 * top[..., 0].abs()  # apart after the scores' rounding
    clear[..., 0] = True
    want = torch.gather(v.float().transpose(1, 2), 2, at[..., :1].expand(-1, -1, -1, 64))
    assert clear.float().mean() > 0.5
    assert torch.equal(y.detach().float().cpu().transpose(1, 2)[clear], want[clear])
    assert torch.isfinite(leaves[2].grad).all()
