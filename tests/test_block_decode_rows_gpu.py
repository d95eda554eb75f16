"""The weight products of the one-token step (csrc/block_decode.hip: rows_kernel, tiles_kernel behind rows_norm_kernel) where
they can go wrong: one and two token tiles full and not, reductions of fewer pieces of 128 than waves, pieces cut by a row's
end, rows longer than are normalised on the way.  Against the step in 64 bits; bars as in test_block_decode_gpu."""
import pytest
import torch

from megalodon_amd.modules import RotaryEmbedding
from megalodon_amd.modules.block_decode import decode_step
from oracle import block as oblock
from test_block_decode_gpu import _block, _err, _prompt, _tensors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,D,S,E,F,heads,groups,dtype", [
    (4, 1024, 256, 2048, 2752, 1, 8, torch.bfloat16),   # a full tile, F cut at half a piece
    (5, 1120, 128, 512, 1056, 2, 5, torch.bfloat16),    # nine pieces of D, the last of 96: waves of one and of two
    (8, 640, 64, 64, 160, 1, 4, torch.float16),         # five pieces for eight waves, an E of half a piece
    (7, 4096, 128, 256, 96, 2, 8, torch.bfloat16),      # the longest row that rows_kernel would take, of more tokens
    (2, 4128, 64, 128, 64, 1, 3, torch.bfloat16),       # one that is longer
    (9, 1024, 256, 512, 416, 2, 8, torch.float16),      # more tokens than two tiles of its width
    (1, 8192, 64, 64, 64, 1, 8, torch.bfloat16),
    (9, 32, 64, 64, 32, 1, 1, torch.bfloat16),          # four token tiles, the third of one token; one piece of 32 values
    (16, 384, 128, 1024, 1056, 2, 12, torch.float16),   # all full, the widest rows
    (13, 352, 64, 256, 160, 1, 11, torch.bfloat16),     # three pieces, the last of 96
])
def test_step_against_float64(B, D, S, E, F, heads, groups, dtype):
    n, chunk = 20, 64
    blk = _block(D, S, E, F, heads, groups, chunk, dtype)
    rotary = RotaryEmbedding(S // heads, chunk).cuda()
    p = {k: v.detach().double().cpu() for k, v in blk.named_parameters()}
    with torch.no_grad():
        cache = _prompt(blk, B, n, D, S, E, heads, dtype, rotary)
        on_host = (tuple(t.cpu() for t in cache[0][:2]) + (n,), tuple(t.cpu() for t in cache[1]), cache[2].cpu())
        x = torch.randn(B, 1, D, generator=torch.Generator().manual_seed(1)).to(dtype).cuda()
        freqs = rotary.get_freqs_cis(n, n + 1)
        want = oblock.mega_block_step(p, x.cpu(), on_host, num_heads=heads, ndim=16, groups=groups,
                                      eps=blk.mega.timenorm.eps, freqs_cis=freqs.cpu())
        y, after = decode_step(blk, x, freqs, cache)
        step = (y, *_tensors(after))
    assert _err(step[0], want[0]) <= 7.8e-3
    for s, w in zip(step[1:3], want[1:3]):
        assert _err(s[:, -1], w[:, -1]) <= 5e-3


def test_infinite_weight_stays_in_its_row():
    """F = 160 ends in a piece of 32: lanes behind the row's end hold its last values, and an infinite one among them
    may reach its own output only."""
    B, D, S, E, F, n = 3, 256, 64, 128, 160, 5
    blk = _block(D, S, E, F, 1, 4, 64)
    rotary = RotaryEmbedding(S, 64).cuda()
    with torch.no_grad():
        cache = _prompt(blk, B, n, D, S, E, 1, torch.bfloat16, rotary)
        x = torch.randn(B, 1, D, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
        freqs = rotary.get_freqs_cis(n, n + 1)
        blk.nffn.fc2.weight[7, F - 1] = float("inf")
        y = decode_step(blk, x, freqs, cache)[0]
        wanted, _ = blk.mega(x, freqs, None, cache)
        wanted = blk.nffn(wanted, x)
    assert torch.equal(y.isfinite(), wanted.isfinite()) and torch.equal(y.isinf(), wanted.isinf())
    assert not y[..., 7].isfinite().any() and y.isfinite().sum() == B * (D - 1)


def test_streams_step_at_once():
    """Six sequences, two token tiles, on eight streams at once: each its own workspace, each the step's own bits."""
    B, D, S, E, F, n = 6, 512, 128, 256, 416, 30
    blk = _block(D, S, E, F, 1, 4, 64)
    rotary = RotaryEmbedding(S, 64).cuda()
    with torch.no_grad():
        cache = _prompt(blk, B, n, D, S, E, 1, torch.bfloat16, rotary)
        xs = [torch.randn(B, 1, D, generator=torch.Generator().manual_seed(i)).bfloat16().cuda() for i in range(8)]
        freqs = rotary.get_freqs_cis(n, n + 1)
        wanted = [decode_step(blk, x, freqs, cache) for x in xs]
        torch.cuda.synchronize()
        streams, got = [torch.cuda.Stream() for _ in xs], []
        for stream, x in zip(streams, xs):
            with torch.cuda.stream(stream):
                got.append(decode_step(blk, x, freqs, cache))
        torch.cuda.synchronize()
    for g, w in zip(got, wanted):
        assert torch.equal(g[0], w[0])
        assert all(torch.equal(a, b) for a, b in zip(_tensors(g[1]), _tensors(w[1])))
