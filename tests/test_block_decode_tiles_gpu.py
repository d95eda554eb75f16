"""The one-token step's products in strips of 16 weight rows (csrc/block_decode.hip: tiles_kernel) where they can go wrong: one and
two token tiles full and not, fewer pieces of 128 values than waves, pieces cut by a row's end, both numbers of waves, the first
width and number of sequences that go there.  Against the step in 64 bits; bars as in test_block_decode_gpu."""
import pytest
import torch

from megalodon_amd.modules import RotaryEmbedding
from megalodon_amd.modules.block_decode import decode_step
from oracle import block as oblock
from test_block_decode_gpu import _block, _err, _prompt, _tensors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,D,S,E,F,heads,groups,dtype", [
    (5, 2048, 256, 512, 416, 1, 8, torch.bfloat16),     # the fewest tokens
    (8, 2048, 256, 8192, 4128, 4, 8, torch.float16),    # two waves a workgroup, else four; the last piece of F 32 values
    (9, 32, 64, 64, 32, 1, 1, torch.bfloat16),          # (rows_kernel's, four token tiles)
    (17, 32, 64, 64, 32, 1, 1, torch.bfloat16),         # one piece of 32 values
    (9, 416, 64, 64, 32, 1, 13, torch.bfloat16),        # the first width of nine tokens
    (16, 1024, 256, 512, 2784, 2, 8, torch.float16),    # a full tile; F cut at 96
    (17, 352, 128, 1024, 160, 2, 11, torch.bfloat16),   # a second tile of one token, three pieces of D, the last of 96
    (32, 1088, 128, 4096, 4192, 2, 2, torch.bfloat16),  # two full tiles, D cut at half a piece
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


def test_infinite_weight_and_token_stay_in_their_places():
    """F = 160 ends in a piece of 32: lanes behind the row's end hold its last values.  An infinite weight reaches its own
    output only, a sequence that is not finite its own only."""
    B, D, S, E, F, n = 18, 256, 64, 128, 160, 5
    blk = _block(D, S, E, F, 1, 4, 64)
    rotary = RotaryEmbedding(S, 64).cuda()
    with torch.no_grad():
        cache = _prompt(blk, B, n, D, S, E, 1, torch.bfloat16, rotary)
        x = torch.randn(B, 1, D, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
        freqs = rotary.get_freqs_cis(n, n + 1)
        clean = decode_step(blk, x, freqs, cache)[0]
        blk.nffn.fc2.weight[7, F - 1] = float("inf")
        x[3, 0, 5] = float("nan")
        y = decode_step(blk, x, freqs, cache)[0]
    rest = [i for i in range(B) if i != 3]
    columns = [i for i in range(D) if i != 7]
    assert not y[3].isfinite().any() and not y[..., 7].isfinite().any()
    assert torch.equal(y[rest][..., columns], clean[rest][..., columns])
