"""The runs of keys that the one-token step's attention takes (csrc/block_decode.hip: key_runs): one for a (sequence, head) and
several, of the last length with short requests and the first with long ones, longer than a thousand keys and than the score
buffer, with the last run cut and of the new key alone.  Against the step in 64 bits (bars as in test_block_decode_rows_gpu); old
keys and values pass on unchanged."""
import pytest
import torch

from megalodon_amd.modules import RotaryEmbedding
from megalodon_amd.modules.block_decode import decode_step
from oracle import block as oblock
from test_block_decode_gpu import _block, _err, _prompt, _tensors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,heads,n,zh,H2", [
    (16, 4, 1195, 64, 64),    # four runs of 299 keys
    (16, 4, 1196, 64, 128),   # four of 300, the last of 297
    (32, 8, 40, 64, 64),      # two runs, of 21 and 20
    (32, 8, 40, 64, 256),     # a run each
    (32, 8, 4100, 64, 64),    # five runs of at most 1024 keys
    (32, 8, 8192, 64, 64),    # nine
    (16, 16, 4100, 64, 256),  # 4101 keys: more than a run holds, two of 2051 and 2050
    (19, 9, 1030, 64, 64),    # the fewest pairs of two runs each for their narrow values
    (17, 10, 1030, 64, 64),   # one pair fewer: three runs of two workgroups a CU
    (19, 9, 1030, 64, 256),   # wide values: one run
    (32, 4, 2200, 128, 64),   # two runs of more than 1024
    (29, 9, 2100, 64, 64),    # more pairs than CUs: three runs of 701, 701 and 699
    (32, 12, 40, 64, 64),     # two runs, of 21 and 20
    (31, 13, 1024, 64, 64),   # one run each, were it not for the last key: 513 and 512
    (20, 8, 301, 64, 64),     # pairs that a workgroup a CU does not fit: three runs of two workgroups a CU
    (5, 4, 176, 256, 256),    # eleven runs of 16 keys and one of the new key alone
    (32, 2, 1, 64, 2048),     # two keys
])
def test_runs_against_float64(B, heads, n, zh, H2):
    D, S, E, chunk = 128, heads * zh, heads * H2, n + 8
    blk = _block(D, S, E, 64, heads, 2, chunk)
    rotary = RotaryEmbedding(zh, chunk).cuda()
    p = {k: v.detach().double().cpu() for k, v in blk.named_parameters()}
    gen = torch.Generator("cuda").manual_seed(n)
    with torch.no_grad():
        cache = _prompt(blk, B, 1, D, S, E, heads, torch.bfloat16, rotary)
        k, v = (torch.randn(B, n, heads, w, generator=gen, device="cuda").bfloat16() for w in (zh, H2))
        cache = ((k, v, n), cache[1], cache[2])
        on_host = ((k.cpu(), v.cpu(), n), tuple(t.cpu() for t in cache[1]), cache[2].cpu())
        x = torch.randn(B, 1, D, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
        freqs = rotary.get_freqs_cis(n, n + 1)
        want = oblock.mega_block_step(p, x.cpu(), on_host, num_heads=heads, ndim=16, groups=2,
                                      eps=blk.mega.timenorm.eps, freqs_cis=freqs.cpu())
        y, after = decode_step(blk, x, freqs, cache)
    step = (y, *_tensors(after))
    assert _err(step[0], want[0]) <= 7.8e-3
    for s, w, old in zip(step[1:3], want[1:3], (k, v)):
        assert torch.equal(s[:, :-1], old)
        assert _err(s[:, -1], w[:, -1]) <= 5e-3
