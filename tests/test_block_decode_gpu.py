"""The fused one-token step of a block (csrc/block_decode.hip) against the same step in 64 bits and taken operator by
operator, at the edges of what the kernels take: token tiles (1, 16, 17, 32 sequences), head
widths, lengths of one key, one run and many runs of keys.  Tolerance: the 16-bit bar, 2e-2."""
import copy
import io

import pytest
import torch

from conftest import rel_err
from megalodon_amd.modules import MegaBlock, RotaryEmbedding
from megalodon_amd.modules.block_decode import decode_step
from oracle import block as oblock

pytestmark = pytest.mark.gpu


def _block(D, S, E, F, heads, groups, chunk, dtype=torch.bfloat16, affine=True, **dropouts):
    torch.manual_seed(3)
    blk = MegaBlock(model_dim=D, z_dim=S, value_dim=E, num_heads=heads, cema_ndim=16, chunk_size=chunk,
                    ffn_hidden_dim=F, norm_num_groups=groups, init_std=0.05, norm_affine=affine, **dropouts).cuda().to(dtype).eval()
    with torch.no_grad():
        for name, p in blk.named_parameters():
            if p.abs().max() == 0:
                p.normal_(0, 0.1)
    return blk


def _prompt(blk, B, n, D, S, E, heads, dtype, rotary):
    empty = ((torch.empty(B, 0, heads, S // heads, dtype=dtype, device="cuda"),
              torch.empty(B, 0, heads, E // heads, dtype=dtype, device="cuda"), 0), (None, None, None), None)
    x = torch.randn(B, n, D, generator=torch.Generator().manual_seed(n)).to(dtype).cuda()
    return blk(x, rotary.get_freqs_cis(0, n), None, empty)[1]


SIZES = pytest.mark.parametrize("B,n,D,S,E,F,heads,groups,dtype,affine", [
    (1, 1, 256, 128, 512, 512, 2, 2, torch.bfloat16, True),       # one cached key, 64-wide heads
    (16, 40, 1024, 256, 2048, 2752, 1, 8, torch.bfloat16, True),  # a full token tile, 2048-wide values
    (17, 513, 256, 512, 128, 96, 2, 8, torch.bfloat16, True),     # two token tiles, narrow values, many runs
    (32, 7, 512, 256, 1024, 320, 2, 2, torch.float16, True),
    (3, 1000, 384, 384, 768, 416, 3, 3, torch.bfloat16, False),   # no affine norms, reductions that do not divide by eight waves
])


@SIZES
def test_step_matches_operators(B, n, D, S, E, F, heads, groups, dtype, affine):
    chunk = 1024
    blk = _block(D, S, E, F, heads, groups, chunk, dtype, affine)
    rotary = RotaryEmbedding(S // heads, chunk).cuda()
    with torch.no_grad():
        cache = _prompt(blk, B, n, D, S, E, heads, dtype, rotary)
        for t in range(3):
            x = torch.randn(B, 1, D, generator=torch.Generator().manual_seed(t)).to(dtype).cuda()
            freqs = rotary.get_freqs_cis(n + t, n + t + 1) if t != 1 else None
            before = [c.clone() for c in (*cache[0][:2], *cache[1], cache[2])]
            y, wanted = blk.mega(x, freqs, None, cache)
            y = blk.nffn(y, x)
            got = decode_step(blk, x, freqs, cache)
            assert got is not None
            for a, b in zip(before, (*cache[0][:2], *cache[1], cache[2])):
                assert torch.equal(a, b)  # the cache that was handed in is what it was
            assert rel_err(got[0], y) <= 2e-2
            assert got[1][0][2] == wanted[0][2] == n + t + 1
            assert torch.equal(got[1][1][0], wanted[1][0])
            for a, b in ((got[1][0][0], wanted[0][0]), (got[1][0][1], wanted[0][1]), (got[1][1][1], wanted[1][1]),
                         (got[1][1][2], wanted[1][2])):
                assert a.shape == b.shape and a.dtype == b.dtype and rel_err(a, b) <= 2e-2
            assert got[1][2].dtype == wanted[2].dtype and rel_err(got[1][2], wanted[2]) <= 2e-2
            cache = got[1]


def _err(got, want):
    got, want = (torch.view_as_real(t.detach().cpu().resolve_conj()) if t.is_complex() else t.detach().cpu() for t in (got, want))
    return ((got.double() - want.double()).norm() / want.double().norm()).item()


@SIZES
def test_step_against_float64(B, n, D, S, E, F, heads, groups, dtype, affine):
    """The step and the operators from one cache, against the same step in 64 bits.  A rounding to bfloat16 is 2^-9 / sqrt(3)
    = 1.1e-3 in the norm; up to five lie in front of keys, values and statistics, twelve in front of the output (normalised
    row, EMA output, its norm, four projections' values, q, k, attention, gate, y1, its norm, hidden): 2.5e-3 and 3.9e-3
    where nothing amplifies them.  Bars twice that.  And the step, which rounds in fewer places than the
    operators, may not be further off than they are."""
    chunk = 1024
    blk = _block(D, S, E, F, heads, groups, chunk, dtype, affine)
    rotary = RotaryEmbedding(S // heads, chunk).cuda()
    p = {k: v.detach().double().cpu() for k, v in blk.named_parameters()}
    with torch.no_grad():
        cache = _prompt(blk, B, n, D, S, E, heads, dtype, rotary)
        on_host = (tuple(t.cpu() for t in cache[0][:2]) + (n,), tuple(t.cpu() for t in cache[1]), cache[2].cpu())
        x = torch.randn(B, 1, D, generator=torch.Generator().manual_seed(1)).to(dtype).cuda()
        freqs = rotary.get_freqs_cis(n, n + 1)
        want = oblock.mega_block_step(p, x.cpu(), on_host, num_heads=heads, ndim=16, groups=groups,
                                      eps=blk.mega.timenorm.eps, freqs_cis=freqs.cpu())
        y, after = blk.mega(x, freqs, None, cache)
        operators = (blk.nffn(y, x), *_tensors(after))
        y, after = decode_step(blk, x, freqs, cache)
        step = (y, *_tensors(after))
    for name, s, o, w in zip(("out", "keys", "values", "count", "mean", "var", "state"), step, operators, want):
        if name == "count":
            assert torch.equal(s.cpu(), w.to(s.dtype))
            continue
        if name in ("keys", "values"):  # the old rows are the cache's own
            assert torch.equal(s[:, :-1].cpu().double(), w[:, :-1])
            s, o, w = s[:, -1], o[:, -1], w[:, -1]
        assert _err(s, w) <= (7.8e-3 if name == "out" else 5e-3), (name, _err(s, w))
        assert _err(s, w) <= 1.1 * _err(o, w) + 2 ** -14, (name, _err(s, w), _err(o, w))


def test_last_token_of_a_chunk_empties_the_cache():
    blk = _block(256, 128, 512, 512, 2, 2, 64)
    rotary = RotaryEmbedding(64, 64).cuda()
    with torch.no_grad():
        cache = _prompt(blk, 2, 63, 256, 128, 512, 2, torch.bfloat16, rotary)
        x = torch.randn(2, 1, 256, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
        y, cache = decode_step(blk, x, rotary.get_freqs_cis(63, 64), cache)
        assert cache[0][0].shape[1] == 0 and cache[0][1].shape[1] == 0 and cache[0][2] == 0
        assert decode_step(blk, x, rotary.get_freqs_cis(0, 1), cache) is None  # the next chunk's first token: operators


def _tensors(cache):
    return [*cache[0][:2], *cache[1], cache[2]]


def test_continued_cache_shares_nothing_with_the_old_one():
    """A cache is a value: continuing it, or writing to what came out, leaves it as it was; what comes out is
    contiguous and can be copied, saved and continued in any gradient mode."""
    blk = _block(256, 128, 512, 512, 2, 2, 512)
    rotary = RotaryEmbedding(64, 512).cuda()
    xs = [torch.randn(2, 1, 256, generator=torch.Generator().manual_seed(s)).bfloat16().cuda() for s in range(2)]
    many = torch.randn(2, 5, 256, generator=torch.Generator().manual_seed(7)).bfloat16().cuda()
    freqs = rotary.get_freqs_cis(30, 31)
    with torch.no_grad():
        cache = _prompt(blk, 2, 30, 256, 128, 512, 2, torch.bfloat16, rotary)
        before = [t.clone() for t in _tensors(cache)]
        _, first = decode_step(blk, xs[0], freqs, cache)
        kept = [t.clone() for t in _tensors(first)]
        _, second = decode_step(blk, xs[1], freqs, cache)
        _, longer = blk(many, rotary.get_freqs_cis(30, 35), None, cache)
        for other in (second, longer):
            storages = {t.untyped_storage().data_ptr() for t in _tensors(other)}
            assert not storages & {t.untyped_storage().data_ptr() for t in _tensors(first) + _tensors(cache)}
        assert all(torch.equal(a, b) for a, b in zip(_tensors(first), kept))
        copied = copy.deepcopy(first)
        saved = io.BytesIO()
        torch.save(first, saved)
        for c in (first, second, longer):
            assert c[0][0].is_contiguous() and c[0][1].is_contiguous()
            for t in _tensors(c):
                t.zero_()
        assert all(torch.equal(a, b) for a, b in zip(_tensors(cache), before))
        saved.seek(0)
        for c in (copied, torch.load(saved)):
            assert all(torch.equal(a, b) for a, b in zip(_tensors(c), kept))
    with torch.inference_mode():
        inferred = _prompt(blk, 2, 30, 256, 128, 512, 2, torch.bfloat16, rotary)
    with torch.no_grad():
        for x, n in ((xs[0], 1), (many, 5)):
            f = rotary.get_freqs_cis(30, 30 + n)
            a, b = blk(x, f, None, inferred), blk(x, f, None, cache)
            assert torch.equal(a[0], b[0]) and all(torch.equal(s, t) for s, t in zip(_tensors(a[1]), _tensors(b[1])))


def test_two_streams_continue_one_cache():
    """One stream's continuation is dropped while its kernels still wait; the other's has to stay what it is."""
    blk = _block(256, 128, 512, 512, 2, 2, 512)
    rotary = RotaryEmbedding(64, 512).cuda()
    xs = [torch.randn(2, 1, 256, generator=torch.Generator().manual_seed(s)).bfloat16().cuda() for s in range(2)]
    freqs = rotary.get_freqs_cis(300, 301)
    with torch.no_grad():
        cache = _prompt(blk, 2, 300, 256, 128, 512, 2, torch.bfloat16, rotary)
        before = [t.clone() for t in _tensors(cache)]
        wanted = [decode_step(blk, x, freqs, cache) for x in xs]
        late, early = torch.cuda.Stream(), torch.cuda.Stream()
        torch.cuda.synchronize()
        for _ in range(3):
            with torch.cuda.stream(late):
                torch.cuda._sleep(10_000_000)
                first = decode_step(blk, xs[0], freqs, cache)[0]
            with torch.cuda.stream(early):
                y, kept = decode_step(blk, xs[1], freqs, cache)
            torch.cuda.synchronize()
            assert torch.equal(first, wanted[0][0]) and torch.equal(y, wanted[1][0])
            assert all(torch.equal(a, b) for a, b in zip(_tensors(kept), _tensors(wanted[1][1])))
            assert all(torch.equal(a, b) for a, b in zip(_tensors(cache), before))


@pytest.mark.parametrize("part", ["mega", "mega.inner_attention", "nffn"])
def test_submodule_in_training_mode_keeps_its_dropout(part):
    """`block.eval()` and one submodule back in training mode, for instance for Monte Carlo dropout."""
    blk = _block(256, 128, 512, 512, 2, 2, 512, dropout=0.5, attention_dropout=0.5, hidden_dropout=0.5)
    rotary = RotaryEmbedding(64, 512).cuda()
    x = torch.randn(2, 1, 256, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    with torch.no_grad():
        cache = _prompt(blk, 2, 30, 256, 128, 512, 2, torch.bfloat16, rotary)
        freqs = rotary.get_freqs_cis(30, 31)
        a, b = (blk(x, freqs, None, cache)[0] for _ in range(2))
        assert torch.equal(a, b)
        blk.get_submodule(part).training = True
        assert decode_step(blk, x, freqs, cache) is None
        a, b = (blk(x, freqs, None, cache)[0] for _ in range(2))
        assert not torch.equal(a, b)


def test_cache_of_a_whole_chunk_is_refused():
    blk = _block(256, 128, 512, 512, 2, 2, 64)
    rotary = RotaryEmbedding(64, 128).cuda()
    x = torch.randn(2, 1, 256, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    with torch.no_grad():
        attn, norm, h = _prompt(blk, 2, 63, 256, 128, 512, 2, torch.bfloat16, rotary)
        keys, values = (torch.cat((t, t[:, :2]), dim=1) for t in attn[:2])
        with pytest.raises(RuntimeError):
            blk(x, rotary.get_freqs_cis(65, 66), None, ((keys, values, 65), norm, h))


@pytest.mark.parametrize("name,shape", [
    ("mega.wr.weight", (480, 256)), ("mega.wr.bias", (480,)), ("mega.wh2.weight", (256, 480)), ("mega.wh1.weight", (128, 512)),
    ("mega.gamma", (2, 64)), ("nffn.fc3.weight", (480, 256)), ("nffn.fc2.weight", (512, 256)), ("mega.rmsnorm.weight", (128,)),
    ("mega.cema.omega", (128, 1)),
])
def test_weights_of_other_shapes_are_refused(name, shape):
    """As the operators do; the step's kernels take the shapes from the block's first weights."""
    blk = _block(256, 128, 512, 512, 2, 2, 64)
    rotary = RotaryEmbedding(64, 64).cuda()
    x = torch.randn(2, 1, 256, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    with torch.no_grad():
        cache = _prompt(blk, 2, 9, 256, 128, 512, 2, torch.bfloat16, rotary)
        owner, leaf = name.rsplit(".", 1)
        setattr(blk.get_submodule(owner), leaf, torch.nn.Parameter(torch.zeros(shape, dtype=torch.bfloat16, device="cuda")))
        with pytest.raises(RuntimeError):
            decode_step(blk, x, rotary.get_freqs_cis(9, 10), cache) or blk(x, rotary.get_freqs_cis(9, 10), None, cache)


def test_step_in_a_graph():
    """A captured step replays on what its input tensors hold then, and leaves the cache that it reads alone."""
    blk = _block(256, 128, 512, 512, 2, 2, 512)
    rotary = RotaryEmbedding(64, 512).cuda()
    xs = [torch.randn(2, 1, 256, generator=torch.Generator().manual_seed(s)).bfloat16().cuda() for s in range(4)]
    freqs = rotary.get_freqs_cis(30, 31)
    with torch.no_grad():
        cache = _prompt(blk, 2, 30, 256, 128, 512, 2, torch.bfloat16, rotary)
        before = [t.clone() for t in _tensors(cache)]
        wanted = [decode_step(blk, x, freqs, cache) for x in xs]
        x = xs[0].clone()
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            decode_step(blk, x, freqs, cache)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            y, after = decode_step(blk, x, freqs, cache)
        for source, (out, kept) in zip(xs, wanted):
            x.copy_(source)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, out) and all(torch.equal(a, b) for a, b in zip(_tensors(after), _tensors(kept)))
            assert all(torch.equal(a, b) for a, b in zip(_tensors(cache), before))
