"""A prompt's cache and what stands around `_InnerAttention`: hooks that keep and change their arguments, a forward of the
signature without `fresh`; and the cache goes on to the next call."""
import pytest
import torch

from test_cached_inference_gpu import _block, _empty_cache

pytestmark = pytest.mark.gpu


def _prompt(blk, x):
    with torch.no_grad():
        return blk(x, None, None, _empty_cache(x.shape[0], blk, x.device))


def _next(blk, x, cache):
    with torch.no_grad():
        return blk(x, None, None, cache)[0]


@pytest.mark.parametrize("kind", ["pre", "post", "global"])
def test_a_hook_that_keeps_its_arguments(kind):
    blk = _block(512)
    x, x2 = (torch.randn(2, n, 256, generator=torch.Generator().manual_seed(n)).bfloat16().cuda() for n in (100, 3))
    y, cache = _prompt(blk, x)
    want = _next(blk, x2, cache)
    inner, held = blk.mega.inner_attention, []

    def keep(module, args, *rest):
        if module is inner:
            held.extend(args[1:3])

    handle = {"pre": inner.register_forward_pre_hook, "post": inner.register_forward_hook,
              "global": torch.nn.modules.module.register_module_forward_pre_hook}[kind](keep)
    try:
        y2, cache2 = _prompt(blk, x)
    finally:
        handle.remove()
    assert torch.equal(y, y2) and len(held) == 2
    for t, c in zip(held, cache2[0]):
        assert t.untyped_storage().data_ptr() != c.untyped_storage().data_ptr()
        t.fill_(float("nan"))
    assert torch.equal(_next(blk, x2, cache2), want)


def test_a_forward_without_the_argument():
    blk = _block(512)
    x = torch.randn(1, 40, 256, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    want, _ = _prompt(blk, x)
    inner = blk.mega.inner_attention
    own = inner.forward
    inner.forward = lambda xq, xk, xv, mask, freqs_cis, cache=None: own(xq, xk, xv, mask, freqs_cis, cache)
    got, cache = _prompt(blk, x)
    assert torch.equal(got, want) and cache[0][0].shape[1] == 40


def test_a_cache_goes_on_while_the_first_one_stays():
    blk = _block(512)
    x, x2 = (torch.randn(2, n, 256, generator=torch.Generator().manual_seed(n)).bfloat16().cuda() for n in (64, 7))
    _, cache = _prompt(blk, x)
    before = [t.clone() for t in cache[0][:2]]
    first, again = _next(blk, x2, cache), _next(blk, x2, cache)
    assert torch.equal(first, again)
    for t, b in zip(cache[0], before):
        assert torch.equal(t, b)
