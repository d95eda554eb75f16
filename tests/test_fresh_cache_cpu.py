"""What a new cache is made of: `_InnerAttention._joined` is `torch.cat` but behind an empty cache of the same layout, where
a tensor that the caller has made for the call is taken as it is."""
import pytest
import torch

from megalodon_amd.modules.chunk_attention import _InnerAttention, takes_fresh


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, dtype=dtype)


NEW = torch.arange(2 * 5 * 3 * 4, dtype=torch.float32).view(2, 5, 3, 4)


def test_an_empty_cache_takes_a_fresh_tensor():
    assert _InnerAttention._joined(_empty(2, 0, 3, 4), NEW, True) is NEW


@pytest.mark.parametrize("old,new,fresh", [
    (_empty(2, 0, 3, 4), NEW, False),                                    # a caller's own tensor
    (NEW[:, :2], NEW, True),                                             # a cache with keys
    (_empty(2, 0, 3, 4, dtype=torch.float64), NEW, True),                # promoted
    (_empty(2, 0, 3, 4), NEW.transpose(0, 1).contiguous().transpose(0, 1), True),  # not contiguous
    (_empty(2, 0, 3, 4).requires_grad_(True), NEW, True),                # a graph
    (_empty(0), NEW, True),                                              # an empty of one dimension, which cat skips
])
def test_everything_else_is_joined(old, new, fresh):
    got, want = _InnerAttention._joined(old, new, fresh), torch.cat((old, new), dim=1)
    assert got is not new and got.data_ptr() != new.data_ptr()
    assert got.dtype == want.dtype and got.stride() == want.stride() and got.requires_grad == want.requires_grad
    assert torch.equal(got, want)


@pytest.mark.parametrize("shape", [(3, 0, 3, 4), (2, 0, 2, 4), (2, 0, 3, 5)])
def test_other_shapes_are_refused_as_before(shape):
    with pytest.raises(RuntimeError):
        torch.cat((_empty(*shape), NEW), dim=1)
    with pytest.raises(RuntimeError):
        _InnerAttention._joined(_empty(*shape), NEW, True)


def _inner():
    return _InnerAttention(4, 8, 2, 16, 0.0, None)


class _Sub(_InnerAttention):
    pass


def test_who_is_told():
    assert takes_fresh(_inner())
    assert not takes_fresh(_Sub(4, 8, 2, 16, 0.0, None)) and not takes_fresh(torch.nn.Identity())
    m = _inner()
    m.forward = lambda q, k, v, mask, freqs, cache=None: (v, None)
    assert not takes_fresh(m)
    for listen in ("register_forward_hook", "register_forward_pre_hook"):
        m = _inner()
        handle = getattr(m, listen)(lambda *a: None)
        assert not takes_fresh(m)
        handle.remove()
        assert takes_fresh(m)
        handle = getattr(torch.nn.modules.module, listen.replace("register", "register_module"))(lambda *a: None)
        assert not takes_fresh(m)
        handle.remove()
        assert takes_fresh(m)


def test_a_forward_in_the_class_place_is_not_told(monkeypatch):
    monkeypatch.setattr(_InnerAttention, "forward", lambda self, q, k, v, mask, freqs, cache=None: (v, None))
    assert not takes_fresh(_inner())
