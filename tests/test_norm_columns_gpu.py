"""The norms' backward by columns (widths 512, 1024, 2048, 4096 in 16 bits): row counts around the four rows of a pass, the
workgroups of a launch and its limits, with and without affine parameters, and both sides of the lines to the kernel that takes
a row to a wave.

Bounds: dx is rounded once to the element type (2^-9 in bfloat16, 2^-12 in float16, of the largest values: 4e-3 / 5e-4 of
the 2-norm); the parameters' gradients are float32 sums rounded once."""
import pytest
import torch

from megalodon_amd import _lib
from megalodon_amd import extension as ext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,bar", [(torch.bfloat16, 4e-3), (torch.float16, 5e-4)])
@pytest.mark.parametrize("rms", [False, True])
@pytest.mark.parametrize("rows,D,affine", [(1, 512, "both"), (3, 1024, "both"), (4, 2048, "weight"), (5, 4096, "both"),
                                           (2047, 512, "none"), (2049, 1024, "both"), (2053, 2048, "both"),
                                           (8193, 512, "both"), (16389, 1024, "weight"), (4101, 4096, "none"),
                                           (2048, 512, "both"), (2049, 512, "both"), (3201, 512, "both"), (4097, 512, "weight"),
                                           (2800, 1024, "both"), (2801, 1024, "weight"), (5201, 1024, "both"),
                                           (12288, 2048, "both"), (12289, 2048, "both"), (5, 1024, "none"), (7, 2048, "none")])
def test_backward_matches_float64(rows, D, affine, rms, dtype, bar):
    gen = torch.Generator("cuda").manual_seed(rows + D)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda").to(dtype)
    x, dy = rand(rows, D) + 0.5, rand(rows, D)
    w = 0.1 * rand(D) if affine != "none" else None
    b = 0.1 * rand(D) if affine == "both" and not rms else None
    x[-1, 7] = 100.0  # a row of its own scale, which the unused rows behind the last would repeat
    y, mean, rstd = ext.layer_norm_fwd(x, w, b, 1e-5, rms)
    dx, dw, db = ext.layer_norm_bwd(dy, x, w, mean, rstd, rms, b is not None)
    xd = x.double().requires_grad_(True)
    wd = (w if w is not None else torch.zeros(D, device="cuda")).double().requires_grad_(True)
    c = xd if rms else xd - xd.mean(-1, keepdim=True)
    want = c * torch.rsqrt(c.square().mean(-1, keepdim=True) + 1e-5) * (wd + 1)
    want.backward(dy.double())
    err = lambda got, ref: ((got.double() - ref).norm() / ref.norm()).item()
    assert err(dx, xd.grad) <= bar
    assert err(dx[-1], xd.grad[-1]) <= 2 * bar
    if w is not None:
        assert err(dw, wd.grad) <= bar
    if b is not None:
        assert err(db, dy.double().sum(0)) <= bar


def test_a_workspace_at_any_float():
    rows, D = 100, 2048
    gen = torch.Generator("cuda").manual_seed(7)
    x, dy, w = (torch.randn(*s, generator=gen, device="cuda").bfloat16() for s in ((rows, D), (rows, D), (D,)))
    _, mean, rstd = ext.layer_norm_fwd(x, w, w, 1e-5, False)
    want = ext.layer_norm_bwd(dy, x, w, mean, rstd, False, True)
    size = _lib.load().mega_layer_norm_workspace_bytes
    size.restype = _lib.ctypes.c_int64
    ws = torch.zeros(size(_lib.i64(rows), _lib.i64(D)) // 4 + 3, device="cuda")
    got = [torch.empty_like(t) for t in want]
    _lib.call("mega_layer_norm_bwd", *map(_lib.ptr, (dy, x, w, mean, rstd)), _lib.i32(_lib.dtype_code(x.dtype)), _lib.i64(rows), _lib.i64(D),
              _lib.i32(0), *map(_lib.ptr, got), _lib.ptr(ws[1:]), _lib.stream_ptr(x.device))
    for a, b in zip(got, want):
        assert torch.equal(a, b)
