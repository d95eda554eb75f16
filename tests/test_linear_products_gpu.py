"""The linear layers' three products on the library's own kernels (`mega_linear_*`), one to three layers of one input in a
launch, against float64: one row, edges of tiles of 128 and 256, tokens off the slabs of 32, layers narrower than a
tile, sizes that take either tile.  A 16-bit result of a float32 accumulation: 2^-8 of each value (bfloat16, float16
2^-11) from its one rounding, in the norm over all of them about half of that, and what the sums themselves are off by."""
import ctypes

import pytest
import torch

from megalodon_amd import _lib
from megalodon_amd.modules.linear import Linear, linear_group

pytestmark = pytest.mark.gpu


def _pointers(tensors):
    return (ctypes.c_void_p * len(tensors))(*[0 if t is None else t.data_ptr() for t in tensors])


def _parts(kind, tokens, n_in, n_out):
    i64 = ctypes.c_int64
    fn = ctypes.CFUNCTYPE(i64, ctypes.c_int, i64, i64, ctypes.c_int, ctypes.c_void_p)(("mega_linear_workspace_bytes", _lib.load()))
    return fn(kind, tokens, n_in, len(n_out), (i64 * len(n_out))(*n_out))


def _poisoned(t):  # NaN behind the last element
    buf = torch.full((t.numel() + 4096,), float("nan"), dtype=t.dtype, device="cuda")
    return buf[:t.numel()].view(t.shape).copy_(t)


def _eps(dtype):
    return 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11


def _sum(a, b, *more):
    """a @ b and summands of its shape in float64, and how far a sum of these terms in float32 can be from it: roundings of
    2^-23 at most (cut off, not to nearest) of no more than the sum of the magnitudes, one for each four terms at
    least (a matrix instruction adds up 16 or 8), one for each summand and a few for parts that are added up."""
    want, size = a @ b, a.abs() @ b.abs()
    for m in more:
        want, size = want + m, size + m.abs()
    return want, size * ((a.shape[-1] / 4 + 16) * 2.0 ** -23)


def _close(got, want, reach=None):
    """In the norm, and with `reach` (the sum's own error) every value: a rounding of what is off by that much."""
    eps = _eps(got.dtype)
    assert torch.isfinite(got.float()).all()
    assert (got.double() - want).norm() <= eps * want.norm()
    if reach is not None:
        assert ((got.double() - want).abs() <= eps * want.abs() + (1 + eps) * reach).all()


@pytest.mark.parametrize("tokens,n_in,n_out,dtype", [
    (1, 64, [64], torch.bfloat16),
    (33, 64, [64, 128], torch.float16),
    (127, 192, [192], torch.bfloat16),
    (129, 128, [64, 320, 128], torch.bfloat16),
    (256, 256, [256, 128, 64], torch.float16),
    (257, 320, [192], torch.bfloat16),
    (1021, 2048, [512, 4096, 2048], torch.bfloat16),   # tiles of 256 for the weight gradients
    (1021, 5504, [2048], torch.bfloat16),
    (2048, 2048, [5504], torch.float16),
    (4084, 1024, [2752, 2752], torch.bfloat16),        # tiles of 256 forward
    (4084, 2048, [512, 4096, 2048], torch.bfloat16),   # and for the weight gradients
    (4100, 704, [2048, 64], torch.float16),
])
def test_products_match_float64(tokens, n_in, n_out, dtype):
    g = torch.Generator("cuda").manual_seed(tokens + n_in)
    rows = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x = _poisoned(rows(tokens, n_in).to(dtype))
    w = [_poisoned((rows(o, n_in) / n_in ** 0.5).to(dtype)) for o in n_out]
    bias = [rows(o).to(dtype) if i != 1 else None for i, o in enumerate(n_out)]
    dy = [_poisoned(rows(tokens, o).to(dtype)) for o in n_out]
    add, code, i64 = rows(tokens, n_out[0]).to(dtype), _lib.dtype_code(dtype), ctypes.c_int64
    y = [torch.empty(tokens, o, dtype=dtype, device="cuda") for o in n_out]
    dw = [torch.empty_like(t) for t in w]
    outs, s = (i64 * len(n_out))(*n_out), _lib.stream_ptr(x.device)
    call = lambda name, *a: _lib.call(name, *a, s)

    def fwd(w, bias, add, n_out, y, cut=True):
        n, outs = len(w), (i64 * len(w))(*n_out)
        size = _parts(0, tokens, n_in, n_out) if cut else 0
        ws = torch.empty(size, dtype=torch.uint8, device="cuda")
        call("mega_linear_fwd", _lib.ptr(x), _pointers(w), bias and _pointers(bias), add, _lib.i32(code), i64(tokens), i64(n_in), _lib.i32(n), outs, _pointers(y), _lib.ptr(ws) if size else None)

    fwd(w, bias, None, n_out, y)
    size = _parts(2, tokens, n_in, n_out)
    ws = torch.empty(size, dtype=torch.uint8, device="cuda")
    call("mega_linear_weight_grads", _pointers(dy), _lib.ptr(x), _lib.i32(code), i64(tokens), i64(n_in), _lib.i32(len(w)), outs, _pointers(dw), _lib.ptr(ws) if size else None)
    x64, w64, dy64 = x.double(), [t.double() for t in w], [t.double() for t in dy]
    for i in range(len(w)):
        forward = _sum(x64, w64[i].t(), *([] if bias[i] is None else [bias[i].double()]))
        _close(y[i], *forward)
        _close(dw[i], *_sum(dy64[i].t(), x64))
        # one layer alone gives the same bits as in the group, where neither is cut
        if len(w) > 1:
            alone, whole = torch.empty_like(y[i]), [torch.empty_like(t) for t in y]
            fwd([w[i]], [bias[i]], None, [n_out[i]], [alone], cut=False)
            fwd(w, bias, None, n_out, whole, cut=False)
            assert torch.equal(alone, whole[i])
            _close(alone, *forward)
    fwd(w[:1], None, _lib.ptr(add), n_out[:1], y[:1])
    _close(y[0], *_sum(x64, w64[0].t(), add.double()))
    dx = torch.empty_like(x)
    for i in range(len(w)):  # added up in place
        before = dx.double()
        call("mega_linear_input_grad", _pointers(dy[i:i + 1]), _pointers(w[i:i + 1]), _lib.ptr(dx) if i else None, _lib.i32(code), i64(tokens), i64(n_in), _lib.i32(1), (i64 * 1)(n_out[i]), _lib.ptr(dx))
        _close(dx, *_sum(dy64[i], w64[i], *([before] if i else [])))
    # all of the layers at once, onto a summand
    start = rows(tokens, n_in).to(dtype)
    dx = torch.full_like(start, float("nan"))
    call("mega_linear_input_grad", _pointers(dy), _pointers(w), _lib.ptr(start), _lib.i32(code), i64(tokens), i64(n_in), _lib.i32(len(w)), outs, _lib.ptr(dx))
    _close(dx, *_sum(torch.cat(dy64, 1), torch.cat(w64), start.double()))


@pytest.mark.parametrize("tokens,n_in,n_out,dtype", [
    (4096, 2752, [1024], torch.bfloat16),
    (4093, 2752, [1024], torch.float16),           # rows that end inside a tile
    (4093, 2744, [1024, 512], torch.bfloat16),     # columns too; two layers, one after the other
])
@pytest.mark.parametrize("onto", ["nothing", "summand", "itself"])
def test_input_gradients_in_tiles_of_256(tokens, n_in, n_out, dtype, onto):
    """Sizes whose input gradients take the large tiles, a launch and a rounding for each layer: without a summand, with one, and
    with the result's own memory as the summand."""
    g = torch.Generator("cuda").manual_seed(tokens + len(onto))
    rows = lambda *s: _poisoned(torch.randn(*s, generator=g, device="cuda").to(dtype))
    dy, w, i64 = [rows(tokens, o) for o in n_out], [rows(o, n_in) for o in n_out], ctypes.c_int64
    start = rows(tokens, n_in)
    behind = torch.full((tokens * n_in + 4096,), float("nan"), dtype=dtype, device="cuda")
    dx = behind[:tokens * n_in].view(tokens, n_in)
    if onto == "itself":
        dx.copy_(start)
    add = {"nothing": None, "summand": _lib.ptr(start), "itself": _lib.ptr(dx)}[onto]
    _lib.call("mega_linear_input_grad", _pointers(dy), _pointers(w), add, _lib.i32(_lib.dtype_code(dtype)), i64(tokens), i64(n_in),
              _lib.i32(len(w)), (i64 * len(w))(*n_out), _lib.ptr(dx), _lib.stream_ptr(dx.device))
    want, reach = (0, 0) if onto == "nothing" else (start.double(), 0)
    for i in range(len(w)):  # what the sum so far is off by, its rounding included, goes into the next
        before = reach if i == 0 else reach + _eps(dtype) * (want.abs() + reach)
        want, own = _sum(dy[i].double(), w[i].double(), *([] if onto == "nothing" and i == 0 else [want]))
        reach = before + own
    _close(dx, want, reach)
    assert behind[tokens * n_in:].isnan().all()


def test_refused_sizes():
    fn = _lib.load().mega_linear_takes
    i64 = ctypes.c_int64
    takes = lambda kind, tokens, n_in, *n_out: fn(kind, 1, i64(tokens), i64(n_in), len(n_out), (i64 * len(n_out))(*n_out))
    assert takes(0, 100, 256, 256) and takes(1, 100, 256, 256) and takes(2, 100, 256, 72)
    for kind, sizes in [(0, (100, 72, 64)), (1, (100, 64, 72)), (2, (100, 64, 77)), (2, (0, 64, 64)), (0, (1 << 24, 64, 64)),
                        (0, (8, 64, 64, 64, 64, 64)), (3, (64, 64, 64))]:
        assert not takes(kind, *sizes)


@pytest.mark.parametrize("tokens,sizes", [(40, (128, 64)), (300, (192, 320))])
def test_layers_whose_operands_need_the_general_path(tokens, sizes):
    """Transposed and misaligned operands, broadcast residuals, more layers than a launch takes, a vmapped backward: as ever."""
    torch.manual_seed(tokens)
    n_in, n_out = sizes
    layer = Linear(n_in, n_out, bias=False).cuda().bfloat16()
    x = torch.randn(tokens, n_in, device="cuda").bfloat16()
    want = x.double() @ layer.weight.double().t()
    with torch.no_grad():
        _close(layer(x.t().contiguous().t()), want)
        shifted = torch.empty(tokens * n_in + 1, dtype=x.dtype, device="cuda")[1:].view(tokens, n_in).copy_(x)
        _close(layer(shifted), want)
        row = torch.randn(n_out, device="cuda").bfloat16()
        _close(layer(x, residual=row.expand(tokens, n_out)), want + row.double())
        with pytest.raises(RuntimeError):
            layer(x[:, : n_in // 2])
    leaf = x.clone().requires_grad_(True)
    four = [Linear(n_in, n_out).cuda().bfloat16() for _ in range(4)]
    ys = linear_group(leaf, four)
    torch.autograd.backward(ys, [torch.ones_like(y) for y in ys])
    _close(leaf.grad, sum(torch.ones(tokens, n_out, dtype=torch.float64, device="cuda") @ l.weight.double() for l in four))
    y = layer(leaf)
    many = torch.randn(3, tokens, n_out, device="cuda").bfloat16()
    dx, dw = torch.autograd.grad(y, (leaf, layer.weight), many, is_grads_batched=True)
    _close(dx, many.double() @ layer.weight.double())
    _close(dw, torch.stack([g.double().t() @ x.double() for g in many]))


@pytest.mark.parametrize("tokens,n_in,n_out,dtype", [
    (4100, 4096, [4096], torch.bfloat16),             # 272 tiles: 16 left over, the last of four rows
    (1531, 4096, [5504, 5568], torch.float16),        # two layers, layers and rows that end inside a tile
    (1531, 11008, [4096], torch.bfloat16),            # fewer tiles than the chip takes
    (16, 4096, [1024, 2048, 1000], torch.bfloat16),   # one row of tiles of 128, of whose rows most are not there
    (129, 2048, [512, 2048], torch.float16),          # two, one row in the second
])
def test_last_tiles_cut_along_k(tokens, n_in, n_out, dtype):
    """The tiles that a last round of the chip would hold alone, cut along k and added up by a second launch: against
    float64, the same twice (the parts are added in order), and without memory for the parts, where nothing is cut."""
    g = torch.Generator("cuda").manual_seed(tokens)
    rows = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x = _poisoned(rows(tokens, n_in).to(dtype))
    w = [_poisoned((rows(o, n_in) / n_in ** 0.5).to(dtype)) for o in n_out]
    bias, add = [rows(o).to(dtype) for o in n_out], rows(tokens, n_out[0]).to(dtype)
    i64, outs = ctypes.c_int64, (ctypes.c_int64 * len(n_out))(*n_out)
    bytes_, summed = _parts(0, tokens, n_in, n_out), add if len(n_out) == 1 else None
    assert 0 < bytes_ <= 64 << 20

    def run(ws):
        y = [torch.full((tokens, o), float("nan"), dtype=dtype, device="cuda") for o in n_out]
        _lib.call("mega_linear_fwd", _lib.ptr(x), _pointers(w), _pointers(bias), None if summed is None else _lib.ptr(summed),
                  _lib.i32(_lib.dtype_code(dtype)), i64(tokens), i64(n_in), _lib.i32(len(w)), outs, _pointers(y), ws, _lib.stream_ptr(x.device))
        return y

    parts = torch.full((bytes_ + 4096,), 255, dtype=torch.uint8, device="cuda")  # NaN
    once, again, whole = run(_lib.ptr(parts)), run(_lib.ptr(parts)), run(None)
    assert (parts[bytes_:] == 255).all()
    for i, o in enumerate(n_out):
        want = _sum(x.double(), w[i].double().t(), bias[i].double(), *([] if summed is None else [summed.double()]))
        _close(once[i], *want)
        _close(whole[i], *want)
        assert torch.equal(once[i], again[i])


def test_group_without_gradients():
    """One launch where no gradient is wanted: the values of the layers one by one, and their own calls where a layer's call is
    more than its product (hooks, a subclass)."""
    torch.manual_seed(3)
    layers = [Linear(1024, o, bias=b).cuda().bfloat16() for o, b in ((256, True), (2048, False), (1024, True))]
    x = torch.randn(500, 1024, device="cuda").bfloat16()
    with torch.no_grad():
        for y, l in zip(linear_group(x, layers), layers):
            _close(y, x.double() @ l.weight.double().t() + (0 if l.bias is None else l.bias.double()))
        seen = []
        hook = layers[1].register_forward_hook(lambda m, a, y: seen.append(y) or y + 1)
        y = linear_group(x, layers)[1]
        assert len(seen) == 1 and torch.equal(y, seen[0] + 1)
        hook.remove()

        class Twice(Linear):
            def forward(self, x, residual=None):
                return 2 * super().forward(x, residual)

        layers[0].__class__ = Twice
        assert torch.equal(linear_group(x, layers)[0], layers[0](x))


def test_products_that_a_mode_watches():
    """Fake tensors have no memory to launch on, and a mode that counts operations has to see the products."""
    from torch._subclasses import FakeTensorMode
    from torch.utils.flop_counter import FlopCounterMode
    layers = [Linear(256, 128).cuda().bfloat16() for _ in range(2)]
    x = torch.randn(64, 256, device="cuda").bfloat16().requires_grad_(True)
    with FlopCounterMode(display=False) as counter:
        y = layers[0](x)
        y.backward(torch.ones_like(y))
        with torch.no_grad():
            linear_group(x, layers)
    assert counter.get_total_flops() == 5 * 2 * 64 * 256 * 128
    with FakeTensorMode(), torch.no_grad():
        fake = Linear(256, 128, device="cuda", dtype=torch.bfloat16)
        assert fake(torch.empty(64, 256, device="cuda", dtype=torch.bfloat16)).shape == (64, 128)


@pytest.mark.parametrize("size", [256, 4096])  # 4096^3: the input gradient takes a transposed copy of the weight
def test_gradients_that_a_mode_watches(size):
    from torch._subclasses import FakeTensorMode
    with FakeTensorMode():
        fake = Linear(size, size, device="cuda", dtype=torch.bfloat16)
        x = torch.empty(size, size, device="cuda", dtype=torch.bfloat16, requires_grad=True)
        y = fake(x)
        grads = torch.autograd.grad(y, (x, fake.weight, fake.bias), torch.empty_like(y))
        assert [tuple(g.shape) for g in grads] == [(size, size), (size, size), (size,)]
    layer = Linear(256, 128).cuda().bfloat16()
    y = layer(torch.randn(64, 256, device="cuda").bfloat16())
    db, = torch.autograd.grad(y, layer.bias, torch._efficientzerotensor((64, 128), dtype=y.dtype, device="cuda"))
    assert torch.equal(db, torch.zeros_like(layer.bias))


def test_products_of_tensors_without_memory():
    """Functional wrappers and zeros that are never written have a storage, but nothing in it to launch on."""
    torch.manual_seed(9)
    layers = [Linear(256, o, bias=b).cuda().bfloat16() for o, b in ((128, True), (64, False))]
    x, residual = torch.randn(64, 256, device="cuda").bfloat16(), torch.randn(64, 64, device="cuda").bfloat16()
    with torch.no_grad():
        for y, l in zip(torch.func.functionalize(lambda x: linear_group(x, layers))(x), layers):
            _close(y, x.double() @ l.weight.double().t() + (0 if l.bias is None else l.bias.double()))
        y = torch.func.functionalize(lambda x, r: layers[1](x, r))(x, residual)
        _close(y, x.double() @ layers[1].weight.double().t() + residual.double())
    leaf = x.clone().requires_grad_(True)
    ys = (layers[1](leaf), *linear_group(leaf, layers))
    zeros = [torch._efficientzerotensor(tuple(y.shape), dtype=y.dtype, device=y.device) for y in ys]
    for wanted in ((ys[:1], zeros[:1]), (ys[1:], zeros[1:])):
        grads = torch.autograd.grad(wanted[0], [leaf, layers[1].weight], wanted[1], retain_graph=True)
        assert all(torch.equal(g, torch.zeros_like(t)) for g, t in zip(grads, [leaf, layers[1].weight]))


class _Layers(torch.nn.Module):
    def __init__(self):
        super().__init__()
        self.one, self.two, self.three = Linear(256, 128), Linear(256, 128, bias=False), Linear(256, 64)

    def forward(self, x, residual):
        return self.one(x), self.two(x, residual), *linear_group(x, [self.one, self.three])


@pytest.mark.parametrize("gradients", [False, True])
def test_products_that_are_traced(gradients):
    """A trace holds the products themselves: called with other inputs it gives what the layers give."""
    torch.manual_seed(5)
    layers = _Layers().cuda().bfloat16()
    draw = lambda: (torch.randn(64, 256, device="cuda").bfloat16(), torch.randn(64, 128, device="cuda").bfloat16())
    with torch.set_grad_enabled(gradients):
        traced = torch.jit.trace(layers, draw(), check_trace=False)
        x, residual = draw()
        got = traced(x, residual)
        weights = [(layers.one, None), (layers.two, residual), (layers.one, None), (layers.three, None)]
        for y, (l, r) in zip(got, weights):
            _close(y.detach(), x.double() @ l.weight.detach().double().t() + (0 if l.bias is None else l.bias.detach().double())
                   + (0 if r is None else r.double()))
        assert all(y.requires_grad == gradients for y in got)


def test_products_under_capture():
    """Captured: layers of one input with last tiles cut along k (parts from the graph's pool), replayed on other inputs with
    eager work between."""
    torch.manual_seed(7)
    layers = [Linear(4096, o).cuda().bfloat16() for o in (5504, 5504)]
    tokens = 1531
    assert _parts(0, tokens, 4096, (5504, 5504)) > 0
    x = torch.randn(tokens, 4096, device="cuda").bfloat16()
    with torch.no_grad():
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            linear_group(x, layers)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            ys = linear_group(x, layers)
        for _ in range(3):
            x.copy_(torch.randn(tokens, 4096, device="cuda"))
            want = linear_group(x, layers)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(ys, want))


@pytest.mark.parametrize("tokens,n_in,n_out,dtype", [
    (4096, 1024, [2048], torch.bfloat16),       # 128 tiles, two parts
    (4093, 1024, [1000], torch.float16),        # 64 tiles that end inside, tokens off the slabs, four parts of unequal length
    (2500, 136, [256, 72], torch.bfloat16),     # two layers, three tiles
])
def test_weight_gradients_cut_along_the_tokens(tokens, n_in, n_out, dtype):
    g = torch.Generator("cuda").manual_seed(tokens)
    rows = lambda *s: _poisoned(torch.randn(*s, generator=g, device="cuda").to(dtype))
    x, dy, i64 = rows(tokens, n_in), [rows(tokens, o) for o in n_out], ctypes.c_int64
    size = _parts(2, tokens, n_in, n_out)
    assert 0 < size <= 64 << 20

    def run(ws):
        dw = [torch.full((o, n_in), float("nan"), dtype=dtype, device="cuda") for o in n_out]
        _lib.call("mega_linear_weight_grads", _pointers(dy), _lib.ptr(x), _lib.i32(_lib.dtype_code(dtype)), i64(tokens), i64(n_in),
                  _lib.i32(len(dy)), (i64 * len(n_out))(*n_out), _pointers(dw), ws, _lib.stream_ptr(x.device))
        return dw

    parts = torch.full((size + 4096,), 255, dtype=torch.uint8, device="cuda")  # NaN
    once, again, whole = run(_lib.ptr(parts)), run(_lib.ptr(parts)), run(None)
    assert (parts[size:] == 255).all()
    for i in range(len(n_out)):
        want = _sum(dy[i].double().t(), x.double())
        _close(once[i], *want)
        _close(whole[i], *want)
        assert torch.equal(once[i], again[i])
