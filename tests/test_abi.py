"""The C-ABI library loads and exports every symbol the public header declares
(no compute calls: runs without a GPU)."""
import ctypes

from megalodon_amd import _lib


def test_library_loads_and_reports_version():
    lib = _lib.load()
    assert lib.mega_version() >= 100
    assert lib.mega_last_error() == b"" or isinstance(lib.mega_last_error(), bytes)


def test_every_declared_symbol_is_exported():
    lib = _lib.load()
    names = _lib.declared_symbols()
    assert "mega_ema_weight_fwd" in names and "mega_version" in names
    missing = [n for n in names if not hasattr(lib, n)]
    assert not missing, f"declared in include/megalodon_hip.h but not exported: {missing}"


def test_invalid_argument_is_reported_not_raised_in_c():
    lib = _lib.load()
    fn = lib.mega_ema_weight_fwd
    fn.restype = ctypes.c_int
    null = ctypes.c_void_p(0)
    code = fn(null, null, null, ctypes.c_int64(1), ctypes.c_int64(16), ctypes.c_int64(8), null, null)
    assert code == 1
    assert b"null" in lib.mega_last_error()


def test_attention_rejects_an_unknown_causal_code():
    """`causal` is 0 (no mask), 1 (mask, whole rows of w written) or 2 (mask, w only as far as
    the backward reads it); anything else is an argument error before any launch."""
    lib = _lib.load()
    fn = lib.mega_attention_fwd
    fn.restype = ctypes.c_int
    null = ctypes.c_void_p(0)
    i64 = ctypes.c_int64
    code = fn(null, null, null, ctypes.c_int(1), i64(1), i64(8), i64(8), i64(1), i64(64), i64(64),
              ctypes.c_double(1.0), ctypes.c_int(3), null, null, null, null)
    assert code == 1
    assert b"causal" in lib.mega_last_error()


def test_attention_layer_pads_only_what_the_scores_kernel_writes():
    """Rows and columns behind the real ones exist only where the kernel that writes them takes the call: the same
    sizes and scales, or the forward would refuse what plain rows take."""
    fn = _lib.load().mega_attention_layer_saved_elements
    fn.restype = ctypes.c_int64
    i64 = ctypes.c_int64

    def saved(L, heads, width, scale, dtype=1):
        return fn(ctypes.c_int(dtype), i64(1), i64(L), i64(L), i64(heads), i64(width), i64(64), ctypes.c_double(scale))

    assert saved(1021, 2, 256, 1.0) == 2 * 1024 * 1024
    for scale in (1e30, 3e38, 1e300, 0.0, -1.0, float("nan")):
        assert saved(1021, 2, 256, scale) == 2 * 1021 * 1021
    assert saved(1021, 5000, 256, 1.0) == 5000 * 1021 * 1021   # a batch entry of 2^30 elements and more
    assert saved(1021, 2, 96, 1.0) == 2 * 1021 * 1021
    assert saved(1021, 2, 256, 1.0, dtype=0) == 2 * 1021 * 1021


def test_questions_about_linear_layers_leave_the_last_error():
    """Whether a launch takes a size and what memory it wants are questions: no is an answer, not an error."""
    lib = _lib.load()
    i64, null = ctypes.c_int64, ctypes.c_void_p(0)
    one = (i64 * 1)(77)
    assert lib.mega_linear_fwd(null, null, null, null, ctypes.c_int(1), i64(100), i64(64), ctypes.c_int(1), one, null, null, null) == 1
    before = lib.mega_last_error()
    assert before == b"mega_linear_fwd: bad sizes"
    lib.mega_linear_workspace_bytes.restype = i64
    for kind, dtype, tokens, n_in, count in [(0, 1, 100, 64, 1), (1, 1, 100, 64, 1), (2, 1, 100, 64, 1), (2, 0, 100, 64, 1), (2, 1, 0, 64, 1), (0, 1, 100, 64, 4)]:
        assert lib.mega_linear_takes(ctypes.c_int(kind), ctypes.c_int(dtype), i64(tokens), i64(n_in), ctypes.c_int(count), one) == 0
        assert lib.mega_linear_workspace_bytes(ctypes.c_int(kind), i64(tokens), i64(n_in), ctypes.c_int(count), one) == 0
    assert lib.mega_last_error() == before
