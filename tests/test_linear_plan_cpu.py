"""The choice of tiles for the linear layers' products, and whether they are taken at all (linear_plan.hpp): plain C++, built
with g++ and asked about a chip of 256 compute units."""
import ctypes
import os
import subprocess

import pytest

SRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "linear_plan_emu.cc")
FORWARD, INPUT_GRAD, WEIGHT_GRAD = 0, 1, 2


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    """ask(name, kind, tokens, n_in, *n_out)"""
    out = tmp_path_factory.mktemp("emu") / "liblinear_plan_emu.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-o", str(out), SRC], check=True)
    lib, i64 = ctypes.CDLL(str(out)), ctypes.c_int64
    lib.emu_linear_time.restype = ctypes.c_double

    def call(name, kind, tokens, n_in, *n_out):
        return getattr(lib, "emu_linear_" + name)(kind, i64(tokens), i64(n_in), len(n_out), (i64 * len(n_out))(*n_out), 256)

    return call


@pytest.mark.parametrize("kind,tokens,n_in,n_out,tile", [  # (among them the sizes that stand for a tile in test_linear_products_gpu.py)
    (FORWARD, 1021, 2048, [512, 4096, 2048], 128),
    (FORWARD, 1531, 4096, [11008, 11008], 256),
    (FORWARD, 4084, 1024, [2752, 2752], 256),
    (INPUT_GRAD, 4096, 2752, [1024], 256),                # one layer
    (INPUT_GRAD, 4093, 2752, [1024], 256),
    (INPUT_GRAD, 4093, 2744, [1024, 512], 256),           # one after the other
    (WEIGHT_GRAD, 1021, 2048, [512, 4096, 2048], 256),
    (INPUT_GRAD, 4084, 2048, [512, 4096, 2048], 128),     # joined along k
    (WEIGHT_GRAD, 4084, 2048, [512, 4096, 2048], 256),
])
def test_tiles(ask, kind, tokens, n_in, n_out, tile):
    assert ask("tile", kind, tokens, n_in, *n_out) == tile


def test_input_gradients_one_after_the_other_are_priced_so(ask):
    """Layers that are not joined along k cost a launch each, not one product along all of their outputs, and all but the
    first read and write the sum so far."""
    apart = 0
    for tokens in (500, 2100, 4096, 7000, 10000, 16384):
        for n_in, n_out in ((1024, (2752, 2752)), (1280, (1280, 1280, 1280)), (1024, (256, 2048, 1024))):
            alone = sum(ask("time", INPUT_GRAD, tokens, n_in, n) for n in n_out)
            together = ask("time", INPUT_GRAD, tokens, n_in, *n_out)
            if ask("joined", INPUT_GRAD, tokens, n_in, *n_out):
                assert together < alone
            else:
                assert together == pytest.approx(alone + (len(n_out) - 1) * 2 * tokens * n_in / 2.2e6)
                apart += 1
    assert apart >= 3


# us measured, (library, here): products that the library's tiles fit, which stay there, and products that they do not fit
@pytest.mark.parametrize("kind,tokens,n_in,n_out,library,here", [
    (FORWARD, 1250, 4096, [11008, 11008], 167, 204),
    (FORWARD, 2500, 4096, [11008, 11008], 317, 374),
    (FORWARD, 5000, 4096, [11008, 11008], 616, 666),
    (FORWARD, 12000, 6912, [2560], 269, 332),
    (FORWARD, 3500, 4608, [4608], 98, 118),
    (FORWARD, 4096, 3584, [3584], 72, 89),
    (FORWARD, 32768, 1536, [1536], 112, 137),
    (FORWARD, 32768, 2048, [5504, 5504], 1025, 1149),
    (INPUT_GRAD, 7000, 1280, [1280, 1280, 1280], 87, 117),
    (INPUT_GRAD, 10000, 1024, [2752, 2752], 105, 128),
    (INPUT_GRAD, 2624, 3584, [512, 512], 37, 46),
    (FORWARD, 1, 13824, [4096], 19.6, 27.6),
    (FORWARD, 1, 8192, [9216, 9216], 57, 69),
    (FORWARD, 22, 11008, [5504], 24.8, 34.5),
    (FORWARD, 64, 9216, [13824], 44.5, 54.5),
    (FORWARD, 1344, 2560, [2752], 27, 31),
    (FORWARD, 43, 4096, [11008, 11008], 39, 32),
    (FORWARD, 16, 5504, [2048], 18.5, 21.1),
    (FORWARD, 64, 5504, [2048], 18.3, 23.0),
    (FORWARD, 512, 2752, [1024], 18.4, 20.1),
    (FORWARD, 640, 2752, [1024], 18.4, 20.8),
    (FORWARD, 16, 1024, [1024], 18.3, 9.7),
    (FORWARD, 16, 2048, [512, 4096, 2048], 54.0, 15.5),
    (FORWARD, 384, 2048, [5504, 5504], 39.3, 29.7),
    (INPUT_GRAD, 384, 2752, [1024], 17.6, 10.2),
    (INPUT_GRAD, 100, 2048, [512, 4096, 2048], 53.4, 46.3),
    (FORWARD, 1531, 4096, [11008, 11008], 261, 244),
    (FORWARD, 2100, 4096, [11008, 11008], 566, 335),
    (FORWARD, 4096, 4096, [11008, 11008], 800, 585),
    (FORWARD, 4096, 1024, [2752, 2752], 66, 55),
    (FORWARD, 4096, 2048, [5504, 5504], 169, 151),
    (FORWARD, 1000, 2048, [512, 4096, 2048], 46, 31),
    (INPUT_GRAD, 4096, 1024, [256, 2048, 1024], 48, 31),
    (INPUT_GRAD, 4096, 2752, [1024], 35, 27),
    (WEIGHT_GRAD, 32768, 512, [512], 152, 41),
])
def test_products_go_where_they_are_faster(ask, kind, tokens, n_in, n_out, library, here):
    assert ask("takes", kind, tokens, n_in, *n_out) == (here < library)
