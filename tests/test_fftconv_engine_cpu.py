"""The register-FFT engine of the convolution kernel, run on the CPU: the
phases in megalodon_amd/csrc/fftconv_core.hpp are plain C++, so a g++ build
emulates one workgroup (lanes one after another, LDS as an array) and is
checked against numpy's float64 FFT.  Catches index / twiddle mistakes
without a GPU."""
import ctypes
import os
import subprocess
import time

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "native", "fftconv_emu.cc")


@pytest.fixture(scope="module")
def emu(tmp_path_factory):
    out = tmp_path_factory.mktemp("emu") / "libfftconv_emu.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", str(out), SRC], check=True)
    return ctypes.CDLL(str(out))


def _p(a):
    return a.ctypes.data_as(ctypes.c_void_p)


@pytest.mark.parametrize("logm", [11, 12, 13, 14])
@pytest.mark.parametrize("h", [0, 1])
def test_half_transform_matches_numpy_fft(emu, logm, h):
    M = 1 << logm
    rng = np.random.default_rng(logm * 2 + h)
    inr = rng.standard_normal(M).astype(np.float32)
    ini = rng.standard_normal(M).astype(np.float32)
    outr = np.zeros(M, np.float32)
    outi = np.zeros(M, np.float32)
    assert emu.emu_fft_half(logm, h, _p(inr), _p(ini), _p(outr), _p(outi)) == 0
    z = inr.astype(np.float64) + 1j * ini.astype(np.float64)
    if h:
        z = z * np.exp(-2j * np.pi * np.arange(M) / (2 * M))
    want = np.fft.fft(z)
    assert np.abs((outr + 1j * outi) - want).max() / np.abs(want).max() < 2e-6


@pytest.mark.parametrize("logm", [11, 12, 13, 14])
def test_convolution_matches_numpy(emu, logm):
    M = 1 << logm
    rng = np.random.default_rng(logm)
    for L in (2 * M, 2 * M - 1, M + 3):
        for flip_a, flip_out in ((0, 0), (1, 1)):
            a = rng.standard_normal(L).astype(np.float32)
            b = rng.standard_normal(L).astype(np.float32)
            y = np.zeros(L, np.float32)
            assert emu.emu_fftconv(logm, _p(a), _p(b), L, flip_a, flip_out, _p(y)) == 0
            aa = a[::-1] if flip_a else a
            n = 4 * M
            want = np.fft.irfft(np.fft.rfft(aa.astype(np.float64), n) * np.fft.rfft(b.astype(np.float64), n), n)[:L]
            if flip_out:
                want = want[::-1]
            assert np.abs(y - want).max() / np.abs(want).max() < 5e-6


def test_rows_are_shared_out_without_looking_at_every_size(emu):
    """The rows of a channel that a workgroup takes: the best of all sizes, the smallest of equals, found in about the square
    root of their number."""
    emu.emu_group_rows.restype = ctypes.c_int64
    i64 = ctypes.c_int64
    choose = lambda B, D, slots, pair, bound: emu.emu_group_rows(i64(B), i64(D), i64(slots), pair, bound)

    def all_sizes(B, D, slots, pair, bound):
        costs = {}
        for nb in range(1, B + 1):
            groups = D * -(-B // nb)
            if not bound or nb == B or groups <= slots:
                costs[nb] = -(-groups // slots) * (nb // 2 * 5 + nb % 2 * 3 if pair == 2 else 3 * nb)
        return min(costs, key=lambda nb: (costs[nb], nb))

    for B in (*range(1, 41), 97, 128, 360, 1001):
        for D in (1, 3, 64, 257, 1024, 4100):
            for slots in (1, 256, 512, 2048):
                for pair in (1, 2):
                    for bound in (0, 1):
                        assert choose(B, D, slots, pair, bound) == all_sizes(B, D, slots, pair, bound), (B, D, slots, pair, bound)
    start = time.perf_counter()
    assert 1 <= choose(10 ** 9, 1, 512, 2, 0) <= 10 ** 9
    assert time.perf_counter() - start < 0.5  # all of them: seconds
