"""The convolution engine's passes as the kernels run them, on the CPU (tests/native/fftconv_emu.cc), against
numpy's float64 FFT.

Bounds: a transform is log2 M <= 14 butterflies deep, each a rounding or two of 2^-24 beside a twiddle that is at most three
squarings from a table value (an error of 8 x 2^-25 there), errors adding up as squares: below 1e-6 in the 2-norm, of a
convolution (three transforms and a product) below 1.5e-6.  Measured 1.5e-7 .. 3e-7 and 2.6e-7 .. 7.5e-7."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

SRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "fftconv_emu.cc")


@pytest.fixture(scope="module")
def emu(tmp_path_factory):
    out = tmp_path_factory.mktemp("emu") / "libfftconv_emu.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", str(out), SRC], check=True)
    return ctypes.CDLL(str(out))


def _p(a):
    return a.ctypes.data_as(ctypes.c_void_p)


@pytest.mark.parametrize("logm", [11, 12, 13, 14])
@pytest.mark.parametrize("h", [0, 1])
def test_half_transform(emu, logm, h):
    M = 1 << logm
    rng = np.random.default_rng(31 * logm + h)
    inr, ini = (rng.standard_normal(M).astype(np.float32) for _ in range(2))
    outr, outi = np.zeros(M, np.float32), np.zeros(M, np.float32)
    assert emu.emu_fft_half(logm, h, _p(inr), _p(ini), _p(outr), _p(outi)) == 0
    z = inr.astype(np.float64) + 1j * ini
    if h:
        z = z * np.exp(-2j * np.pi * np.arange(M) / (2 * M))
    want = np.fft.fft(z)
    assert np.linalg.norm(outr + 1j * outi - want) / np.linalg.norm(want) < 1e-6


@pytest.mark.parametrize("logm", [11, 12, 13, 14])
@pytest.mark.parametrize("flip", [0, 1])
def test_convolution(emu, logm, flip):
    M = 1 << logm
    rng = np.random.default_rng(logm)
    for L in (2 * M, 2 * M - 1, M + 1, M + 2):
        a, b = (rng.standard_normal(L).astype(np.float32) for _ in range(2))
        y = np.zeros(L, np.float32)
        assert emu.emu_fftconv(logm, _p(a), _p(b), L, flip, flip, _p(y)) == 0
        aa = a[::-1] if flip else a
        n = 4 * M
        want = np.fft.irfft(np.fft.rfft(aa.astype(np.float64), n) * np.fft.rfft(b.astype(np.float64), n), n)[:L]
        if flip:
            want = want[::-1]
        assert np.linalg.norm(y - want) / np.linalg.norm(want) < 1.5e-6
