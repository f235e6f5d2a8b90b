"""CPU check of the mixed-radix LDS FFT (curig_amd/csrc/fft_mix.h): the code the
GPU kernels run, threads emulated by loops, every access bounds-checked, against
numpy.fft, over the lengths 2^a 3^b 5^c a grid axis can have."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "native", "fft_mix_check.cpp")
CSRC = os.path.join(ROOT, "curig_amd", "csrc")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("fftm") / "libfftm.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, "-o", out, SRC])
    L = ctypes.cdll.LoadLibrary(out)
    L.fftm_check_run.argtypes = [ctypes.c_int] * 5 + [np.ctypeslib.ndpointer(np.float64, flags="C"),
                                                      np.ctypeslib.ndpointer(np.int32, flags="C")]
    L.fftm_check_run.restype = ctypes.c_int
    return L


def _smooth(limit):
    return sorted(2 ** a * 3 ** b * 5 ** c for a in range(1, 15) for b in range(9) for c in range(7)
                  if 2 ** a * 3 ** b * 5 ** c <= limit)


def _run(lib, x, nt, sign, dbl):
    count, n = x.shape
    data = np.ascontiguousarray(np.stack([x.real, x.imag], -1).reshape(-1))
    rad = np.zeros(14, np.int32)
    code = lib.fftm_check_run(n, count, nt, sign, dbl, data, rad)
    return code, data.reshape(-1, 2) @ np.array([1, 1j]), rad[rad > 0]


def _threads(n, count, nb_elems=12):
    return max(64, -(-n * count // (64 * nb_elems)) * 64)


@pytest.mark.parametrize("n", _smooth(2000) + [2250, 2592, 3000, 3750, 4374, 5000, 6000, 6250, 7500, 8100, 10000, 12288,
                                               14580, 15000, 16200])
def test_length(lib, n):
    rng = np.random.default_rng(n)
    for count, sign in ((1, 1), (3, -1)):
        if n * count > 16400:
            continue
        x = rng.standard_normal((count, n)) + 1j * rng.standard_normal((count, n))
        want = np.fft.ifft(x, axis=1) * n if sign > 0 else np.fft.fft(x, axis=1)
        code, got, rad = _run(lib, x, _threads(n, count), sign, 1)
        assert code == 0 and np.prod(rad) == n
        assert np.max(np.abs(got.reshape(count, n) - want)) < 1e-12 * np.max(np.abs(want))
        code, got, _ = _run(lib, x, _threads(n, count), sign, 0)
        e = np.linalg.norm(got.reshape(count, n) - want) / np.linalg.norm(want)
        assert code == 0 and e < 4e-7


def test_refused(lib):
    x = np.zeros((1, 14), complex)
    assert _run(lib, x, 64, 1, 1)[0] == 1  # 7 is no radix
    x = np.zeros((1, 6000), complex)
    assert _run(lib, x, 64, 1, 1)[0] == 1  # more butterflies than the threads hold
