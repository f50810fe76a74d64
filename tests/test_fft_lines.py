"""The power-of-two butterflies and their twiddle seeds (swem_fft.hpp), compiled for the host and run line by
line: against the 64-bit transform, and the error that many of them leave in a march.

A march repeats one transform with the same table entries at every depth, so the rounding of the entries
(half a unit in the last place of each part) adds up over the depths while the rounding of the sums does
not.  A line of 256 points takes four radix-4 levels, hence at most one entry per level and input; its march
may be no further from 64 bits than one of plain products and sums with those same entries.  What differs
between the two is the rounding of the sums, which is a few per cent of the error of 200 depths: bound 1.05.
The same holds for lengths with factors 7, 11 and 13, whose passes take one table entry per input, against
the same butterflies with those entries.
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "seismic.jl_amd", "csrc")
SIZES = [(128, 2), (128, 8), (128, 16), (256, 4), (256, 8), (256, 16), (512, 8), (1024, 8), (1024, 16), (2048, 8),
         (2048, 16), (4096, 16)]


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("fft") / "fft_lines.so")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-O2", "-std=c++17", "-mfma", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", f"-I{rocm}/include",
                    f"-I{CSRC}", os.path.join(HERE, "fft_lines.cpp"), "-o", out], check=True)
    return ctypes.CDLL(out)


def _floats(z):
    return np.ascontiguousarray(np.stack([z.real, z.imag], -1).astype(np.float32))


def _ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


@pytest.mark.parametrize("half", [0, 1])
@pytest.mark.parametrize("sign", [-1, 1])
@pytest.mark.parametrize("n,p", SIZES)
def test_line(lib, n, p, sign, half):
    rng = np.random.default_rng(n + p)
    z = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    x = _floats(z)
    if half:
        x[n // 2:] = 0
    ref = x.astype(np.float64) @ [1, 1j]
    ref = np.fft.fft(ref) if sign < 0 else np.fft.ifft(ref) * n
    if half:
        x[n // 2:] = np.nan  # not read
    assert lib.fft_lines(n, p, sign, half, _ptr(x)) == 0
    err = np.linalg.norm(x.astype(np.float64) @ [1, 1j] - ref) / np.linalg.norm(ref)
    # each of the log2 n levels rounds a product and two sums: 3 rms roundings of 2^-24 / sqrt(3) each
    assert err <= np.sqrt(3 * np.log2(n)) * 2.0 ** -24


def _case(n, s):
    """(phase of a step, start) of the s-th medium"""
    k = np.minimum(np.arange(n), n - np.arange(n))
    a = 1.0 - (k / ((0.2 + 0.02 * s) * n)) ** 2
    phase = np.where(a > 0, np.exp(1j * (3 + 0.5 * s) * np.sqrt(np.abs(a))), np.exp(-1.2 * np.sqrt(np.abs(a)))) / n
    z = np.zeros(n, complex)
    z[n // 8 + s * n // 40] = 1 + 0.3j
    return phase, z


def _errors(n, steps, media, run):
    """mean errors of run(0, ...) and run(1, ...) over some media"""
    e = np.zeros(2)
    for s in range(media):
        phase, z = _case(n, s)
        ph, x = _floats(phase), [_floats(z), _floats(z)]
        z = x[0].astype(np.float64) @ [1, 1j]
        for _ in range(steps):
            z = np.fft.ifft(np.fft.fft(z) * phase) * n
            z[n // 2:] = 0
        for i in (0, 1):
            assert run(i, _ptr(x[i]), _ptr(ph), steps) == 0
            e[i] += np.linalg.norm(x[i].astype(np.float64) @ [1, 1j] - z) / np.linalg.norm(z) / media
    return e


@pytest.mark.parametrize("p", [4, 8, 16])
def test_march_error_of_256_points(lib, p):
    mine, plain = _errors(256, 200, 12, lambda i, x, ph, n: lib.fft_march_256(0 if i else p, x, ph, n))
    print(f"{p} points per thread: {mine:.2e}, plain {plain:.2e}")
    assert mine <= 1.05 * plain


@pytest.mark.parametrize("n", [91, 140, 700, 1014, 2002])
def test_march_error_with_prime_factors(lib, n):
    mine, plain = _errors(n, 60, 4, lambda i, x, ph, k: lib.mixed_march(n, i, x, ph, k, 0))
    print(f"{n} points: {mine:.2e}, plain {plain:.2e}")
    assert mine <= 1.05 * plain


@pytest.mark.parametrize("sign", [-1, 1])
@pytest.mark.parametrize("n", [7, 91, 100, 121, 160, 700, 1014, 2000, 2002])
def test_mixed_line(lib, n, sign):
    rng = np.random.default_rng(n)
    x = _floats(rng.standard_normal(n) + 1j * rng.standard_normal(n))
    ref = x.astype(np.float64) @ [1, 1j]
    ref = np.fft.fft(ref) if sign < 0 else np.fft.ifft(ref) * n
    assert lib.mixed_march(n, 0, _ptr(x), None, 0, sign) == 0
    err = np.linalg.norm(x.astype(np.float64) @ [1, 1j] - ref) / np.linalg.norm(ref)
    # as above, a butterfly of radix r counted as the r sums of its definition
    r, k = 0, n
    for q in (13, 11, 7, 5, 3, 2):
        while k % q == 0:
            r, k = r + q, k // q
    assert err <= np.sqrt(3 * r) * 2.0 ** -24
