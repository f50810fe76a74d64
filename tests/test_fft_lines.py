"""The power-of-two butterflies and their twiddle seeds (swem_fft.hpp), compiled for the host and run line by
line: against the 64-bit transform, and the error that many of them leave in a march.

A march repeats one transform with the same table entries at every depth, so the rounding of the entries
(half a unit in the last place of each part) adds up over the depths while the rounding of the sums does
not.  A line of 256 points takes four radix-4 levels, hence at most one entry per level and input; its march
may be no further from 64 bits than one of plain products and sums with those same entries.  What differs
between the two is the rounding of the sums, which is a few per cent of the error of 200 depths: bound 1.05.
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


@pytest.mark.parametrize("p", [4, 8, 16])
def test_march_error_of_256_points(lib, p):
    n, steps = 256, 200
    mine, plain = 0.0, 0.0
    for s in range(12):
        k = np.minimum(np.arange(n), n - np.arange(n))
        a = 1.0 - (k / ((0.2 + 0.02 * s) * n)) ** 2
        phase = np.where(a > 0, np.exp(1j * (3 + 0.5 * s) * np.sqrt(np.abs(a))), np.exp(-1.2 * np.sqrt(np.abs(a)))) / n
        z = np.zeros(n, complex)
        z[n // 8 + s * n // 40] = 1 + 0.3j
        ph, x = _floats(phase), [_floats(z), _floats(z)]
        z = x[0].astype(np.float64) @ [1, 1j]
        for _ in range(steps):
            z = np.fft.ifft(np.fft.fft(z) * phase) * n
            z[n // 2:] = 0
        assert lib.fft_march_256(p, _ptr(x[0]), _ptr(ph), steps) == 0
        assert lib.fft_march_256(0, _ptr(x[1]), _ptr(ph), steps) == 0
        e = [np.linalg.norm(v.astype(np.float64) @ [1, 1j] - z) / np.linalg.norm(z) for v in x]
        mine, plain = mine + e[0] / 12, plain + e[1] / 12
    print(f"{p} points per thread: {mine:.2e}, plain {plain:.2e}")
    assert mine <= 1.05 * plain
