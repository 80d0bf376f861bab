"""csrc/soft_math.h on the CPU (std::exp2 and a division in place of the GPU's
instructions) against tanh in 64 bits."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sana.cpp_amd", "csrc")
SRC = """
#include "soft_math.h"
extern "C" void run(const float * x, float * y, float * z, long n) {
    for (long i = 0; i < n; ++i) {
        y[i] = sana::soft_tanh(x[i]);
        z[i] = sana::soft_tanh_below_1(x[i]);
    }
}
"""


@pytest.fixture(scope="module")
def tanh(tmp_path_factory):
    d = tmp_path_factory.mktemp("soft_math")
    (d / "t.cpp").write_text(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, "-o", str(d / "t.so"),
                    str(d / "t.cpp")], check=True)
    lib = ctypes.CDLL(str(d / "t.so"))

    def f(x):
        x = np.ascontiguousarray(x, np.float32)
        y, z = np.empty_like(x), np.empty_like(x)
        p = [a.ctypes.data_as(ctypes.POINTER(ctypes.c_float)) for a in (x, y, z)]
        lib.run(*p, ctypes.c_long(x.size))
        return y, z
    return f


def test_tanh_ulp(tanh):
    """The result's rounding (1/2 ulp) and, below 1, that of x P and the polynomial
    (x^2 / 3 < 0.44 of the result: under 1/2 ulp together); above, e^2|x| and the
    reciprocal each within an ulp, times 2 / (c + 1) < 0.32 of the result."""
    x = np.concatenate([np.linspace(lo, hi, 400001) for lo, hi in
                        [(0, 1e-3), (1e-3, 0.25), (0.25, 1), (1, 1.5), (1.5, 10), (10, 40)]] +
                       [np.geomspace(1e-37, 1e38, 400001), np.nextafter(np.float32(1), np.float32([0, 2]))])
    x = x.astype(np.float32)
    y, z = tanh(x)
    ref = np.tanh(x.astype(np.float64))
    ulp = np.spacing(np.abs(ref).astype(np.float32)).astype(np.float64)
    assert (np.abs(y - ref) <= 1.2 * ulp).all()
    assert np.array_equal(y[x < 1], z[x < 1])
    assert np.array_equal(tanh(-x)[0], -y)


def test_tanh_special(tanh):
    y, z = tanh(np.float32([0.0, -0.0, np.inf, -np.inf, np.nan, 1e-45, -1e-40]))
    assert y[0] == 0 and y[1] == 0  # +0 either way
    assert y[2] == 1 and y[3] == -1 and np.isnan(y[4]) and np.isnan(z[4])
    assert y[5] == np.float32(1e-45) and y[6] == np.float32(-1e-40)
