"""The device's sine and cosine, compiled for the host: the float rounding of
the double-precision functions, without exception, for every azimuth a sampler
can draw (2 pi times a 23-bit fraction) and over the other arguments' ranges."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "barnacle_amd", "csrc")
SRC = """
#include "trig.hpp"
extern "C" void run(const float* x, float* s, float* c, long n) {
    for (long i = 0; i < n; ++i) bnd::sincos_f(x[i], s[i], c[i]);
}
"""


@pytest.fixture(scope="module")
def sincos(tmp_path_factory):
    d = tmp_path_factory.mktemp("trig")
    (d / "t.cpp").write_text(SRC)
    so = str(d / "t.so")
    subprocess.run(["g++", "-O2", "-mfma", "-ffp-contract=off", "-shared", "-fPIC", "-I", CSRC, str(d / "t.cpp"),
                    "-o", so], check=True)
    lib = ctypes.CDLL(so)

    def f(x):
        x = np.ascontiguousarray(x, np.float32)
        s, c = np.empty_like(x), np.empty_like(x)
        p = [a.ctypes.data_as(ctypes.c_void_p) for a in (x, s, c)]
        lib.run(*p, ctypes.c_long(x.size))
        return s, c

    return f


def azimuths():
    u = np.arange(1 << 23, dtype=np.uint32) | np.uint32(0x3F800000)
    return np.float32(2.0) * np.float32(np.pi) * (u.view(np.float32) - np.float32(1.0))


RANGES = {
    "azimuth": azimuths,
    "polar": lambda: np.linspace(0, 0x3FC90FDB, 1 << 22).astype(np.uint32).view(np.float32),     # 0 .. pi/2, all scales
    "lens": lambda: np.random.default_rng(3).uniform(-np.pi, np.pi, 1 << 20).astype(np.float32),
}


@pytest.mark.parametrize("name", list(RANGES))
def test_float_rounding_of_the_double_result(sincos, name):
    x = RANGES[name]()
    s, c = sincos(x)
    assert np.array_equal(s, np.sin(x.astype(np.float64)).astype(np.float32))
    assert np.array_equal(c, np.cos(x.astype(np.float64)).astype(np.float32))


def test_not_a_number(sincos):
    s, c = sincos(np.float32([np.nan, np.inf]))
    assert np.isnan(s).all() and np.isnan(c).all()
