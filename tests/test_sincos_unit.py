"""The FP32 sine and cosine of the facet rotors (csrc/sincos_unit.h) on the CPU, compiled from the
source that the kernels include, against extended precision.

The bars are the errors of the device library's sincospif over the same distribution, measured on
an MI355X: 0.965 ulp, 1.504e-8 rms, and a mean amplitude 8.6e-11 from 1.  The mean amplitude is
what a summed visibility keeps: its standard error here is 1.5e-8 / sqrt(2 M) = 1e-11."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bullseye_amd",
                    "csrc")
SOURCE = """
#define __device__
#define __forceinline__ inline
#include "sincos_unit.h"
extern "C" void sincos_all(const float *x, float *s, float *c, long n) {
    for (long i = 0; i < n; ++i) bam::sincospi_unit(x[i], s + i, c + i);
}
"""


@pytest.fixture(scope="module")
def sincos(tmp_path_factory):
    d = tmp_path_factory.mktemp("sincos")
    (d / "s.cpp").write_text(SOURCE)
    so = str(d / "s.so")
    subprocess.run(["g++", "-O2", "-mfma", "-ffp-contract=off", "-shared", "-fPIC", "-I", CSRC,
                    str(d / "s.cpp"), "-o", so], check=True)
    lib = ctypes.CDLL(so)

    def call(x):
        s, c = np.empty_like(x), np.empty_like(x)
        ptr = ctypes.POINTER(ctypes.c_float)
        lib.sincos_all(x.ctypes.data_as(ptr), s.ctypes.data_as(ptr), c.ctypes.data_as(ptr),
                       ctypes.c_long(x.size))
        return s, c
    return call


def true_values(x):
    L = np.longdouble
    pi = 4 * np.arctan(L(1))
    n = np.rint(2 * x.astype(L))
    r = x.astype(L) - n / 2
    q = n.astype(int) % 4
    s, c = np.sin(pi * r), np.cos(pi * r)
    return np.choose(q, [s, c, -s, -c]), np.choose(q, [c, -s, -c, s])


def test_accuracy_and_mean_amplitude(sincos):
    x = np.random.default_rng(3).uniform(-1, 1, 2_000_000).astype(np.float32)
    s, c = sincos(x)
    ts, tc = true_values(x)
    for got, want in ((s, ts), (c, tc)):
        err = got - want
        far = np.abs(want) > 1e-6
        ulp = np.abs(np.spacing(want.astype(np.float32)))
        assert float((np.abs(err) / ulp)[far].max()) <= 0.965
        assert float(np.sqrt((err ** 2).mean())) <= 1.504e-8
    amplitude = float((s * ts + c * tc).mean() - 1)
    print("mean amplitude - 1: %.2e" % amplitude)
    assert abs(amplitude) <= 8.6e-11


def test_exact_points(sincos):
    x = np.array([0, 0.5, 1, -0.5, -1], np.float32)
    s, c = sincos(x)
    np.testing.assert_array_equal(s, np.array([0, 1, 0, -1, 0], np.float32))
    np.testing.assert_array_equal(c, np.array([1, 0, -1, 0, -1], np.float32))
    s, c = sincos(np.array([np.nan], np.float32))
    assert np.isnan(s[0]) and np.isnan(c[0])
