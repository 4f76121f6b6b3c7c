"""The V steps' sine and cosine (atus2_amd/csrc/trig.hpp), compiled for the
host, against 64-bit-mantissa references over their whole range: both sides of
the switches at 2^-5 and 10^6, the doubles at and beside the multiples of
pi/2, infinities, NaN and the sign of zero."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = """
#include <cmath>
#define __device__
#define __forceinline__ inline
struct double2 { double x, y; };
static double2 make_double2(double x, double y) { return {x, y}; }
using std::fabs; using std::fma; using std::rint;
#include "trig.hpp"
extern "C" void run(const double* x, double* s, double* c, long n) {
  for (long i = 0; i < n; ++i) atus::sincos_mid(x[i], s + i, c + i);
}
"""


@pytest.fixture(scope="module")
def sincos_mid(tmp_path_factory):
    d = tmp_path_factory.mktemp("trig")
    (d / "t.cpp").write_text(SRC)
    so = str(d / "t.so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-shared", "-fPIC", "-Wno-attributes", "-I",
                    os.path.join(ROOT, "atus2_amd", "csrc"), str(d / "t.cpp"), "-o", so], check=True)
    f = C.CDLL(so).run
    dp = C.POINTER(C.c_double)

    def run(x):
        x = np.ascontiguousarray(x, np.float64)
        s, c = np.empty_like(x), np.empty_like(x)
        f(x.ctypes.data_as(dp), s.ctypes.data_as(dp), c.ctypes.data_as(dp), C.c_long(x.size))
        return s, c
    return run


def _ulps(got, ref):
    return np.abs(got - ref) / np.spacing(np.abs(ref.astype(np.float64)))


def _arguments():
    rng = np.random.default_rng(2)
    yield "random", rng.uniform(-1e6, 1e6, 500_000)
    yield "log", np.exp(rng.uniform(np.log(1e-9), np.log(1e6), 500_000)) * rng.choice([-1.0, 1.0], 500_000)
    k = np.arange(1, 636_620, dtype=np.longdouble)
    m = (k * (2 * np.arctan(np.longdouble(1)))).astype(np.float64)
    yield "multiples of pi/2", np.concatenate([m, np.nextafter(m, 0), np.nextafter(m, 1e9)])
    for edge in (0.03125, 1e6):
        e = np.array([edge, np.nextafter(edge, 0), np.nextafter(edge, 1e9)])
        yield f"beside {edge}", np.concatenate([e, -e])
    yield "beyond", rng.uniform(1e6, 1e15, 1000)


def test_under_one_ulp(sincos_mid):
    # half an ulp of the last addition, and the correction it adds: at most a
    # fifth of the result, of a few roundings
    for name, x in _arguments():
        s, c = sincos_mid(x)
        xl = x.astype(np.longdouble)
        es, ec = _ulps(s, np.sin(xl)).max(), _ulps(c, np.cos(xl)).max()
        assert es < 1 and ec < 1, (name, es, ec)


def test_special_values(sincos_mid):
    s, c = sincos_mid(np.array([0.0, -0.0, np.inf, -np.inf, np.nan]))
    assert s[0] == 0 and s[1] == 0 and not np.signbit(s[0]) and np.signbit(s[1])
    assert c[0] == 1 and c[1] == 1
    assert np.all(np.isnan(s[2:])) and np.all(np.isnan(c[2:]))
