"""The kernels' double arithmetic (csrc/gqa_math.h) built for the host.

RoPE's sines and cosines against numpy's long double (64-bit mantissa) at the rounded angle, the
one the golden rotates at (pyfiles/gen_gqa_wrapper_vectors.py:30); the prefill epilogue's quotient
against division.

Bounds: the library's double sincos of the angle reduced modulo 2 pi, which these replace, has a
largest error of 2.45e-16 against 113-bit values, over all angles below 2^53; sincos_f64 and a
cached key's turned rotation may have no more."""
from __future__ import annotations

import ctypes
import subprocess

import numpy as np
import pytest

from conftest import ROOT

LIBRARY_ERROR = 2.45e-16

_SRC = r"""
#define __host__
#define __device__
#define __forceinline__ inline
#include "gqa_math.h"
extern "C" void sincos_all(const double* a, int n, double* s, double* c) {
    for (int i = 0; i < n; ++i) gqa::sincos_f64(a[i], s[i], c[i]);
}
extern "C" void turned(const double* kc, const double* d, const double* f, int n, double* s, double* c) {
    for (int i = 0; i < n; ++i) {
        double bc, bs, dc, ds;
        gqa::rot_exact(kc[i], f[i], bc, bs);
        gqa::rot_exact(d[i], f[i], dc, ds);
        gqa::rot_turn(bc, bs, dc, ds, kc[i] + d[i], f[i], c[i], s[i]);
    }
}
extern "C" void quotients(const double* a, const double* b, int n, double* q) {
    for (int i = 0; i < n; ++i) q[i] = gqa::quotient(a[i], b[i], 1.0 / b[i]);
}
extern "C" double max_angle() { return gqa::kKRopeMaxAngle; }
"""


@pytest.fixture(scope="module")
def math(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("host_math")
    (tmp / "m.cpp").write_text(_SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-ffp-contract=off",
                    f"-I{ROOT / 'attention_accelerator_amd/csrc'}", "-o", str(tmp / "m.so"), str(tmp / "m.cpp")],
                   check=True)
    lib = ctypes.CDLL(str(tmp / "m.so"))
    lib.max_angle.restype = ctypes.c_double
    return lib


def _ptr(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))


def _error(angle, s, c):
    a = angle.astype(np.longdouble)
    return float(max(np.abs(np.sin(a) - s).max(), np.abs(np.cos(a) - c).max()))


@pytest.mark.parametrize("lo,hi", [(-30, 1), (1, 20), (20, 45), (45, 50), (50, 53)])
def test_sincos_error(math, lo, hi):
    rng = np.random.default_rng(lo + 100)
    n = 100_000
    a = np.ldexp(1.0 + rng.random(n), rng.integers(lo, hi, n)) * rng.choice([-1.0, 1.0], n)
    a[:64] = np.pi / 4 * np.arange(64) if hi <= 20 else a[:64]       # the ends of the reduced range
    s, c = np.empty(n), np.empty(n)
    math.sincos_all(_ptr(a), n, _ptr(s), _ptr(c))
    assert _error(a, s, c) <= LIBRARY_ERROR


def test_sincos_stays_bounded(math):
    """Angles with no meaningful reduction left still give a point near the unit circle."""
    a = np.array([2.0 ** e for e in range(54, 1024)])
    s, c = np.empty(a.size), np.empty(a.size)
    math.sincos_all(_ptr(a), a.size, _ptr(s), _ptr(c))
    assert (np.abs(s * s + c * c - 1.0) < 1e-12).all()


@pytest.mark.parametrize("theta,top", [
    (500000.0, 4096), (500000.0, 131072), (500000.0, 400000), (10000.0, 32768),
    (1.0, 2 ** 26), (1e-3, 2 ** 16),          # angles up to the shared rotations' bound
])
def test_turned_rotation_error(math, theta, top):
    rng = np.random.default_rng(top)
    n = 400_000
    f = np.array([theta ** (-2.0 * i / 128) for i in range(64)])[rng.integers(0, 64, n)]
    d = rng.integers(0, 16, n).astype(np.float64)
    kc = np.floor(rng.random(n) * (top - 16))
    assert ((kc + d) * f).max() <= math.max_angle()
    s, c = np.empty(n), np.empty(n)
    math.turned(_ptr(kc), _ptr(d), _ptr(f), n, _ptr(s), _ptr(c))
    assert _error((kc + d) * f, s, c) <= LIBRARY_ERROR


def test_quotient_is_division(math):
    """Bit for bit over O's and l's ranges (the product with 1 / l differs in about one of four)."""
    rng = np.random.default_rng(9)
    n = 1_000_000
    b = np.ldexp(1.0 + rng.random(n), rng.integers(8, 44, n))
    a = np.ldexp(1.0 + rng.random(n), rng.integers(-200, 180, n)) * rng.choice([-1.0, 1.0], n)
    a[:100] = 0.0
    q = np.empty(n)
    math.quotients(_ptr(a), _ptr(b), n, _ptr(q))
    assert (a * (1.0 / b) != a / b).mean() > 0.2
    assert np.array_equal(q, a / b)
