"""The FP64 functions of the step kernels (magpy_amd/csrc/normal64.h), built for
the host, against extended precision (x87 80-bit) at the edges of their ranges:
words next to 0 and 2^32 (u next to 0 and 1), powers of two and of sqrt(2)
(where the logarithm's exponent changes), every octant boundary of the angle,
phases next to multiples of a quarter cycle and of many cycles.

Bounds in ulp of the result, from the operations: the logarithm's quotient is
within an ulp and the sum with e ln 2 can cancel half of it (3 ulp); sqrt,
reciprocal and reciprocal square root end on a residual correction (1 ulp, and
1.5 where the correction is not the last rounding); sine and cosine are within
1.5 ulp of 1 and, reduced exactly, of themselves; the phase c cycles is exact,
so its sine is within 2 ulp of 1.  A Box-Muller normal is then within 5 ulp of
its radius.  The reciprocal seeds of the device (2^-23) are stood in for by
float arithmetic (2^-23).
"""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "magpy_amd", "csrc")
EPS = 2.0 ** -52
LD = np.longdouble
PI = LD("3.14159265358979323846264338327950288")
DRIVER = r'''
#include "normal64.h"
extern "C" {
void pairs(const uint32_t *a, const uint32_t *b, int n, double *l, double *c, double *s, double *z0,
           double *z1)
{
    for (int i = 0; i < n; ++i) {
        l[i] = mp::minus_two_log_u(a[i]);
        mp::sincos_u(b[i], c[i], s[i]);
        mp::box_muller64(a[i], b[i], z0[i], z1[i]);
    }
}
void sines(const double *x, int n, double *o) { for (int i = 0; i < n; ++i) o[i] = mp::sin_cycles(x[i]); }
void roots(const double *x, int n, double *q, double *r, double *v)
{
    for (int i = 0; i < n; ++i) {
        q[i] = mp::sqrt_normal(x[i]);
        r[i] = mp::rsqrt_normal(x[i]);
        v[i] = mp::rcp_normal(x[i]);
    }
}
}
'''


@pytest.fixture(scope="module")
def n64(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ is not available")
    if np.finfo(LD).nmant < 63:
        pytest.skip("no extended precision")
    d = tmp_path_factory.mktemp("normal64")
    (d / "n.cpp").write_text(DRIVER)
    subprocess.run([gxx, "-std=c++17", "-O2", "-mfma", "-ffp-contract=off", "-fPIC", "-shared",
                    "-I", CSRC, "-o", str(d / "n.so"), str(d / "n.cpp")], check=True)
    return C.CDLL(str(d / "n.so"))


def ptr(a):
    return a.ctypes.data_as(C.c_void_p)


def ulp(x):
    return np.spacing(np.abs(x.astype(np.float64))).astype(LD)


def edge_words(n, seed):
    near = lambda x: (np.asarray(x)[:, None] + np.arange(-2, 3)).ravel() % 2 ** 32  # noqa: E731
    edges = np.concatenate([near([0]), near(2 ** np.arange(32)), near(np.arange(8) * 2 ** 29),
                            near((2.0 ** (np.arange(32) + 0.5)).astype(np.int64))])
    rest = np.random.default_rng(seed).integers(0, 2 ** 32, size=n - edges.size)
    return np.concatenate([edges, rest]).astype(np.uint32)


def test_box_muller_pair(n64):
    n = 200000
    a = edge_words(n, 1)
    b = np.random.default_rng(2).permutation(edge_words(n, 3))
    l, c, s, z0, z1 = (np.empty(n) for _ in range(5))
    n64.pairs(ptr(a), ptr(b), n, ptr(l), ptr(c), ptr(s), ptr(z0), ptr(z1))
    u = (a.astype(LD) + LD(0.5)) / LD(2) ** 32
    ref_l = -2 * np.where(u > 0.9, np.log1p(u - 1), np.log(u))
    assert np.max(np.abs(l - ref_l) / ulp(ref_l)) < 3
    q = (b.astype(np.int64) + 2 ** 29) >> 30
    t = (b.astype(LD) + LD(0.5) - q.astype(LD) * 2 ** 30) / 2 ** 30 * (PI / 2)
    cs, sn = np.cos(t), np.sin(t)
    ref_c, ref_s = np.choose(q & 3, [cs, -sn, -cs, sn]), np.choose(q & 3, [sn, cs, -sn, -cs])
    for got, ref in ((c, ref_c), (s, ref_s)):
        assert np.max(np.abs(got - ref) / ulp(ref)) < 1.5
    r = np.sqrt(ref_l)
    for got, ref in ((z0, r * ref_c), (z1, r * ref_s)):
        assert np.max(np.abs(got - ref) / (EPS * r)) < 5


def test_sine_of_cycles(n64):
    rng = np.random.default_rng(4)
    quarters = np.arange(-40, 41) / 4.0
    x = np.concatenate([quarters, np.nextafter(quarters, 9e9), np.nextafter(quarters, -9e9),
                        rng.uniform(-6, 6, 100000), rng.uniform(0, 1e7, 100000), [0.0, -0.0]])
    o = np.empty(x.size)
    n64.sines(ptr(x), x.size, ptr(o))
    f = x.astype(LD)
    f = f - np.rint(f)
    assert np.max(np.abs(o - np.sin(2 * PI * f))) < 2 * EPS


def test_roots_and_reciprocals(n64):
    rng = np.random.default_rng(5)
    x = np.concatenate([2.0 ** np.arange(-60, 61), 10.0 ** rng.uniform(-18, 18, 100000)])
    q, r, v = (np.empty(x.size) for _ in range(3))
    n64.roots(ptr(x), x.size, ptr(q), ptr(r), ptr(v))
    xl = x.astype(LD)
    assert np.max(np.abs(q - np.sqrt(xl)) / ulp(np.sqrt(xl))) < 1
    assert np.max(np.abs(r - 1 / np.sqrt(xl)) / ulp(1 / np.sqrt(xl))) < 1.5
    assert np.max(np.abs(v - 1 / xl) / ulp(1 / xl)) < 1
