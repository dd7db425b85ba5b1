"""Division of an FP64 value by a constant (gpe_amd/csrc/divc.h), built for
the host: the device evaluates the same IEEE operations.  Every quotient has
to equal the reference's logb-scaled division in every bit: on ordinary
numerators, on tiny ones and on the numerators whose quotient lies next to
the middle of two doubles, where a quotient formed without a division can
round the wrong way.  (A zero stays a zero; its sign may not.)"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SHIM = r"""
#include "divc.h"
extern "C" void divc(double s, const double *a, long n, double *got, double *want) {
  const gpe::DivC d = gpe::make_divc(s);
  const int e = std::ilogb(s);
  const double c = std::ldexp(s, -e), den = c * c + 0.0 * 0.0;
  for (long i = 0; i < n; ++i) {
    got[i] = gpe::div_const(a[i] * d.cs, d);
    want[i] = std::ldexp((a[i] * c) / den, -e);
  }
}
// numerators whose quotients lie next to the midpoints after the q
extern "C" long near_mid(double s, const double *q, long n, double *a) {
  const int e = std::ilogb(s);
  const double c = std::ldexp(s, -e);
  for (long i = 0; i < n; ++i) {
    const long double m = (long double)q[i] + (long double)(std::nextafter(q[i], 4.0) - q[i]) / 2;
    a[i] = (double)(m * c);  // t = a*c, quotient a*c/(c*c)
  }
  return n;
}
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    d = tmp_path_factory.mktemp("divc")
    (d / "shim.cpp").write_text(SHIM)
    so = str(d / "shim.so")
    subprocess.check_call(["g++", "-O2", "-ffp-contract=off", "-fPIC", "-shared",
                           "-I" + os.path.join(ROOT, "gpe_amd", "csrc"), str(d / "shim.cpp"), "-o", so])
    L = ctypes.CDLL(so)
    vp = ctypes.c_void_p
    L.divc.argtypes = [ctypes.c_double, vp, ctypes.c_long, vp, vp]
    L.near_mid.argtypes = [ctypes.c_double, vp, ctypes.c_long, vp]
    return L


def _p(v):
    return v.ctypes.data_as(ctypes.c_void_p)


def test_quotients_equal_the_division(shim):
    rng = np.random.default_rng(11)
    # the package's divisors (12 dx^2, dx^2, 12 dx, 6, 3) and random ones, some with few bits
    div = [12 * 0.4 ** 2, 0.4 ** 2, 12 * 0.25 ** 2, 12 * 0.5 ** 2, 0.25, 1.0, 6.0, 3.0, 12 * 0.1, 1 - 2.0 ** -53,
           2 - 2.0 ** -52, 1 + 2.0 ** -52, 1e-30, 1e30]
    div += list(np.exp(rng.uniform(-8, 8, 120)))
    div += [float(np.round(v * 2 ** 8) / 2 ** 8) for v in rng.uniform(1, 4, 30)]
    n = 20000
    zeros = np.array([0.0, -0.0])
    for s in div:
        q = rng.uniform(1, 2, n)
        near = np.empty(n)
        shim.near_mid(s, _p(q), n, _p(near))
        a = np.concatenate([rng.standard_normal(n), near, -near * 2.0 ** rng.integers(-200, 200, n),
                            rng.standard_normal(n) * 2.0 ** rng.integers(-900, 250, n), zeros])
        got, want = np.empty_like(a), np.empty_like(a)
        shim.divc(s, _p(a), len(a), _p(got), _p(want))
        same = got == want
        assert same.all(), (s, a[~same][:3], got[~same][:3], want[~same][:3])


def test_undefined_divisors_give_nan(shim):
    a = np.array([1.0, -2.0, 0.0])
    got, want = np.empty(3), np.empty(3)
    for s in (0.0, float("inf"), float("nan")):
        shim.divc(s, _p(a), 3, _p(got), _p(want))
        assert np.isnan(got).all()


def test_numerators_to_the_end_of_the_range(shim):
    # quotients of the largest numerators whose a*c does not overflow; by the
    # package's own divisors also where it does, and of infinities
    rng = np.random.default_rng(12)
    own = [1.92, 12 * 0.4 ** 2, 0.4 ** 2, 12 * 0.25 ** 2, 12 * 0.5 ** 2, 0.25, 0.5, 1.0, 2.0, 4.0, 6.0, 3.0, 12 * 0.1]
    with np.errstate(over="ignore"):
        for s in own + [0.01, 1e-30, 1e30] + list(np.exp(rng.uniform(-8, 8, 200))):
            a = np.concatenate([rng.standard_normal(4000) * 2.0 ** rng.integers(240, 1022, 4000),
                                rng.uniform(-1, 1, 2000) * (1.79e308 if s in own else 0.89e308), [1e232],
                                [1.7976931348623157e308, np.inf, -np.inf] if s in own else []])
            got, want = np.empty_like(a), np.empty_like(a)
            shim.divc(s, _p(a), len(a), _p(got), _p(want))
            same = got == want
            assert same.all(), (s, a[~same][:3], got[~same][:3], want[~same][:3])
