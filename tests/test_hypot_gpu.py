"""The device's hypot (csrc/refmath.h, hypot_ref with its fast inner range)
equals the host libm's in every bit.

Imprinting a vortex line of charge 0 replaces psi by abs(psi) * exp(0 i)
(variables.f90:1166-1180), so an FP64 field's real part comes back as the
device's abs of each value: millions of operand pairs over the whole double
range, and densely where the fast form begins and ends (the larger operand at
2^-383 and 2^511, the smaller at 2^-54 of it) or takes its other formula (the
result at twice the smaller operand)."""
import numpy as np
import pytest

from gpe_amd.config import RunConfig
from test_refmath import _call, shim  # noqa: F401  (the host libm's hypot)

pytestmark = pytest.mark.gpu
N = 128  # N^3 = 2 097 152 pairs a case


def _around(rng, n, centre, width=4.0):
    return centre * np.exp2(rng.uniform(-width, width, n))


def _steps(rng, n, value):
    """value and its nearest neighbours"""
    return (np.full(n, value).view(np.int64) + rng.integers(-3, 4, n)).view(np.float64)


def _cases(rng, n):
    sign = rng.choice([-1.0, 1.0], n)
    yield "normal", rng.standard_normal(n), rng.standard_normal(n)
    yield "wide", np.exp(rng.uniform(-700, 700, n)) * sign, np.exp(rng.uniform(-700, 700, n))
    a = np.exp(rng.uniform(-40, 40, n))
    yield "close", a, a * np.exp(rng.uniform(-40, 0, n)) * sign
    yield "tiny", np.exp(rng.uniform(-744, -600, n)), -np.exp(rng.uniform(-744, -600, n))
    yield "huge", np.exp(rng.uniform(300, 709, n)), np.exp(rng.uniform(300, 709, n))
    for name, limit in (("lower limit", 2.0 ** -383), ("upper limit", 2.0 ** 511)):
        a = np.where(rng.random(n) < 0.25, _steps(rng, n, limit), _around(rng, n, limit))
        yield name, a, a * np.exp2(rng.uniform(-56, 0, n)) * sign
        yield name + ", equal", a, (a.view(np.int64) + rng.integers(-4, 5, n)).view(np.float64)
        yield name + ", small", a, a * 2.0 ** -54 * (1.0 + 2.0 ** -50 * rng.integers(-8, 9, n))
    for k in (-300, 0, 300):
        a = np.exp2(rng.uniform(-2, 2, n) + k)
        yield "small at 2^%d" % k, a * 2.0 ** -54 * (1.0 + 2.0 ** -50 * rng.integers(-8, 9, n)), a
        # h = 2 ay where ax = sqrt(3) ay
        yield "formulas meet at 2^%d" % k, a, a * np.sqrt(3.0) * (1.0 + 2.0 ** -50 * rng.integers(-64, 65, n))
        # few bits: exact squares and short sums
        p, q = rng.integers(1, 1 << 20, n), rng.integers(1, 1 << 20, n)
        yield "integers at 2^%d" % k, p * 2.0 ** k, q * 2.0 ** k
    special = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 5e-324, 1.7976931348623157e308, 1.0, 2.0 ** -383,
                        2.0 ** 511])
    yield "special", rng.choice(special, n), rng.choice(special, n)


def test_device_hypot_equals_host_libm(gpu, shim):  # noqa: F811
    from gpe_amd.sim import Simulation
    cfg = RunConfig(nx=N, ny=N, nz=N, xr=6.0, yr=6.0, zr=6.0, precision="fp64", scheme="euler")
    line = dict(x0=0.1, y0=0.2, z0=0.3, amp1=0.0, amp2=0.0, ll=3.2, sgn=0.0, dir="z", imprint_phase=True)
    rng = np.random.default_rng(20261205)
    with Simulation(cfg) as sim:
        for name, x, y in _cases(rng, N ** 3):
            print("[case] device hypot", name, flush=True)
            psi = np.empty(N ** 3, np.complex128)
            psi.real, psi.imag = x, y
            sim.upload(psi.reshape(cfg.shape))
            sim.imprint_vortex_line(line)
            got = np.ascontiguousarray(sim.download(np.complex128).ravel().real)
            want = _call(shim.ref_hypot, x, y)[1]
            same = (got == want) | (np.isnan(got) & np.isnan(want))
            assert same.all(), (name, [(a.hex(), b.hex(), g.hex(), w.hex()) for a, b, g, w in
                                       zip(x[~same][:4], y[~same][:4], got[~same][:4], want[~same][:4])])
