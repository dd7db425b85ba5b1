"""FP64 fields of very small and very large amplitude equal the oracle's in
every value.

The device forms abs() and the Laplacian's divisions by faster sequences in
an inner range of operands and by the general ones outside it, and measures
the rk45 error ratio only at sites that can hold its maximum: the field's
scale decides which of these run, so it is taken across their limits."""
import os

import numpy as np
import pytest

from gpe_amd import ic
from gpe_amd.config import RunConfig

pytestmark = pytest.mark.gpu
NT = min(16, os.cpu_count() or 1)


def _cfg(**kw):
    base = dict(nx=70, ny=21, nz=19, xr=7.0, yr=4.0, zr=3.6, eqn=4, g=1.0, mu=1.0, omx=0.3, omy=0.2, omz=0.4,
                tau=0.005, order=4, bcs=1)
    base.update(kw)
    return RunConfig(**base)


def _field(cfg, scale):
    rng = np.random.default_rng(5)
    psi = ic.vortex_ring(cfg, 2.0) * (1 + 0.05 * rng.standard_normal(cfg.shape)) * scale
    psi[:, :4, :] = 0.0  # and exact zeros beside it
    return psi


@pytest.mark.parametrize("scale", [1e-150, 1e-116, 1e-60, 1e-10, 1e10, 1e60])
@pytest.mark.parametrize("eqn", [4, 2])
def test_rhs(gpu, oracle, scale, eqn):
    from gpe_amd.sim import Simulation
    cfg = _cfg(eqn=eqn)
    psi = _field(cfg, scale)
    print("[case] rhs", scale, eqn, flush=True)
    with Simulation(cfg, psi) as sim:
        got = sim.rhs()
    assert np.array_equal(got, oracle.rhs(cfg, psi, NT))


@pytest.mark.parametrize("scale", [1e-60, 1e-10, 1.0])
@pytest.mark.parametrize("shape", [(70, 21, 19), (64, 64, 70)])
def test_rk45_steps(gpu, oracle, scale, shape):
    # chunks of 8 planes and whole columns: the largest ratio met so far is
    # kept per wave and per chunk
    from gpe_amd.sim import Simulation
    nx, ny, nz = shape
    cfg = _cfg(nx=nx, ny=ny, nz=nz, scheme="rk45", tau=0.02)
    psi = _field(cfg, scale)
    psi[:, :4, :] = 0.5 * scale  # (zeros beside a field shrink dt without end)
    print("[case] rk45", scale, shape, flush=True)
    st = oracle.make_state(cfg.dt)
    want, _ = oracle.run(cfg, st, psi, 3, NT)
    for zc in (8, nz):
        with Simulation(cfg, psi) as sim:
            sim.tune_set("ck_6", 4, zc)
            sim.advance(3)
            got, s = sim.download(), sim.state()
        assert np.array_equal(got, want)
        assert s["dt"].real == st.dt_re and s["errmax"] == st.errmax


@pytest.mark.parametrize("scale", [1e-200, 1.0, 1e235, 1e300])
def test_renormalise(gpu, scale):
    # (sqrt(nn) psi) / sqrt(norm) as the reference divides a complex by a real:
    # (a c) / c^2 * 2^-e with norm's root c 2^e
    from gpe_amd.sim import Simulation
    cfg = _cfg(nx=20, ny=12, nz=10)
    psi = _field(cfg, scale)
    print("[case] renormalise", scale, flush=True)
    for norm in (1.92 ** 2, 0.0625, 702.0):
        b = np.sqrt(norm)
        e = np.floor(np.log2(b))
        c = b * 2.0 ** -e
        with Simulation(cfg, psi) as sim:
            sim.renormalise(2.25, norm)
            got = sim.download()
        assert np.array_equal(got.view(np.float64), (1.5 * psi.view(np.float64) * c) / (c * c) * 2.0 ** -e)
