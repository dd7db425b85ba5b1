"""The rk45 error measure where every ratio |err/scale| is below the single
range: fields so small that the scale's 1e-30 (solve.f90:176-178) is all of it.
The largest ratio has to be found whatever the tile and chunk, as the oracle
finds it, although the test that passes sites over keeps its bound in single
precision."""
import os

import numpy as np
import pytest

from gpe_amd.config import RunConfig

pytestmark = pytest.mark.gpu
NT = min(16, os.cpu_count() or 1)
UNIT = 2.0 ** -149  # the least single


@pytest.mark.parametrize("units", [2.9, 4.95, 9.95, 40.9, 1e3, 2.0 ** 22])
def test_ratios_below_the_single_range(gpu, oracle, units):
    from gpe_amd.sim import Simulation
    cfg = RunConfig(nx=70, ny=21, nz=48, xr=7.0, yr=2.1, zr=4.8, eqn=4, g=1.0, mu=1.0, tau=0.1, order=4, bcs=1,
                    scheme="rk45", precision="fp64")
    # the ratio rises along z by a few per cent, from below the largest one's
    # rounding to a single up to it
    hump = 1.0 + 0.05 * np.cos(2 * np.pi * (np.arange(cfg.nz) / cfg.nz - 0.9))
    psi = np.broadcast_to(hump[:, None, None], cfg.shape).astype(np.complex128)
    st = oracle.make_state(cfg.dt)
    oracle.run(cfg, st, psi * 1e-60, 1, NT)
    psi = psi * (1e-60 * units * UNIT / (st.errmax * cfg.eps))
    st = oracle.make_state(cfg.dt)
    oracle.run(cfg, st, psi, 1, NT)
    print("[case] error lead", units, st.errmax * cfg.eps / UNIT, flush=True)
    for tile in (None, (4, 8), (4, 48), (3, 16)):
        with Simulation(cfg, psi) as sim:
            if tile:
                sim.tune_set("ck_6", *tile)
            sim.advance(1)
            assert sim.state()["errmax"] == st.errmax, tile
