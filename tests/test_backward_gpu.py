"""Adaptive steps backwards in time.  With dt < 0 the rk45 error scale is
|psi| - |dt| |f| + 1e-30 (solve.f90:176-178 with its signed dt), which nearly
vanishes where |dt| |f| comes near |psi|: the error measure's maximum lies there,
and every storage form has to find it."""
import numpy as np
import pytest

from gpe_amd.config import RunConfig

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [None, (4, 32), (1, 16)], ids=str)
@pytest.mark.parametrize("order", [2, 4])
def test_compensated_error_measure_backwards(gpu, order, tile):
    from gpe_amd.sim import Simulation
    n, tau = 64, 0.02
    cfg = RunConfig(nx=n, ny=n, nz=n, xr=8.0, yr=8.0, zr=8.0, tau=tau, scheme="rk45", order=order, bcs=1, eqn=4,
                    precision="fp64", g=1.0, mu=1.0, eps=1.0)
    # |f| = | |psi|^2 - 1 | |psi| where psi varies slowly: at the top of the hump
    # |dt| |f| is some 0.96 |psi|, at its foot 0; the top lies inside a chunk of
    # planes, behind sites of larger |err| / |psi| than its own
    x = np.arange(n) / n - 0.6
    h = np.exp(4.0 * (np.cos(2 * np.pi * x) - 1.0))
    psi = 1.0 + (np.sqrt(1.0 + 0.95 / tau) - 1.0) * h[:, None, None] * h[None, :, None] * h[None, None, :]
    got = {}
    for precision in ("fp64", "fp32c"):
        print("[case] backward rk45", precision, order, tile, flush=True)
        with Simulation(cfg.with_(precision=precision), psi.astype(np.complex128)) as sim:
            if tile:
                sim.tune_set("ck_6", *((4, 32) if precision == "fp64" else tile))
            sim.set_state(dt=complex(-tau, 0.0))
            sim.advance(1)
            got[precision] = sim.state()
    # FP32 rounding: 1e-6 of f, against a scale of 0.035 |psi|; a site passed over
    # costs a factor of ten
    a, b = got["fp64"], got["fp32c"]
    assert a["n_rejects"] == 0 and a["t"] == -tau
    assert b["errmax"] == pytest.approx(a["errmax"], rel=0.01)
