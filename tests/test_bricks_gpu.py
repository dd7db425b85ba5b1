"""Brick sweeps (csrc/brick.hpp) give the z march's fields bit for bit: at the
edges of a brick (64 x 8 x 2 and 4 sites), on grids smaller than one, in every
scheme, storage form, order and boundary condition, and where the automatic
choice changes from one to the other.  The norm history of a long call equals
the norms of single steps."""
import numpy as np
import pytest

from gpe_amd import ic
from gpe_amd.config import RunConfig

pytestmark = pytest.mark.gpu

KINDS = {"euler": ["euler"], "rk2": ["rk2_1", "rk2_2"], "rk4": ["rk4_%d" % i for i in range(1, 5)],
         "rk45": ["ck_%d" % i for i in range(1, 7)]}


def _cfg(shape, **kw):
    nx, ny, nz = shape
    base = dict(nx=nx, ny=ny, nz=nz, xr=0.2 * (nx - 1), yr=0.2 * (ny - 1), zr=0.2 * (nz - 1), tau=0.004, omx=0.3,
                omy=0.2, omz=0.4)
    base.update(kw)
    return RunConfig(**base)


def _field(cfg):
    rng = np.random.default_rng(9)
    psi = ic.vortex_ring(cfg, 0.4 * cfg.xr) * (1 + 0.05 * rng.standard_normal(cfg.shape))
    return psi.astype(np.complex64) if cfg.precision == "fp32" else psi


def _run(cfg, psi, steps, march):
    from gpe_amd.sim import Simulation
    with Simulation(cfg, psi, tuned=False) as sim:
        if march:
            for k in KINDS[cfg.scheme] + ["rhs", "energy"]:
                sim.tune_set(k, 4, 8)
        f = sim.rhs()
        h = sim.advance(steps, record_norm=True)
        return f, sim.download(), h, sim.energy(), sim.state()


@pytest.mark.parametrize("shape", [(5, 5, 5), (64, 8, 6), (65, 9, 7), (63, 17, 31), (130, 24, 5)])
@pytest.mark.parametrize("precision", ["fp64", "fp32", "fp32c"])
@pytest.mark.parametrize("scheme", ["euler", "rk2", "rk4", "rk45"])
def test_bricks_equal_march(gpu, shape, precision, scheme):
    for order, bcs, eqn in ((2, 1, 4), (2, 2, 1), (4, 1, 2), (4, 2, 4)):
        cfg = _cfg(shape, precision=precision, scheme=scheme, order=order, bcs=bcs, eqn=eqn,
                   urhs=0.0 if eqn == 4 else 0.2)
        psi = _field(cfg)
        print("[case] bricks", shape, precision, scheme, order, bcs, eqn, flush=True)
        a, b = _run(cfg, psi, 3, False), _run(cfg, psi, 3, True)
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
        # sums: partials of other tiles, in another order (a few hundred terms of one sign)
        assert np.allclose(a[2], b[2], rtol=1e-13, atol=0)
        assert abs(a[3] - b[3]) <= 1e-12 * abs(b[3]) if precision == "fp64" else True
        assert a[4]["t"] == b[4]["t"] and a[4]["dt"] == b[4]["dt"] and a[4]["errmax"] == b[4]["errmax"]


@pytest.mark.parametrize("shape", [(170, 171, 172), (193, 171, 157)])  # 5.00 and 5.18 million sites
def test_four_plane_bricks_equal_march(gpu, shape):
    for scheme, order in (("euler", 2), ("rk2", 4), ("rk4", 4), ("rk45", 2)):
        cfg = _cfg(shape, scheme=scheme, order=order, bcs=2 if order == 4 else 1)
        rng = np.random.default_rng(3)
        psi = rng.standard_normal(cfg.shape) + 1j * rng.standard_normal(cfg.shape)
        print("[case] four planes", shape, scheme, order, flush=True)
        a, b = _run(cfg, psi, 1, False), _run(cfg, psi, 1, True)
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


@pytest.mark.parametrize("scheme", ["rk4", "rk2", "rk45"])
def test_norm_history_equals_single_steps(gpu, scheme):
    from gpe_amd.sim import Simulation
    cfg = _cfg((40, 20, 18), scheme=scheme)
    psi = _field(cfg)
    print("[case] norm history", scheme, flush=True)
    with Simulation(cfg, psi) as sim:
        together = np.concatenate([sim.advance(n, record_norm=True) for n in (1, 70, 130)])
    with Simulation(cfg, psi) as sim:
        single = np.concatenate([sim.advance(1, record_norm=True) for _ in range(201)])
        last = sim.norm()
    assert np.array_equal(together, single)
    assert abs(single[-1] - last) <= 1e-13 * last


@pytest.mark.parametrize("shape", [(5, 5, 5), (64, 8, 6), (65, 9, 7), (63, 17, 31), (130, 24, 5)])
@pytest.mark.parametrize("precision", ["fp64", "fp32", "fp32c"])
def test_brick_energy_equals_march(gpu, shape, precision):
    # every site's term has the same bits either way and they are summed in
    # double: the sums differ by at most (terms) 2^-53 of the sum of |term|
    from gpe_amd.sim import Simulation
    cfg = _cfg(shape, precision=precision, scheme="euler", order=2, bcs=1)
    psi = _field(cfg)
    print("[case] brick energy", shape, precision, flush=True)
    got = []
    for tile in (None, (4, 8), (0, 8)):
        with Simulation(cfg, psi, tuned=False) as sim:
            if tile:
                sim.tune_set("energy", *tile)
            got.append(sim.energy())
    lap = sum((np.roll(psi, 1, a) - 2 * psi + np.roll(psi, -1, a)) / d ** 2
              for a, d in ((0, cfg.dz), (1, cfg.dy), (2, cfg.dx)))
    m = np.abs(psi)
    terms = 1.01 * np.sum(np.abs(lap).astype(np.float64) * m + 0.5 * m.astype(np.float64) ** 4) * cfg.dx * cfg.dy * cfg.dz
    for g in got[1:]:
        assert abs(g - got[0]) <= psi.size * 2.0 ** -53 * terms
