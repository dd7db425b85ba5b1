"""Field transfers between host arrays and device storage (csrc/transfer.hip):
every pair of storage form and host type, at sizes around the 8 MiB staging
buffer, arrays with ghost layers, and several threads at once.  Expected
values are formed with numpy."""
import threading

import numpy as np
import pytest

from gpe_amd.config import RunConfig

pytestmark = pytest.mark.gpu

# sites: below, at and past one and four buffers of complex128, and ragged
SHAPES = [(5, 5, 5), (64, 64, 128), (65, 64, 128), (128, 128, 128), (131, 129, 127)]


def _cfg(shape, precision, **kw):
    nx, ny, nz = shape
    return RunConfig(nx=nx, ny=ny, nz=nz, xr=0.2 * nx, yr=0.2 * ny, zr=0.2 * nz, precision=precision, scheme="euler",
                     tau=1e-3, **kw)


def _psi(cfg, dtype, seed=1):
    rng = np.random.default_rng(seed)
    p = rng.standard_normal(cfg.shape) + 1j * rng.standard_normal(cfg.shape)
    p[0, 0, :3] = 0, -0.0, 1e-300
    return p.astype(dtype)


def _stored(psi, precision):
    """hi and lo words of the storage form, as float64 pairs"""
    v = psi.astype(np.complex128).view(np.float64)
    if precision == "fp64":
        return v, np.zeros_like(v)
    hi = v.astype(np.float32).astype(np.float64)
    lo = (v - hi).astype(np.float32).astype(np.float64) if precision == "fp32c" else np.zeros_like(v)
    return hi, lo


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("precision,up", [("fp64", np.complex128), ("fp32", np.complex64), ("fp32", np.complex128),
                                          ("fp32c", np.complex64), ("fp32c", np.complex128)])
def test_round_trip(gpu, shape, precision, up):
    from gpe_amd.sim import Simulation
    cfg = _cfg(shape, precision)
    psi = _psi(cfg, up)
    hi, lo = _stored(psi, precision)
    print("[case] transfer", shape, precision, up.__name__, flush=True)
    with Simulation(cfg) as sim:
        for seed in (2, 1):  # buffers used before hold another field
            sim.upload(_psi(cfg, up, seed))
        got = sim.download(np.complex128)
        assert np.array_equal(got.view(np.float64), hi + lo)
        if precision != "fp64":
            assert np.array_equal(sim.download(np.complex64).view(np.float32), (hi + lo).astype(np.float32))


@pytest.mark.parametrize("shape", [(5, 6, 7), (67, 65, 130)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("halo", [0, 2, 3])
def test_ghost_layers(gpu, shape, precision, halo):
    from gpe_amd.sim import Simulation
    cfg = _cfg(shape, precision)
    psi = _psi(cfg, np.complex128 if precision == "fp64" else np.complex64)
    var_in = np.full((cfg.nz + 2 * halo, cfg.ny + 2 * halo, cfg.nx), np.nan, psi.dtype)
    var_in[halo:halo + cfg.nz, halo:halo + cfg.ny] = psi
    print("[case] ghost layers", shape, precision, halo, flush=True)
    with Simulation(cfg, psi) as sim:
        sim.advance(1)
        want = sim.download(psi.dtype)
    with Simulation(cfg) as sim:
        got = sim.solver_step(var_in, halo=halo)
    assert np.array_equal(got, want)


def test_threads(gpu):
    from gpe_amd.sim import Simulation
    bad = []

    def work(seed):
        cfg = _cfg((97, 101 + seed, 60), ("fp64", "fp32c", "fp32")[seed % 3])
        psi = _psi(cfg, np.complex64 if cfg.precision == "fp32" else np.complex128, seed)
        hi, lo = _stored(psi, cfg.precision)
        for _ in range(4):
            with Simulation(cfg, psi) as sim:
                if not np.array_equal(sim.download(np.complex128).view(np.float64), hi + lo):
                    bad.append(seed)

    print("[case] six threads", flush=True)
    th = [threading.Thread(target=work, args=(s,)) for s in range(6)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
