"""The automatic launch configuration is a configuration of its own: a reading
names what runs, every explicit pair (the default tile's too) stands as it was
set, what was read can be set, and a stored table brings back what it was
written from."""
import numpy as np
import pytest

from gpe_amd import ic, tuning
from gpe_amd.config import RunConfig
from test_bricks_gpu import KINDS

pytestmark = pytest.mark.gpu


def _cfg(n, **kw):
    nx, ny, nz = n
    base = dict(nx=nx, ny=ny, nz=nz, xr=0.2 * (nx - 1), yr=0.2 * (ny - 1), zr=0.2 * (nz - 1), tau=0.004, omx=0.3,
                omy=0.2, omz=0.4, order=4)
    base.update(kw)
    return RunConfig(**base)


def _default(precision, kind):
    """variant, waves, rows of the tile a new context names"""
    return (4, 8, 1) if precision == "fp64" and kind.startswith("ck") else (1, 8, 2)


def test_reading_names_what_runs(gpu):
    from gpe_amd.sim import Simulation
    print("[case] readings", flush=True)
    with Simulation(_cfg((48, 48, 48), scheme="rk45"), tuned=False) as sim:  # bricks of 2 planes
        got = sim.tune_get()
        assert all(got[k][1:] == (-2, 8, 1) for k in KINDS["rk45"])
    with Simulation(_cfg((193, 171, 157), scheme="rk45", order=2), tuned=False) as sim:  # 5.2 million sites
        got = sim.tune_get()
        assert got["ck_1"][1:] == (-4, 8, 1)                  # bricks of 4 planes
        assert got["ck_3"] == (3, -1, 4, 2) and got["ck_6"] == (4, -1, 8, 1)  # marches


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("scheme", ["euler", "rk2", "rk4", "rk45"])
def test_explicit_default_pair_stands(gpu, scheme, precision):
    from gpe_amd.sim import Simulation
    cfg = _cfg((70, 37, 29), scheme=scheme, precision=precision)
    psi = ic.vortex_ring(cfg, 2.0)
    print("[case] explicit default", scheme, precision, flush=True)
    with Simulation(cfg, psi, tuned=False) as sim:
        auto = sim.tune_get()
        for k in KINDS[scheme]:
            v, nw, rows = _default(precision, k)
            sim.tune_set(k, v, 0)
            assert sim.tune_get()[k] == (v, 0, nw, rows) != auto[k]
        sim.advance(2)
        a = sim.download(np.complex128)
    with Simulation(cfg, psi, tuned=False) as sim:
        for k in KINDS[scheme]:
            sim.tune_set(k, 3, 16)
        for k in KINDS[scheme]:
            sim.tune_set(k, *auto[k][:2])  # what was read: the automatic choice again
        assert sim.tune_get() == auto
        sim.advance(2)
        assert np.array_equal(sim.download(np.complex128), a)


def test_stored_table_brings_it_back(gpu, tmp_path):
    from gpe_amd.sim import Simulation
    path = str(tmp_path / "t.json")
    for scheme, precision in (("rk4", "fp64"), ("rk45", "fp32c")):
        cfg = _cfg((64, 40, 36), scheme=scheme, precision=precision)
        psi = ic.vortex_ring(cfg, 2.0)
        print("[case] stored table", scheme, precision, flush=True)
        with Simulation(cfg, psi, tuned=False) as sim:
            tuning.tune(sim, reps=1, path=path)
            want = {k: v[:2] for k, v in sim.tune_get().items()}
        with Simulation(cfg, psi, tuned=False) as sim:
            assert sim.tune_load(path)
            assert {k: v[:2] for k, v in sim.tune_get().items()} == want


def test_refused_pairs_stay_refused(gpu):
    from gpe_amd import _lib
    from gpe_amd.sim import Simulation
    print("[case] refused", flush=True)
    with Simulation(_cfg((24, 20, 18), scheme="rk45"), tuned=False) as sim:
        before = sim.tune_get()
        for pair in ((-1, 0), (5, 0), (4, -3), (4, -8), (1, -1)):
            with pytest.raises(_lib.GpeError):
                sim.tune_set("ck_6", *pair)
        assert sim.tune_get() == before


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("scheme", ["rk4", "rk45"])
def test_batch(gpu, scheme, precision):
    from gpe_amd.batch import Batch
    cfg = _cfg((48, 40, 36), scheme=scheme, precision=precision)
    psi = ic.vortex_ring(cfg, 2.0)
    kinds = KINDS[scheme]
    print("[case] batch readings", scheme, precision, flush=True)

    def run(setting):
        with Batch() as b:
            i = b.add(cfg, psi, 2)
            auto = [b.tune_get(precision, 4, scheme, k) for k in kinds]
            assert all(z < 0 for _, z in auto)
            for k, a in zip(kinds, auto):
                v = 4 if precision == "fp64" and scheme == "rk45" else 0
                if setting == "default":
                    b.tune_set(precision, 4, scheme, k, v, 32)
                    assert b.tune_get(precision, 4, scheme, k) == (v, 32)
                elif setting == "restored":
                    b.tune_set(precision, 4, scheme, k, 3, 16)
                    b.tune_set(precision, 4, scheme, k, *a)
                    assert b.tune_get(precision, 4, scheme, k) == a
            b.run_to_completion(chunk=2)
            return b.download(i)

    want = run("automatic")
    assert np.array_equal(run("default"), want) and np.array_equal(run("restored"), want)
