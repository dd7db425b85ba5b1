"""The vortex passes' cell lists and the spectrum's shells at the sizes where
they can go wrong: cell counts on both sides of a workgroup's 4096 cells, one
cell, rows longer than a workgroup, lists without a cell, points beyond the
room given, and wave numbers beyond the last shell.  Per-cell arithmetic is
the oracle's, so points are compared bit for bit and lengths to 1e-12 (the
order of the sum)."""
import ctypes

import numpy as np
import pytest

from gpe_amd import _lib
from gpe_amd.config import RunConfig
from oracle import spectral as S

pytestmark = pytest.mark.gpu


def _cfg(n, precision):
    nx, ny, nz = n
    return RunConfig(nx=nx, ny=ny, nz=nz, xr=0.25 * (nx - 1), yr=0.25 * (ny - 1), zr=0.25 * (nz - 1), order=2, bcs=1,
                     precision=precision)


def _field(cfg, kind):
    rng = np.random.default_rng(5)
    z = rng.standard_normal(cfg.shape) + 1j * rng.standard_normal(cfg.shape)
    if kind == "sparse":  # a few sign changes in a field of one sign, exact zeros among them
        z = np.where(rng.random(cfg.shape) < 0.003, z, 2.0 + 1.5j)
        z[rng.random(cfg.shape) < 0.001] = 0.0
    elif kind == "none":
        z = 2.0 + np.abs(z.real) + 1j * (1.0 + np.abs(z.imag))
    return np.ascontiguousarray(z)


# (nx - 2)(ny - 2)(nz - 2) cells: 27; 4095, 4096 and 4100; 8192 in rows of 512
# (two turns of a workgroup); 4.5 M, more than 1024 workgroups' worth
LARGEST = (202, 162, 142)
SHAPES = [(5, 5, 5), (15, 37, 11), (18, 18, 18), (207, 7, 6), (514, 6, 6), LARGEST]


@pytest.mark.parametrize("precision", ["fp64", "fp32c", "fp32"])
@pytest.mark.parametrize("kind", ["dense", "sparse", "none"])
@pytest.mark.parametrize("n", SHAPES, ids=str)
def test_lists_match_the_oracle(oracle, n, kind, precision):
    from gpe_amd.sim import Simulation
    cfg = _cfg(n, precision)
    psi = _field(cfg, "sparse" if n == LARGEST and kind == "dense" else kind)
    print("[case] diagnostic lists", n, kind, precision, flush=True)
    with Simulation(cfg, psi.astype(np.complex64) if precision == "fp32" else psi) as sim:
        held = sim.download()
        length = sim.linelength()
        lists = [sim.zeros(w) for w in ("zeros", "re_zeros", "im_zeros")]
        # fewer places than points: the count is whole, the points are the first ones
        few = np.empty(3, _lib.ZERO_DTYPE)
        count = ctypes.c_int64()
        _lib.check(sim._L.gpe_sim_zeros(sim._ctx, 1, few.ctypes.data_as(ctypes.c_void_p), 3, ctypes.byref(count)))
    single = precision == "fp32"
    assert length == pytest.approx(oracle.linelength(cfg, held), rel=1e-5 if single else 1e-12, abs=0)
    for w, got in enumerate(lists):
        want = oracle.zeros(cfg, held, w)
        assert len(got) == len(want)
        for k in ("section", "cell", "x", "y", "z"):
            np.testing.assert_array_equal(got[k], want[k], err_msg=f"{w} {k}")
    assert count.value == len(lists[1])
    for k in ("section", "cell", "x"):
        np.testing.assert_array_equal(few[k][:min(3, count.value)], lists[1][k][:3])


@pytest.mark.parametrize("n", [(6, 6, 1700), (8, 820, 8), (64, 12, 10)], ids=str)
def test_shells_and_zero_mode(n):
    # 1e-12 of sums of positive terms; the zero mode is compared by its size,
    # and the oracle's transform rounds it by some 1e-16 of sum |psi| / sqrt(V)
    from gpe_amd.sim import Simulation
    cfg = _cfg(n, "fp64")
    psi = _field(cfg, "dense")
    print("[case] shells", n, flush=True)
    with Simulation(cfg, psi) as sim:
        nh, eta, idf = sim.spectrum()
        rec = sim.condensed_particles()
    wn, we, wf = S.spectrum(S.forward(psi))
    assert list(nh) == list(wn)
    np.testing.assert_allclose(eta, we, rtol=1e-12)
    np.testing.assert_allclose(idf, wf, rtol=1e-12)
    V = psi.size
    zero = abs(psi.sum()) / np.sqrt(V)
    assert abs(np.sqrt(rec["n0"]) - zero) <= 1e-14 * np.abs(psi).sum() / np.sqrt(V)
