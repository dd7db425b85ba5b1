"""Field transfers where no page-locked memory is to be had: they go on as
plain copies, with the same values, in every storage form, host type and
layout.  A process of its own meets a hipHostMalloc that refuses everything
larger than the few words a context needs."""
import os
import subprocess
import sys

import pytest

from gpe_amd import _lib

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHIM = r"""
#include <dlfcn.h>
#include <stddef.h>
typedef int (*alloc_t)(void **, size_t, unsigned);
static long refused_;
long refused(void) { return refused_; }
int hipHostMalloc(void **p, size_t n, unsigned flags) {
  static alloc_t real;
  if (n > 4096) {
    ++refused_;
    return 2; /* hipErrorOutOfMemory */
  }
  if (!real) real = (alloc_t)dlsym(dlopen(HIPLIB, RTLD_NOW), "hipHostMalloc");
  return real(p, n, flags);
}
"""

CHILD = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # before the library that calls hipHostMalloc
sys.path[:0] = [sys.argv[2], sys.argv[2] + "/tests"]
import numpy as np
from gpe_amd import _lib
from gpe_amd.batch import Batch
from gpe_amd.sim import Simulation
from test_transfers_gpu import _cfg, _psi, _stored
shim.refused.restype = ctypes.c_long
last = 0
for shape in ((5, 5, 5), (65, 64, 33), (131, 129, 127)):
    for precision, up in (("fp64", np.complex128), ("fp32", np.complex64), ("fp32", np.complex128),
                          ("fp32c", np.complex64), ("fp32c", np.complex128)):
        print("[case] plain transfer", shape, precision, up.__name__, flush=True)
        cfg = _cfg(shape, precision)
        psi = _psi(cfg, up)
        hi, lo = _stored(psi, precision)
        with Simulation(cfg) as sim:
            for seed in (2, 1):
                sim.upload(_psi(cfg, up, seed))
            assert np.array_equal(sim.download(np.complex128).view(np.float64), hi + lo)
            if precision != "fp64":
                assert np.array_equal(sim.download(np.complex64).view(np.float32), (hi + lo).astype(np.float32))
            if shape == (65, 64, 33):
                assert len(sim.zeros()) > 0
                assert np.array_equal(sim.filtered(3.0).astype(np.complex64), sim.filtered(3.0, single=True))
        if precision != "fp32c":
            var_in = np.full((cfg.nz + 4, cfg.ny + 4, cfg.nx), np.nan, psi.dtype if precision == "fp64" else np.complex64)
            var_in[2:-2, 2:-2] = psi
            with Simulation(cfg, var_in[2:-2, 2:-2].copy()) as sim:
                sim.advance(1)
                want = sim.download(var_in.dtype)
            with Simulation(cfg) as sim:
                assert np.array_equal(sim.solver_step(var_in, halo=2), want)
        if precision != "fp32":
            with Batch() as b:
                i = b.add(cfg, psi, 1)
                b.run_to_completion(chunk=1)
                got = b.download(i)
            with Simulation(cfg, psi) as sim:
                sim.advance(1)
                assert np.array_equal(got, sim.download(np.complex128))
        assert shim.refused() > last
        last = shim.refused()
print("all plain", flush=True)
"""


def test_transfers_without_locked_memory(gpu, tmp_path):
    hip = [l.split("=>")[1].split("(")[0].strip() for l in subprocess.check_output(["ldd", _lib.LIB_PATH], text=True)
           .splitlines() if "libamdhip64" in l][0]
    (tmp_path / "shim.c").write_text(SHIM)
    so = str(tmp_path / "shim.so")
    subprocess.check_call(["gcc", "-O2", "-fPIC", "-shared", '-DHIPLIB="%s"' % hip, str(tmp_path / "shim.c"), "-o", so,
                           "-ldl"])
    r = subprocess.run([sys.executable, "-u", "-c", CHILD, so, ROOT], capture_output=True, text=True, timeout=100)
    print(r.stdout[-2000:], r.stderr[-3000:], flush=True)
    assert r.returncode == 0 and "all plain" in r.stdout
