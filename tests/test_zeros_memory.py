"""Memory of Simulation.zeros, without a GPU: the result holds its points and at
most 64 MiB more, and a grid whose dense list would not fit memory is counted
first."""
import ctypes

import numpy as np
import pytest

from gpe_amd import _lib
from gpe_amd.config import RunConfig
from gpe_amd.sim import Simulation


class _Points:
    """gpe_sim_zeros of a field with `count` points."""

    def __init__(self, count):
        self.count, self.caps = count, []

    def gpe_sim_zeros(self, ctx, which, out, cap, n):
        self.caps.append(cap)
        take = min(cap, self.count)
        if take:
            buf = (ctypes.c_char * (take * _lib.ZERO_DTYPE.itemsize)).from_address(ctypes.cast(out, ctypes.c_void_p).value)
            np.frombuffer(buf, _lib.ZERO_DTYPE)["cell"] = np.arange(take)
        n._obj.value = self.count
        return 0


def _sim(count, n=64):
    sim = Simulation.__new__(Simulation)
    sim._L, sim._ctx, sim.cfg = _Points(count), None, RunConfig(nx=n, ny=n, nz=n)
    sim.close = lambda: None
    return sim


@pytest.mark.parametrize("n", [64, 320, 512])
@pytest.mark.parametrize("count", [0, 1, 1000, 16384, 16385, 40000])
def test_result_holds_its_points(count, n):
    got = _sim(count, n).zeros()
    assert got.dtype == _lib.ZERO_DTYPE and np.array_equal(got["cell"], np.arange(count))
    held = got if got.base is None else got.base
    assert held.nbytes <= got.nbytes + (64 << 20)


def test_list_that_does_not_fit_is_counted_first(monkeypatch):
    empty = np.empty

    def limited(shape, *a, **k):
        if np.prod(shape) > 50000:
            raise MemoryError
        return empty(shape, *a, **k)

    sim = _sim(40000, n=1024)
    monkeypatch.setattr(np, "empty", limited)
    assert np.array_equal(sim.zeros()["cell"], np.arange(40000))
