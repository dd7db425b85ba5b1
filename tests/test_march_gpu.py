"""The automatic march (tile variant and z-chunk by kind, order, size and how
many workgroups a CU holds) gives the fields of one explicit tile bit for bit,
on both sides of every line of the choice, on grids with partly filled tiles and
on one a single tile wide.  The norm sums another tile's partials (terms of one
sign: 1e-13 of it)."""
import numpy as np
import pytest

from gpe_amd.config import RunConfig
from test_bricks_gpu import KINDS

pytestmark = pytest.mark.gpu

# million sites: 2.45, 3.5, 5.9 (rows of whole tiles), 6.5, 16.8, 21, 52 (FP32 kinds of one field)
SHAPES = [(193, 131, 97), (33, 520, 203), (192, 175, 176), (201, 190, 170), (256, 256, 256), (290, 280, 260)]


def _run(cfg, march):
    from gpe_amd.sim import Simulation
    with Simulation(cfg, tuned=False) as sim:
        if march:
            for k in KINDS[cfg.scheme] + ["rhs"]:
                sim.tune_set(k, 4, 24)
        sim.random_phase(7, 1.5)
        f = sim.rhs()
        sim.advance(2)
        return f, sim.download(), sim.state(), sim.norm()


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("precision", ["fp64", "fp32", "fp32c"])
@pytest.mark.parametrize("scheme", ["euler", "rk2", "rk4", "rk45"])
def test_automatic_equals_one_tile(gpu, shape, precision, scheme):
    nx, ny, nz = shape
    for order, bcs in ((2, 2), (4, 1)):
        cfg = RunConfig(nx=nx, ny=ny, nz=nz, xr=0.2 * (nx - 1), yr=0.2 * (ny - 1), zr=0.2 * (nz - 1), omx=0.3, omy=0.2,
                        omz=0.4, tau=0.0005 if scheme in ("euler", "rk2") else 0.004, precision=precision,
                        scheme=scheme, order=order, bcs=bcs)
        print("[case] march", shape, precision, scheme, order, bcs, flush=True)
        a, m = _run(cfg, False), _run(cfg, True)
        assert np.array_equal(a[0], m[0]) and np.array_equal(a[1], m[1])
        assert a[2] == m[2]
        assert abs(a[3] - m[3]) <= 1e-13 * abs(m[3])


def test_largest_single_precision_kinds(gpu):
    cfg = RunConfig(nx=400, ny=381, nz=341, xr=80.0, yr=76.0, zr=68.0, tau=0.004, precision="fp32", scheme="rk4",
                    order=4, bcs=1)
    print("[case] march largest fp32", flush=True)
    a, m = _run(cfg, False), _run(cfg, True)
    assert np.array_equal(a[0], m[0]) and np.array_equal(a[1], m[1])
