"""A batch swept as its group's size decides (bricks of 2 or 4 planes, other
tiles and chunks) gives the fields of an explicit march bit for bit: ragged
grids at the edges of a brick, groups on both sides of every line of the
choice, each scheme, order and storage form.  The norm sums another tile's
partials (terms of one sign: 1e-13 of it)."""
import numpy as np
import pytest

from gpe_amd.config import RunConfig
from test_bricks_gpu import KINDS

pytestmark = pytest.mark.gpu

RAGGED = [(5, 5, 5), (64, 8, 6), (65, 9, 7), (63, 17, 31), (130, 24, 5)]
# million sites: below every line; above the FP64 ones of 5 M fields; above 8 and 10 M; above 16 M
GROUPS = {"ragged": RAGGED, "three": [(129, 96, 97)] + [(96, 95, 94)] * 2, "ten": [(131, 127, 128)] * 5,
          "seventeen": [(128, 130, 127)] * 8}


def _run(scheme, precision, order, shapes, march):
    from gpe_amd.batch import Batch
    with Batch() as b:
        if march:
            for k in KINDS[scheme]:
                b.tune_set(precision, order, scheme, k, 4, 24)
        ids = []
        for i, (nx, ny, nz) in enumerate(shapes):
            cfg = RunConfig(nx=nx, ny=ny, nz=nz, xr=0.2 * (nx - 1), yr=0.2 * (ny - 1), zr=0.2 * (nz - 1),
                            tau=0.0005 if scheme in ("euler", "rk2") else 0.004, precision=precision, scheme=scheme,
                            order=order, bcs=1 + i % 2, omx=0.3, omy=0.2, omz=0.4)
            ids.append(b.add_random_phase(cfg, 11 + i, 2, kmax=1.5))
        done = b.run_to_completion(chunk=2)
        assert all(done[i] == 1 for i in ids)
        keep = ids if len(set(shapes)) > 2 else [ids[0], ids[-1]]
        return [(b.download(i), b.query(i)) for i in keep]


@pytest.mark.parametrize("group", list(GROUPS))
@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("scheme", ["euler", "rk2", "rk4", "rk45"])
def test_automatic_equals_march(gpu, scheme, precision, group):
    for order in (2, 4):
        print("[case] batch sweeps", scheme, precision, order, group, flush=True)
        a, m = (_run(scheme, precision, order, GROUPS[group], march) for march in (False, True))
        for (fa, qa), (fm, qm) in zip(a, m):
            assert np.array_equal(fa, fm)
            assert qa["t"] == qm["t"] and qa["dt"] == qm["dt"]
            assert abs(qa["norm"] - qm["norm"]) <= 1e-13 * abs(qm["norm"])


def test_default_values_mean_the_automatic_choice(gpu):
    # a configuration read from a batch and set in another one is the same
    # configuration, whether a choice stands behind it or not
    from gpe_amd.batch import Batch
    with Batch() as b:
        for k, want in (("rk4_1", (0, 32)), ("rk4_4", (0, 32))):
            assert b.tune_get("fp64", 4, "rk4", k) == want
        assert b.tune_get("fp64", 4, "rk45", "ck_3") == (4, 32)
        b.tune_set("fp64", 4, "rk4", "rk4_2", 3, 16)
        assert b.tune_get("fp64", 4, "rk4", "rk4_2") == (3, 16)
