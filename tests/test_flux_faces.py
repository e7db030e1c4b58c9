"""The faces per thread that a stage's flux launch takes by the size of the grid (1, 2 or
4) against a launch per direction with 2: state, fluxes, flags and counters bit for
bit, on both sides of each line and with partial groups."""
import numpy as np
import pytest

from coolharm3d_amd import Harm3D, bbh_disk, bbh_grid, torus, torus_grid
from coolharm3d_amd.pn import PnMetric
from coolharm3d_amd.problems import bbh_gdet

pytestmark = pytest.mark.gpu

CASES = [
    dict(n=(24, 30, 26)), dict(n=(26, 30, 28)),                       # about 65536 faces: one or two per thread
    dict(n=(24, 30, 26), precision="mixed"), dict(n=(26, 30, 28), precision="mixed"),
    dict(n=(67, 71, 68), precision="mixed"), dict(n=(73, 70, 69), precision="mixed"),   # about 2^20: two or four
    dict(disk=True, n=(73, 70, 71), precision="mixed"), dict(disk=True, n=(15, 17, 19), precision="mixed"),
]


@pytest.mark.parametrize("case", CASES, ids=str)
def test_faces_per_thread(case):
    kw = dict(case)
    n, disk = kw.pop("n"), kw.pop("disk", False)
    grid = bbh_grid(*n) if disk else torus_grid(*n)
    p = bbh_disk(grid, bbh_gdet(grid, PnMetric)) if disk else torus(grid)
    runs = []
    for per_direction in (False, True):
        H = Harm3D(grid, **kw)
        if per_direction:
            for f in ("flux1", "flux2", "flux3"):
                bs, kc, flags = H.launch_shape(f)
                H.set_launch_shape(f, bs, kc, flags & ~128)
                assert (H.launch_shape(f)[2] >> 4) & 3 == 1
        H.set_prims(p)
        H.fixup_bounds()
        H.set_time(0.0, grid.dx[0])
        H.step_ch(2)
        runs.append(H)
    A, B = runs
    assert np.array_equal(A.prims(), B.prims()) and np.array_equal(A.fluxes(), B.fluxes())
    assert np.array_equal(A.pflag(), B.pflag()) and np.array_equal(A.nfail(), B.nfail())
    assert A.time() == B.time() and np.array_equal(A.status()[1], B.status()[1])
