"""The face fluxes of a stage in one launch against a launch per direction: state,
fluxes, flags and counters bit for bit, on planes smaller than a workgroup, ragged
planes, degenerate directions, every precision and metric."""
import numpy as np
import pytest

from coolharm3d_amd import Harm3D, balsara1, balsara1_grid, bbh_disk, bbh_grid, torus, torus_grid
from coolharm3d_amd.pn import PnMetric
from coolharm3d_amd.problems import bbh_gdet

pytestmark = pytest.mark.gpu

CASES = [
    dict(problem="shock", n=64), dict(problem="shock", n=514, precision="mixed"),      # 1D: planes of 9 points
    dict(problem="torus", n=(13, 3, 5)), dict(problem="torus", n=(12, 10, 64)),
    dict(problem="torus", n=(17, 21, 19), precision="mixed"),
    dict(problem="torus", n=(12, 12, 9), recon=2, ct_para=0, flux=0),                   # one face per thread
    dict(problem="torus", n=(9, 12, 8), recon=2, ct_para=0, precision="mixed"),
    dict(problem="disk", n=(12, 8, 10)), dict(problem="disk", n=(11, 9, 16), precision="mixed"),
]


@pytest.mark.parametrize("case", CASES, ids=str)
def test_one_launch_equals_three(case):
    kw = dict(case)
    problem, n = kw.pop("problem"), kw.pop("n")
    if problem == "shock":
        grid = balsara1_grid(n)
        p = balsara1(grid)
    elif problem == "torus":
        grid = torus_grid(*n)
        p = torus(grid)
    else:
        grid = bbh_grid(*n)
        p = bbh_disk(grid, bbh_gdet(grid, PnMetric))
    runs = []
    for per_direction in (False, True):
        H = Harm3D(grid, **kw)
        if per_direction:
            bs, kc, flags = H.launch_shape("flux1")
            assert flags & 128
            H.set_launch_shape("flux1", bs, kc, flags & ~128)
        H.set_prims(p)
        H.fixup_bounds()
        H.set_time(0.0, grid.dx[0])
        H.step_ch(4)
        runs.append(H)
    A, B = runs
    assert np.array_equal(A.prims(), B.prims()) and np.array_equal(A.fluxes(), B.fluxes())
    assert np.array_equal(A.pflag(), B.pflag()) and np.array_equal(A.nfail(), B.nfail())
    assert A.time() == B.time() and np.array_equal(A.status()[1], B.status()[1])
