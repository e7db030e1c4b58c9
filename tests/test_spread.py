"""Small grids with short x3 rows take fewer points per wavefront: the same state,
fluxes, flags and counters, bit for bit, as with full wavefronts (launch shapes set
by the caller), at remainders, around the largest grid spread and the shortest row not."""
import numpy as np
import pytest

from coolharm3d_amd import Harm3D, balsara1, balsara1_grid, torus, torus_grid

pytestmark = pytest.mark.gpu

CASES = [
    dict(n=4), dict(n=62), dict(n=514, precision="mixed"), dict(n=1026), dict(n=16382), dict(n=16386),
    dict(n=(20, 13, 3)), dict(n=(24, 17, 4), precision="mixed"), dict(n=(9, 11, 7)), dict(n=(9, 11, 8)),
    dict(n=(12, 12, 3), recon=2, ct_para=0, flux=0),
]


@pytest.mark.parametrize("case", CASES, ids=str)
def test_spread_equals_full_wavefronts(case):
    kw = dict(case)
    n = kw.pop("n")
    grid = balsara1_grid(n) if isinstance(n, int) else torus_grid(*n)
    p = balsara1(grid) if isinstance(n, int) else torus(grid)
    runs = []
    for full in (False, True):
        H = Harm3D(grid, **kw)
        if full:
            for f in ("flux1", "emf", "conserved"):
                bs, kc, flags = H.launch_shape(f)
                assert f == "flux1" or flags & 256
                H.set_launch_shape(f, bs, kc, flags & ~(128 | 256))   # neither one launch nor spread
        H.set_prims(p)
        H.fixup_bounds()
        H.set_time(0.0, min(grid.dx[0], 1e-7) if isinstance(n, int) else grid.dx[0])
        H.step_ch(3)
        runs.append(H)
    A, B = runs
    assert np.array_equal(A.prims(), B.prims()) and np.array_equal(A.fluxes(), B.fluxes())
    assert np.array_equal(A.pflag(), B.pflag()) and np.array_equal(A.nfail(), B.nfail())
    assert A.time() == B.time() and np.array_equal(A.status()[1], B.status()[1])
