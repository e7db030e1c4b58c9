"""The queued full recovery tree with many zones queued (hundreds of workgroup
tiles, the last one partly filled) and with few, against the host build of the same
bodies: primitives to 1e-9, flags and counters exactly."""
import numpy as np
import pytest

from helpers import interior
from coolharm3d_amd import Harm3D, torus, torus_grid


@pytest.mark.gpu
@pytest.mark.parametrize("n,scale", [((30, 23, 17), 1e-4), ((12, 10, 8), 1e-4), ((13, 11, 64), 1.0)], ids=str)
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_queue_matches_host_build(n, scale, precision):
    g = torus_grid(*n)
    p = torus(g)
    p[..., 1] *= scale                 # u far below b^2: the entropy fix takes the magnetised zones
    runs = []
    for host in (False, True):
        H = Harm3D(g, hostcheck=host, precision=precision)
        H.set_prims(p)
        H.fixup_bounds()
        H.set_time(0.0, 1e-4)
        H.step_ch(2)
        runs.append(H)
    G, C = runs
    if scale < 1.0:
        assert C.nfailtot()[5] > 64    # NFAIL_USE_EE: more than one tile of 64
    assert np.array_equal(interior(G.pflag()), interior(C.pflag()))
    assert np.array_equal(G.nfailtot(), C.nfailtot())
    tol = 1e-9 if precision == "fp64" else 1e-5
    for v in (0, 1, 2, 4):
        a, b = interior(C.prims())[..., v], interior(G.prims())[..., v]
        assert np.abs(a - b).sum() <= tol * np.abs(a).sum(), v
