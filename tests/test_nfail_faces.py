"""Faces of several directions that fail at the same zone: the zone's map entry
counts every one of them.  The face records carry a negative spatial metric, so
gamma_calc() fails for both states of every face of the launch; against a launch
per direction, and against the totals, exactly."""
import numpy as np
import pytest

from coolharm3d_amd import Harm3D, torus, torus_grid
from helpers import interior

pytestmark = pytest.mark.gpu

GAMMA_CALC = 3                 # NFAIL_GAMMA_CALC
FACES, GCOV = slice(0, 3), 16  # FACE1..FACE3 of [5 pos][N1T][N2T]; gcov[4][4] within a record


@pytest.mark.parametrize("case", [
    dict(n=(20, 18, 13)),                                            # one face per thread
    dict(n=(44, 40, 37)), dict(n=(44, 40, 37), precision="mixed"),   # two
    dict(n=(70, 72, 71), precision="mixed"),                         # four
    dict(n=(40, 36, 33), recon=2, ct_para=0, flux=0),                # MC slopes
], ids=str)
def test_every_failing_face_counts(case):
    kw = dict(case)
    grid = torus_grid(*kw.pop("n"))
    p = torus(grid)
    p[..., 2:5] = np.random.default_rng(5).uniform(1e-3, 2e-3, p.shape[:3] + (3,))
    maps = []
    for per_direction in (False, True):
        H = Harm3D(grid, **kw)
        if per_direction:
            for f in ("flux1", "flux2", "flux3"):
                bs, kc, flags = H.launch_shape(f)
                H.set_launch_shape(f, bs, kc, flags & ~128)
        H.set_prims(p)
        H.fixup_bounds()
        g, _ = H.geometry()
        r = g.reshape(5, H.shape[0], H.shape[1], 42)
        for a in (1, 2, 3):
            r[FACES, :, :, GCOV + 4*a + 1:GCOV + 4*a + 4] *= -1.0
        H.set_geometry(geom=g)
        H.reset_nfail()
        H.set_time(0.0, 1e-10)
        H.advance_only(0)
        maps.append(H.nfail()[GAMMA_CALC])
        assert maps[-1].sum() == H.nfailtot()[GAMMA_CALC]
    assert (interior(maps[0]) >= 6).mean() > 0.99      # two states of three faces
    assert np.array_equal(maps[0], maps[1])
