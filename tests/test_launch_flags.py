"""Launch shapes as they are reported: what runs, and what runs again after a caller
has set shapes of its own and put the old ones back."""
import pytest

from coolharm3d_amd import Harm3D, balsara1, balsara1_grid, torus, torus_grid

pytestmark = pytest.mark.gpu

ONE_LAUNCH, SPREAD = 128, 256


def _context(n, **kw):
    grid = balsara1_grid(n) if isinstance(n, int) else torus_grid(*n)
    H = Harm3D(grid, **kw)
    H.set_prims(balsara1(grid) if isinstance(n, int) else torus(grid))
    H.fixup_bounds()
    H.set_time(0.0, 1e-6)
    H.step_ch(1)
    return H


def _flux_launches(H):
    H.profile_enable(True)
    H.step_ch(1)
    n = H.profile_read("flux")[1]
    H.profile_enable(False)
    return n


FLUXES = ("flux1", "flux2", "flux3")


@pytest.mark.parametrize("n", [(13, 12, 9), 64], ids=str)
def test_flux_shapes_set_and_put_back(n):
    H = _context(n)
    before = [H.launch_shape(f) for f in FLUXES]
    assert all(s[2] & ONE_LAUNCH for s in before) and _flux_launches(H) == 2
    for f, (bs, kc, flags) in zip(FLUXES, before):          # one family at a time
        H.set_launch_shape(f, bs, kc, flags & ~ONE_LAUNCH)
        assert H.launch_shape(f) == (bs, kc, flags & ~ONE_LAUNCH) and _flux_launches(H) == 6
        H.set_launch_shape(f, bs, kc, flags)
        assert _flux_launches(H) == 2
    for f in FLUXES:                                        # all of them, back in another order
        H.set_launch_shape(f, 128, 0, 1)
    assert _flux_launches(H) == 6
    for f, s in list(zip(FLUXES, before))[::-1]:
        H.set_launch_shape(f, *s)
    assert [H.launch_shape(f) for f in FLUXES] == before and _flux_launches(H) == 2


def test_no_shared_launch_with_a_degenerate_direction():
    H = _context(64, recon=5)
    assert not any(H.launch_shape(f)[2] & ONE_LAUNCH for f in FLUXES) and _flux_launches(H) == 6
    with pytest.raises(RuntimeError):
        H.set_launch_shape("emf", 256, 0, ONE_LAUNCH)


@pytest.mark.parametrize("n", [(13, 12, 9), 64], ids=str)
def test_autotuner_reports_the_launch_that_runs(n):
    H = _context(n)
    rep = H.autotune(reps=1)
    ones = [bool(rep[f][2] & ONE_LAUNCH) for f in FLUXES]
    assert all(ones) or not any(ones)
    assert [H.launch_shape(f) for f in FLUXES] == [rep[f][:3] for f in FLUXES]
    assert _flux_launches(H) == (2 if ones[0] else 6)


def test_autotuner_keeps_the_spread():
    H = _context(1024)
    before = {f: H.launch_shape(f) for f in ("emf", "conserved")}
    assert all(s[2] & SPREAD for s in before.values())
    rep = H.autotune(reps=1)
    for f in before:
        assert rep[f][2] & SPREAD and H.launch_shape(f)[2] & SPREAD
        H.set_launch_shape(f, *before[f])
        assert H.launch_shape(f) == before[f]
    with pytest.raises(RuntimeError):
        H.set_launch_shape("flux1", 256, 0, SPREAD)
