"""Copies of whole arrays between host and device through the pinned chunks: the
state there and back bit for bit, at sizes below one chunk, of several chunks,
and beyond the ring (several host threads, chunks reused), with a ragged end."""
import numpy as np
import pytest

from coolharm3d_amd import Harm3D, torus, torus_grid

pytestmark = pytest.mark.gpu


# zones with ghosts: 1089 (0.07 MB), 32760 (just below one 2 MB chunk), 32890 (just above),
# 170016 (10.9 MB, 6 chunks), 663136 (42 MB: 21 chunks through 8 slots)
@pytest.mark.parametrize("n", [(5, 3, 5), (22, 20, 39), (20, 17, 49), (60, 50, 40), (130, 100, 40)], ids=str)
def test_state_there_and_back(n):
    H = Harm3D(torus_grid(*n), track_nfail=0)
    rng = np.random.default_rng(sum(n))
    p = rng.random(H.shape + (8,))
    for which in (0, 1, 0):
        H.set_prims(p, which)
        assert np.array_equal(H.prims(which), p)
    # the box copy reads the same arrays by another route
    hi = [s - 1 for s in H.shape]
    assert np.array_equal(H.download_box(0, (0, 0, 0), hi)[0], p)


@pytest.mark.parametrize("n", [(12, 10, 8), (67, 45, 33)], ids=str)
def test_maps_after_a_step(n):
    g = torus_grid(*n)
    H = Harm3D(g)
    H.set_prims(torus(g))
    H.fixup_bounds()
    H.reset_nfail()
    H.set_time(0.0, 1e-5)
    H.step_ch(1)
    assert np.array_equal(H.nfail().sum(axis=(1, 2, 3)), H.nfailtot())
    hi = [s - 1 for s in H.shape]
    assert np.array_equal(H.download_box(0, (0, 0, 0), hi)[1], H.pflag())
    gam = H.gamma()[3:-3, 3:-3, 3:-3]
    assert (gam >= 1.0).all() and np.isfinite(gam).all()


@pytest.mark.parametrize("chunks", [0, 1, 2, 5])
@pytest.mark.parametrize("n", [(5, 3, 5), (60, 50, 40), (130, 100, 40)], ids=str)
def test_fewer_pinned_chunks(monkeypatch, chunks, n):
    """Rings of fewer chunks than a copy wants, and none: the plain copies."""
    monkeypatch.setenv("HGPU_PINNED_CHUNKS", str(chunks))
    H = Harm3D(torus_grid(*n), track_nfail=0)
    p = np.random.default_rng(chunks).random(H.shape + (8,))
    for which in (0, 1):
        H.set_prims(p, which)
        assert np.array_equal(H.prims(which), p)
    hi = [s - 1 for s in H.shape]
    box, flags = H.download_box(1, (0, 0, 0), hi)
    assert np.array_equal(box, p) and np.array_equal(flags, H.pflag())


def test_threads_read_one_context():
    """Several host threads read one context at the same time."""
    from concurrent.futures import ThreadPoolExecutor
    H = Harm3D(torus_grid(60, 50, 40))
    p = np.random.default_rng(2).random(H.shape + (8,))
    H.set_prims(p)
    H.set_prims(2.0 * p, 1)
    H.set_time(1.5, 0.25)

    def read(k):
        if k % 3 == 2:
            return H.time() == (1.5, 0.25, 0.25)
        return np.array_equal(H.prims(k % 3), p * (1 + k % 3))
    with ThreadPoolExecutor(4) as pool:
        assert all(pool.map(read, range(24)))
