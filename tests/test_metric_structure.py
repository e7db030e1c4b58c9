"""Kernels compiled for the geometry records' structure (Kerr-Schild zero
pattern, Minkowski) against the general ones: the same state, flags and counters
bit for bit.  The general kernels are reached with records whose zero pattern is
broken by the smallest subnormal, which changes no sum that is not zero."""
import os
import subprocess

import numpy as np
import pytest

from coolharm3d_amd import Harm3D, balsara1, balsara1_grid, torus, torus_grid

GCON, GCOV = 0, 16       # offsets of gcon[4][4] and gcov[4][4] in a 42-double record


def _run(grid, p, general, hostcheck, steps, **kw):
    H = Harm3D(grid, hostcheck=hostcheck, **kw)
    if general:
        g, _ = H.geometry()
        g[0, GCON + 2] = g[0, GCON + 8] = 5e-324      # gcon[0][2], gcon[2][0] of the first record
        H.set_geometry(geom=g)
    H.set_prims(p)
    H.fixup_bounds()
    H.set_time(0.0, grid.dx[0])
    H.step_ch(steps)
    return H


def _compare(case, hostcheck):
    kw = dict(case)
    steps = 6
    if kw.pop("problem") == "shock":
        grid = balsara1_grid(kw.pop("n"))
        p = balsara1(grid)
    else:
        grid = torus_grid(*kw.pop("n"), coords=kw.pop("coords", "mks"))
        p = torus(grid)
    A = _run(grid, p, False, hostcheck, steps, **kw)
    B = _run(grid, p, True, hostcheck, steps, **kw)
    # where a sum is exactly zero the subnormal shows; nothing else may differ
    assert np.abs(A.prims() - B.prims()).max() <= 1e-300
    assert np.array_equal(A.pflag(), B.pflag()) and np.array_equal(A.nfail(), B.nfail())
    assert A.time() == B.time() and A.m_tot() == B.m_tot()


CASES = [
    dict(problem="torus", n=(14, 13, 9)),                                   # ragged rows
    dict(problem="torus", n=(12, 12, 64), precision="mixed"),               # row-aligned update
    dict(problem="torus", n=(12, 10, 64)),
    dict(problem="torus", n=(13, 12, 8), precision="mixed", coords="diag3"),
    dict(problem="torus", n=(12, 12, 8), recon=2, ct_para=0, flux=0),       # one face per thread
    dict(problem="torus", n=(12, 12, 8), recon=2, ct_para=0, flux=0, precision="mixed"),
    dict(problem="shock", n=128),
    dict(problem="shock", n=128, precision="mixed"),
]


CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "coolharm3d_amd", "csrc")
GK_GEN, GK_FLAT, GK_KS = 0, 1, 2
KIND = r"""
#include <cstdio>
#include <vector>
#include "hgpu_types.h"
int main(int, char** a) {
  FILE* f = fopen(a[1], "rb");
  fseek(f, 0, SEEK_END);
  const long long n = ftell(f) / (long long)sizeof(hgpu::Geom);
  rewind(f);
  std::vector<hgpu::Geom> r(n);
  if (fread(r.data(), sizeof(hgpu::Geom), n, f) != (size_t)n) return 1;
  printf("%d\n", hgpu::metric_structure(r.data(), n, a[2][0] == '1'));
}
"""


def test_structure_found(tmp_path):
    """The contexts compared here do run the kernels of the structure that they are
    named for: what metric_structure() finds on their records, and on broken ones."""
    src, exe, rec = tmp_path / "kind.cpp", tmp_path / "kind", tmp_path / "records"
    src.write_text(KIND)
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + CSRC, "-o",
                    str(exe), str(src)], check=True)

    def kind(g, flat_metric):
        np.ascontiguousarray(g).tofile(rec)
        return int(subprocess.run([str(exe), str(rec), "1" if flat_metric else "0"], capture_output=True, text=True,
                                  check=True).stdout)
    for coords in ("mks", "diag3"):
        g, _ = Harm3D(torus_grid(13, 12, 8, coords=coords), hostcheck=True).geometry()
        assert kind(g, False) == GK_KS
        for at in (GCON + 2, GCOV + 6, 35 + 1, 38 + 2):       # g^{t2}, g_{12}, beta^2, n^2 of one record
            b = g.copy()
            b[len(b) // 2, at] = 5e-324
            assert kind(b, False) == GK_GEN
        b = g.copy()
        b[3, GCOV + 5] = np.nan
        assert kind(b, False) == GK_GEN
    m, _ = Harm3D(balsara1_grid(64), hostcheck=True).geometry()
    assert kind(m, True) == GK_FLAT and kind(m, False) != GK_FLAT
    m[0, 32] = 1.0 + 2.0 ** -52
    assert kind(m, True) != GK_FLAT


@pytest.mark.parametrize("case", CASES, ids=str)
def test_structure_equals_general_hostbuild(case):
    _compare(case, hostcheck=True)


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=str)
def test_structure_equals_general_gpu(case):
    _compare(case, hostcheck=False)


def _minkowski_on_kerr_context(hostcheck, general, conn_scale, **kw):
    """A context of the Kerr metric given Minkowski records and a connection of its
    own (cooling on): its source terms stay."""
    grid = torus_grid(12, 11, 8)
    H = Harm3D(grid, hostcheck=hostcheck, **kw)
    g, c = H.geometry()
    r = np.zeros(42)
    r[GCON:GCON + 16] = r[GCOV:GCOV + 16] = np.diag([-1.0, 1.0, 1.0, 1.0]).ravel()
    r[32:35] = 1.0                                        # g, g_inv, alpha
    r[38] = 1.0                                           # ncon[0]
    g[:] = r
    if general:
        g[0, GCON + 2] = g[0, GCON + 8] = 5e-324
    rng = np.random.default_rng(11)
    H.set_geometry(geom=g, conn=conn_scale * rng.standard_normal(c.shape))
    p = np.empty(H.shape + (8,))
    p[..., :2] = rng.uniform(1.0, 2.0, H.shape + (2,))
    p[..., 2:] = rng.uniform(-0.1, 0.1, H.shape + (6,))
    H.set_prims(p)
    H.fixup_bounds()
    H.set_time(0.0, 1e-4)
    H.step_ch(2)
    return H


def _compare_minkowski(hostcheck, precision):
    A, B, N = (_minkowski_on_kerr_context(hostcheck, general, scale, precision=precision)
               for general, scale in ((False, 1.0), (True, 1.0), (True, 0.0)))
    assert np.abs(A.prims() - B.prims()).max() <= 1e-300
    assert np.array_equal(A.nfail(), B.nfail())
    assert np.abs(B.prims() - N.prims()).max() > 1e-5     # the connection's terms are there


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_minkowski_records_keep_sources_hostbuild(precision):
    _compare_minkowski(True, precision)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_minkowski_records_keep_sources_gpu(precision):
    _compare_minkowski(False, precision)
