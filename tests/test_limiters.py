"""The limiters by selects against the limiters by branches (FP64: both forms of the
header; FP32: the branches written out here), bit for bit, on ordinary values, ties,
signed zeros, denormals, infinities and NaN."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "coolharm3d_amd", "csrc")

SOURCE = r"""
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>
#include "hgpu_mixed.h"
using namespace hgpu;
static float slope_f(float a, float b) {
  if (a*b <= 0.f) return 0.f;
  const float aa = fabsf(a), ab = fabsf(b);
  if (aa + aa + aa <= ab) return a + a;
  if (ab + ab + ab <= aa) return b + b;
  return 0.5f*(a + b);
}
static void limit_f(float l, float r, float* ln, float* rn) {
  if (-r*l <= 0.f) { *ln = *rn = 0.f; return; }
  const float r2 = r + r, l2 = l + l;
  *ln = l; *rn = r;
  if (r > l) {
    if (0.f > (l + r2)) *ln = -r2;
    if (0.f < (l2 + r)) *rn = -l2;
  } else {
    if (0.f < (l + r2)) *ln = -r2;
    if (0.f > (l2 + r)) *rn = -l2;
  }
}
static double slope_linear(double y1, double y2, double y3) {   // src/recon.c:88-132
  const double m = 2.*(y2 - y1), p = 2.*(y3 - y2), c = 0.5*(y3 - y1);
  if (m*p <= 0.) return 0.;
  if (fabs(m) <= fabs(p) && fabs(m) <= fabs(c)) return m;
  return (fabs(p) <= fabs(c)) ? p : c;
}
template <class T> static bool same(T a, T b) { return (a != a && b != b) || !memcmp(&a, &b, sizeof(T)); }
template <class T> static T pick(std::mt19937_64& g) {
  typedef std::numeric_limits<T> L;
  const T edge[] = {T(0), -T(0), T(1), T(-1), T(3), T(1)/3, L::denorm_min(), -L::min(), L::max(), L::lowest(), L::infinity(), -L::infinity(), L::quiet_NaN(), T(2), T(0.5)};
  const unsigned k = g() % 24;
  if (k < 15) return edge[k];
  if (k < 19) return T(int(g() % 9)) - T(4);
  return std::normal_distribution<T>(0, 1)(g);
}
int main() {
  std::mt19937_64 g(7);
  long bad = 0;
  for (int n = 0; n < 2000000; n++) {
    double y[6], l1, r1, l2, r2;
    for (double& v : y) v = pick<double>(g);
    if (!same(mc_slope_vect(y[0], y[1], y[2]), mc_slope_sel(y[0], y[1], y[2]))) bad++;
    if (!same(slope_linear(y[0], y[1], y[2]), mc_slope(y[0], y[1], y[2]))) bad++;
    ppm_limit(y[0], y[1], y[2], &l1, &r1);
    ppm_limit_sel(y[0], y[1], y[2], &l2, &r2);
    if (!same(l1, l2) || !same(r1, r2)) bad++;
    ppm_interface<true>(y, &l1, &r1);
    ppm_interface<false>(y, &l2, &r2);
    if (!same(l1, l2) || !same(r1, r2)) bad++;
    const float a = pick<float>(g), b = pick<float>(g);
    float fl1, fr1, fl2, fr2;
    if (!same(slope_f(a, b), mc_slope_diff(a, b))) bad++;
    limit_f(a, b, &fl1, &fr1);
    ppm_limit_rel(a, b, &fl2, &fr2);
    if (!same(fl1, fl2) || !same(fr1, fr2)) bad++;
  }
  printf("%ld\n", bad);
  return bad != 0;
}
"""


def test_selects_equal_branches(tmp_path):
    src, exe = tmp_path / "limiters.cpp", tmp_path / "limiters"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + CSRC, "-o", str(exe), str(src)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout + out.stderr
