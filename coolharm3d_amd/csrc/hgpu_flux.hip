// hgpu_flux.hip -- face-flux kernels of the GRMHD advance (reconstruction and
// Riemann solve), FP64 and mixed precision, static and binary metric.
#include "hgpu_launch.h"

namespace hgpu {

// n GAMMA_CALC failures of a face into the map's zone c.  The faces (i,j,k) of the
// three directions share the zone and may run at the same time, in workgroups of
// one launch, so the (rare) addition is atomic.
__device__ __forceinline__ void tally_face(const Params& P, const Ptrs& X, long long c, int n) {
  if (P.track_nfail && n) atomicAdd(&X.nfail[NFAIL_GAMMA_CALC*P.nt + c], n);
}

// W: minimum waves per SIMD the register allocation must allow (1 = the
// compiler's choice; larger values cap the VGPRs, trading spills for occupancy).
// K: structure of the geometry records (GK_*).
template <int D, int W, int K>
__global__ __launch_bounds__(BLOCK, W) void k_flux(Params P, Ptrs X, const double* __restrict__ src, Box b, Tiling T) {
  int i, j, k;
  const bool active = tile_index(b, T, i, j, k);
  FailRec fr; fr.clear();
  long long c = 0;
  if (active) {
    flux_face<D, K>(P, X, src, i, j, k, fr);
    c = cidx(P, i, j, k);
  }
  if (active) tally_face(P, X, c, fr.nf[NFAIL_GAMMA_CALC]);
  commit_flux(X, fr, active, D + 1);
}

template <int D, int W, int K>
__global__ __launch_bounds__(BLOCK, W) void k_flux_mixed(Params P, Ptrs X, const double* __restrict__ src, Box b,
                                                         Tiling T) {
  int i, j, k;
  const bool active = tile_index(b, T, i, j, k);
  FailRec fr; fr.clear();
  long long c = 0;
  if (active) {
    flux_face_mixed<D, K>(P, X, src, i, j, k, fr);
    c = cidx(P, i, j, k);
  }
  if (active) tally_face(P, X, c, fr.nf[NFAIL_GAMMA_CALC]);
  commit_flux(X, fr, active, D + 1);
}

__device__ __forceinline__ long long wave_min_ll(long long v) {
  for (int off = 32; off > 0; off >>= 1) {
    const long long o = __shfl_xor(v, off, 64);
    v = (o < v) ? o : v;
  }
  return v;
}
__device__ __forceinline__ long long wave_max_ll(long long v) {
  for (int off = 32; off > 0; off >>= 1) {
    const long long o = __shfl_xor(v, off, 64);
    v = (o > v) ? o : v;
  }
  return v;
}

// Orders LDS accesses of a wavefront to a buffer of its own: its LDS operations
// complete in order, so a wavefront-scope fence (no workgroup barrier) puts
// one lane's stores before the other lanes' reads, and those before the next
// stores.
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// LDS capacity (doubles) of one primitive's x3 pencil of a wavefront: 64 face
// groups of F faces need 64 F + 5 consecutive zones, plus the ghost zones
// skipped where the wavefront's groups continue on the next (i,j) row.
template <int F> constexpr int stage_cap() { return 64 * F + 5 + 3 * (F + 8); }

// PPM+MC face states of the F consecutive x3 faces of every lane (ppm_faces()
// with d = 2) from LDS-staged pencils.  The zones the wavefront's stencils
// cover form one contiguous range of the array (k is its fastest index), so
// each primitive's range is loaded once, coalesced, by all 64 lanes (about
// F + 1 loads per lane instead of F + 5), stored to LDS, and each lane reads
// its F + 5 window from there; the next primitive's loads are in flight
// while this one's limiters run (double-buffered).  A wavefront whose range
// exceeds the buffer (rows shorter than the wavefront) reads its windows from
// global memory instead.  Same values, same arithmetic as ppm_faces(): the
// face states are bit-identical.  Every lane of the wavefront must call it;
// inactive lanes only help stage.
template <int F>
__device__ void ppm_faces_x3_staged(const Params& P, const Ptrs& X, const double* __restrict__ src, bool active,
                                    int i, int j, int k, double (*pl)[NP], double (*pr)[NP], double* buf) {
  constexpr int M = F + 5;
  constexpr int CAP = stage_cap<F>();
  constexpr int NL = (CAP + 63) / 64;
  const long long NT = P.nt;
  const int lane = threadIdx.x & 63;
  int ii = i, jj = j;
  if (P.degen[0]) ii = NG;
  if (P.degen[1]) jj = NG;
  const long long c0 = active ? cidx(P, ii, jj, k - 3) : 0;
  int zm[M];
#pragma unroll
  for (int m = 0; m < M; m++) zm[m] = imin(m, P.n3t - 1 - (k - 3));
  const long long lo = wave_min_ll(active ? c0 : LLONG_MAX);
  const long long hi = wave_max_ll(active ? c0 + zm[M - 1] : LLONG_MIN);
  const long long span = (hi >= lo) ? hi - lo + 1 : 0;
  const bool staged = span > 0 && span <= CAP;   // wavefront-uniform
  const int off = (int)(c0 - lo);
  double r[NL];
  if (staged) {
#pragma unroll
    for (int q = 0; q < NL; q++) {
      const int e = q * 64 + lane;
      r[q] = (e < span) ? src[lo + e] : 0.;
    }
  }
#pragma unroll
  for (int v = 0; v < NP; v++) {
    double* bv = buf + (v & 1) * CAP;
    if (staged) {
#pragma unroll
      for (int q = 0; q < NL; q++) {
        const int e = q * 64 + lane;
        if (e < span) bv[e] = r[q];
      }
      if (v + 1 < NP) {
#pragma unroll
        for (int q = 0; q < NL; q++) {
          const int e = q * 64 + lane;
          r[q] = (e < span) ? src[(v + 1) * NT + lo + e] : 0.;
        }
      }
    }
    wave_lds_order();
    if (active) {
      const int s = rs_slot(v);
      const double ra = X.rscale[s * P.n1t + ii], ri = X.irscale[s * P.n1t + ii];
      double y[M];
#pragma unroll
      for (int m = 0; m < M; m++) {
        const double raw = staged ? bv[off + zm[m]] : src[v * NT + c0 + zm[m]];
        y[m] = (raw * ra) * ri;
      }
      double dq[M - 1], fi[M - 2], le[M - 2], re[M - 2];
#pragma unroll
      for (int m = 1; m < M - 1; m++) dq[m] = mc_slope_vect(y[m - 1], y[m], y[m + 1]);
#pragma unroll
      for (int m = 1; m < M - 2; m++) fi[m] = 0.5 * (y[m + 1] + y[m]) - PPM_FACTOR * (dq[m + 1] - dq[m]);
#pragma unroll
      for (int m = 2; m < M - 2; m++) ppm_limit(fi[m - 1], fi[m], y[m], &le[m], &re[m]);
#pragma unroll
      for (int f = 0; f < F; f++) {
        pl[f][v] = re[2 + f];
        pr[f][v] = le[3 + f];
      }
    }
  }
}

// F consecutive faces along D per thread (PPM+MC, D not degenerate): the
// thread's tile index along D counts groups of F faces from bg.lo[D]; faces
// past hi_d (the flux box end) are skipped.  Each zone's parabola is computed
// once per group.  The per-face fail() tally goes to the face's zone here,
// the totals through commit_flux().
// Along x3 (the fastest index of the arrays) a lane's F faces are adjacent in
// memory, so the fluxes go through LDS: slot s of lane l stores element
// s*64 + l of the wavefront's F*64 faces, and each store instruction writes
// consecutive faces.
// OTF: the face records are evaluated from the orbit of level lvl (binary
// metric) instead of read.
// STG (x3, FP64): reconstruction from LDS-staged pencils (ppm_faces_x3_staged).
// K: structure of the stored geometry records (the evaluated ones are GK_DIAG).
// active, (i, j, k): the thread's point of the box of face groups.
template <int D, int F, bool MIXED, int K, bool OTF, bool STG>
__device__ __forceinline__ void flux_multi_block(const Params& P, const Ptrs& X, const double* __restrict__ src,
                                                 const Box& bg, int hi_d, const PnGrid& G, int lvl, bool active, int i,
                                                 int j, int k) {
  using Real = typename std::conditional<MIXED, float, double>::type;
  static_assert(!STG || (D == 2 && !MIXED && !OTF), "staged pencils: FP64 x3 faces of a static metric");
  constexpr bool TRANSPOSE = (D == 2);
  __shared__ Real tbuf[TRANSPOSE ? BLOCK * F : 1];
  __shared__ double sbuf[STG ? (BLOCK / 64) * 2 * stage_cap<F>() : 1];
  FailRec fr; fr.clear();
  Real fo[F][NP];
  long long cb = 0;
  int nv = 0;
  Real pl[F][NP], pr[F][NP];
  if (active) {
    const int lo = bg.lo[D];
    if (D == 0) i = lo + (i - lo) * F;
    else if (D == 1) j = lo + (j - lo) * F;
    else k = lo + (k - lo) * F;
  }
  if constexpr (STG) ppm_faces_x3_staged<F>(P, X, src, active, i, j, k, pl, pr, sbuf + (threadIdx.x >> 6) * 2 * stage_cap<F>());
  if (active) {
    constexpr int di = (D == 0), dj = (D == 1), dk = (D == 2);
    const int nvalid = min(F, hi_d - ((D == 0) ? i : ((D == 1) ? j : k)) + 1);
    if constexpr (STG) {
    } else if constexpr (MIXED) {
      ppm_faces_mixed<D, F>(P, X, src, i, j, k, pl, pr);
    } else {
      ppm_faces<D, F>(P, X, src, i, j, k, pl, pr);
    }
    PnOrbit orb;
    if constexpr (OTF) orb = orbit_load(X.orbit + lvl);
#pragma unroll
    for (int f = 0; f < F; f++) {
      if (f >= nvalid) break;
      const int g0 = fr.nf[NFAIL_GAMMA_CALC];
      const int fi = i + f*di, fj = j + f*dj, fk = k + f*dk;
      if constexpr (OTF) {
        if constexpr (MIXED) {
          GeomF gfb;
          pn_zone_geomf(P, G, orb, fi, fj, fk, D, &gfb);
          flux_riemann_mixed_g<D>(P, X, pl[f], pr[f], fi, fj, fk, fr, TRANSPOSE ? fo[f] : nullptr,
                                  GeomView<GK_DIAG, const GeomF*>{&gfb});
        } else {
          Geom gb;
          pn_zone_geom(P, G, orb, fi, fj, fk, D, &gb);
          flux_riemann_g<D>(P, X, pl[f], pr[f], fi, fj, fk, fr, TRANSPOSE ? fo[f] : nullptr,
                            GeomView<GK_DIAG, const Geom*>{&gb});
        }
      } else {
        if constexpr (MIXED) flux_riemann_mixed<D, K>(P, X, pl[f], pr[f], fi, fj, fk, fr, TRANSPOSE ? fo[f] : nullptr);
        else flux_riemann<D, K>(P, X, pl[f], pr[f], fi, fj, fk, fr, TRANSPOSE ? fo[f] : nullptr);
      }
      const int dv = fr.nf[NFAIL_GAMMA_CALC] - g0;
      tally_face(P, X, cidx(P, fi, fj, fk), dv);
    }
    cb = cidx(P, i, j, k);
    nv = nvalid;
  }
  if constexpr (TRANSPOSE) {
    Real* Fa = MIXED ? (Real*)X.Ff : (Real*)X.F;
    const int lane = threadIdx.x & 63;
    Real* wbuf = tbuf + (threadIdx.x & ~63) * F;
    long long cs[F];
    bool ok[F];
#pragma unroll
    for (int s = 0; s < F; s++) {
      const int e = s*64 + lane, sl = e / F, f = e % F;
      cs[s] = __shfl(cb, sl, 64) + f;
      ok[s] = f < __shfl(nv, sl, 64);
    }
#pragma unroll
    for (int l = 0; l < NP; l++) {
      if (l == B3) continue;   // the normal field's flux: never read
      wave_lds_order();
#pragma unroll
      for (int f = 0; f < F; f++) wbuf[lane*F + f] = fo[f][l];
      wave_lds_order();
#pragma unroll
      for (int s = 0; s < F; s++)
        if (ok[s]) Fa[(2*NFLUX + l)*(long long)P.nt + cs[s]] = wbuf[s*64 + lane];
    }
  }
  commit_flux(X, fr, active, D + 1);
}

template <int D, int F, int W, bool MIXED, int K, bool OTF = false, bool STG = false>
__global__ __launch_bounds__(BLOCK, W) void k_flux_multi(Params P, Ptrs X, const double* __restrict__ src, Box bg,
                                                         Tiling T, int hi_d, PnGrid G, int lvl) {
  int i, j, k;
  const bool active = tile_index(bg, T, i, j, k);
  flux_multi_block<D, F, MIXED, K, OTF, STG>(P, X, src, bg, hi_d, G, lvl, active, i, j, k);
}

// The three directions in one launch.  The workgroups go through the grid in
// slabs of F x1-planes, every slab's x1 face groups, then its x2 and x3 ones, so
// the state a slab reads is read by all three directions while it is in the
// caches (three launches read it from HBM three times), and the launch has
// one tail instead of three.  Fluxes of a step, three launches -> one: FP64
// 192x192x128 1.74 -> 1.62 ms, mixed 1.15 -> 1.11, binary disk 120x64x160 0.42 ->
// 0.35, 67x45x33 0.136 -> 0.081, a 1024-zone shock tube 0.055 -> 0.022.
struct FluxAll {
  Box bg[3];
  int hi[3];
  Tiling T[3];
  unsigned rows[3];          // tile rows of each direction in a slab
  unsigned per, nblocks;     // workgroups per slab, in all
  unsigned remap;            // XCD-contiguous slabs
};
static FluxAll make_flux_all(const Params& P, unsigned F, LaunchShape& L, unsigned simds) {
  FluxAll A;
  long long points = 0;
  bool small = false;
  for (int d = 0; d < 3; d++) {
    const Box b = flux_box(P, d);
    A.bg[d] = b;
    A.hi[d] = b.hi[d];
    A.bg[d].hi[d] = b.lo[d] + (b.hi[d] - b.lo[d] + (int)F) / (int)F - 1;
    points += A.bg[d].count();
  }
  L = spread_shape(L, A.bg[0], points, simds);
  for (int d = 0; d < 3; d++) {
    A.T[d] = make_tiling(A.bg[d], L);
    small = small || A.T[d].pp > 1;
  }
  // planes smaller than a workgroup: one slab
  unsigned slabs = 1;
  for (int d = 0; d < 3; d++) {
    A.rows[d] = small ? A.T[d].ni : ((d == 0) ? 1u : F);
    slabs = std::max(slabs, (A.T[d].ni + A.rows[d] - 1) / A.rows[d]);
  }
  A.per = A.rows[0] * A.T[0].X + A.rows[1] * A.T[1].X + A.rows[2] * A.T[2].X;
  A.remap = L.remap;
  A.nblocks = A.per * slabs;
  if (A.remap) A.nblocks = (A.nblocks + 7u) / 8u * 8u;
  return A;
}
// direction, tile row (of the direction's box) and tile of this workgroup;
// false where there is none
__device__ __forceinline__ bool flux_all_slot(const FluxAll& A, int& d, unsigned& ii, unsigned& t) {
  const unsigned p = blockIdx.x;
  const unsigned L = A.remap ? (p & 7u) * (A.nblocks >> 3) + (p >> 3) : p;
  const unsigned slab = L / A.per;
  unsigned s = L - slab * A.per, X = A.T[0].X, rows = A.rows[0], ni = A.T[0].ni;
  d = 0;
  if (s >= rows * X) {
    s -= rows * X;
    X = A.T[1].X; rows = A.rows[1]; ni = A.T[1].ni;
    d = 1;
    if (s >= rows * X) {
      s -= rows * X;
      X = A.T[2].X; rows = A.rows[2]; ni = A.T[2].ni;
      d = 2;
    }
  }
  const unsigned q = s / X;
  ii = slab * rows + q;
  t = s - q * X;
  return ii < ni;
}
template <int F, int W, bool MIXED, int K, bool OTF>
__global__ __launch_bounds__(BLOCK, W) void k_flux_all(Params P, Ptrs X, const double* __restrict__ src, FluxAll A,
                                                       PnGrid G, int lvl) {
  int d;
  unsigned ii, t;
  if (!flux_all_slot(A, d, ii, t)) return;   // the same in every thread
  int i = 0, j = 0, k = 0;
  if (d == 0) {
    const bool active = tile_point(A.bg[0], A.T[0], ii, t, i, j, k);
    flux_multi_block<0, F, MIXED, K, OTF, false>(P, X, src, A.bg[0], A.hi[0], G, lvl, active, i, j, k);
  } else if (d == 1) {
    const bool active = tile_point(A.bg[1], A.T[1], ii, t, i, j, k);
    flux_multi_block<1, F, MIXED, K, OTF, false>(P, X, src, A.bg[1], A.hi[1], G, lvl, active, i, j, k);
  } else {
    const bool active = tile_point(A.bg[2], A.T[2], ii, t, i, j, k);
    flux_multi_block<2, F, MIXED, K, OTF, false>(P, X, src, A.bg[2], A.hi[2], G, lvl, active, i, j, k);
  }
}

// The same with one face per thread (MC slopes, degenerate directions, small grids)
template <int D, bool MIXED, int K>
__device__ __forceinline__ void flux_one_block(const Params& P, const Ptrs& X, const double* __restrict__ src,
                                               bool active, int i, int j, int k) {
  FailRec fr; fr.clear();
  long long c = 0;
  if (active) {
    if constexpr (MIXED) flux_face_mixed<D, K>(P, X, src, i, j, k, fr);
    else flux_face<D, K>(P, X, src, i, j, k, fr);
    c = cidx(P, i, j, k);
  }
  if (active) tally_face(P, X, c, fr.nf[NFAIL_GAMMA_CALC]);
  commit_flux(X, fr, active, D + 1);
}
template <int W, bool MIXED, int K>
__global__ __launch_bounds__(BLOCK, W) void k_flux_all_one(Params P, Ptrs X, const double* __restrict__ src,
                                                           FluxAll A) {
  int d;
  unsigned ii, t;
  if (!flux_all_slot(A, d, ii, t)) return;
  int i = 0, j = 0, k = 0;
  if (d == 0) {
    const bool active = tile_point<true>(A.bg[0], A.T[0], ii, t, i, j, k);
    flux_one_block<0, MIXED, K>(P, X, src, active, i, j, k);
  } else if (d == 1) {
    const bool active = tile_point<true>(A.bg[1], A.T[1], ii, t, i, j, k);
    flux_one_block<1, MIXED, K>(P, X, src, active, i, j, k);
  } else {
    const bool active = tile_point<true>(A.bg[2], A.T[2], ii, t, i, j, k);
    flux_one_block<2, MIXED, K>(P, X, src, active, i, j, k);
  }
}

// f(constant of the geometry records' structure)
template <class F>
static void with_kind(int kind, F&& f) {
  if (kind == GK_FLAT) f(std::integral_constant<int, GK_FLAT>());
  else if (kind == GK_KS) f(std::integral_constant<int, GK_KS>());
  else f(std::integral_constant<int, GK_GEN>());
}

// Face fluxes along D with launch shape L: one face per thread, or fpt faces
// per thread (PPM+MC with D not degenerate) over the box of face groups.
template <int D, int F, bool MIXED>
static void launch_flux_multi(const Params& P, const Ptrs& X, const LaunchShape& L, const double* src, const Box& b,
                              hipStream_t st, const PnGrid& G, int lvl) {
  Box bg = b;
  const int n = b.hi[D] - b.lo[D] + 1;
  bg.hi[D] = b.lo[D] + (n + F - 1) / F - 1;
  const Tiling T = make_tiling(bg, L);
  const dim3 grid(T.nblocks), blk(T.bs);
  if (P.otf) {
    // three waves per SIMD fit the FP32 face solve without spilling
    if constexpr (MIXED) hipLaunchKernelGGL((k_flux_multi<D, F, 3, true, GK_GEN, true>), grid, blk, 0, st, P, X, src, bg, T, b.hi[D], G, lvl);
    else hipLaunchKernelGGL((k_flux_multi<D, F, 1, false, GK_GEN, true>), grid, blk, 0, st, P, X, src, bg, T, b.hi[D], G, lvl);
    return;
  }
  if constexpr (D == 2 && !MIXED) {
    if (L.stage) {   // reconstruction from LDS-staged pencils
      if (L.occ) hipLaunchKernelGGL((k_flux_multi<D, F, 3, false, GK_GEN, false, true>), grid, blk, 0, st, P, X, src, bg, T, b.hi[D], G, lvl);
      else hipLaunchKernelGGL((k_flux_multi<D, F, 1, false, GK_GEN, false, true>), grid, blk, 0, st, P, X, src, bg, T, b.hi[D], G, lvl);
      return;
    }
  }
  // register-capped variants: 4 waves/SIMD for the FP32 solve, 3 for FP64
  const auto go = [&](auto K) {
    constexpr int k = decltype(K)::value;
    if (L.occ) hipLaunchKernelGGL((k_flux_multi<D, F, MIXED ? 4 : 3, MIXED, k>), grid, blk, 0, st, P, X, src, bg, T, b.hi[D], G, lvl);
    else hipLaunchKernelGGL((k_flux_multi<D, F, 1, MIXED, k>), grid, blk, 0, st, P, X, src, bg, T, b.hi[D], G, lvl);
  };
  if (P.gkind == GK_KS) go(std::integral_constant<int, GK_KS>());
  else go(std::integral_constant<int, GK_GEN>());
}

// G, lvl: the binary metric's grid and the stage's level, read when P.otf
// (which implies PPM and no degenerate direction: the face-group kernels,
// with at least 2 faces per thread).
template <int D>
static void launch_flux_d(const Params& P, const Ptrs& X, const LaunchShape& L, const double* src, const Box& b,
                          hipStream_t st, const PnGrid& G, int lvl) {
  if ((L.fpt > 1 || P.otf) && P.recon == RECON_PPM_MC && !P.degen[D]) {
    if (P.mixed) {
      if (L.fpt == 4) launch_flux_multi<D, 4, true>(P, X, L, src, b, st, G, lvl);
      else launch_flux_multi<D, 2, true>(P, X, L, src, b, st, G, lvl);
    } else {
      if (L.fpt == 4) launch_flux_multi<D, 4, false>(P, X, L, src, b, st, G, lvl);
      else launch_flux_multi<D, 2, false>(P, X, L, src, b, st, G, lvl);
    }
    return;
  }
  const Tiling T = make_tiling(b, L);
  const dim3 grid(T.nblocks), blk(T.bs);
  with_kind(P.gkind, [&](auto K) {
    constexpr int k = decltype(K)::value;
    if (P.mixed) {
      if (L.occ) hipLaunchKernelGGL((k_flux_mixed<D, 6, k>), grid, blk, 0, st, P, X, src, b, T);
      else hipLaunchKernelGGL((k_flux_mixed<D, 1, k>), grid, blk, 0, st, P, X, src, b, T);
    } else {
      if (L.occ) hipLaunchKernelGGL((k_flux<D, 4, k>), grid, blk, 0, st, P, X, src, b, T);
      else hipLaunchKernelGGL((k_flux<D, 1, k>), grid, blk, 0, st, P, X, src, b, T);
    }
  });
}

void launch_flux_dir(int d, const Params& P, const Ptrs& X, const LaunchShape& L, const double* src, hipStream_t st,
                     const PnGrid& G, int lvl) {
  const Box b = flux_box(P, d);
  if (d == 0) launch_flux_d<0>(P, X, L, src, b, st, G, lvl);
  else if (d == 1) launch_flux_d<1>(P, X, L, src, b, st, G, lvl);
  else launch_flux_d<2>(P, X, L, src, b, st, G, lvl);
}

// All three directions have face groups, or none has: a mix of both kinds
// keeps a launch per direction.
static bool flux_all_multi(const Params& P) {
  return P.recon == RECON_PPM_MC && !P.degen[0] && !P.degen[1] && !P.degen[2];
}
bool flux_all_possible(const Params& P) {
  return flux_all_multi(P) || P.recon != RECON_PPM_MC;
}
// Faces per thread.  A group's zones are reconstructed once for the whole group, so
// more faces per thread are less work, in fewer and longer wavefronts.  Up to one
// wavefront per SIMD (simds: the device's, 1024 where the figures were taken) a
// launch is one wavefront's chain: one face (24x24x16, a step's fluxes: FP64 0.045 -> 0.027 ms, mixed 0.037 -> 0.026; at 48x48x32, 3900 wavefronts
// of single faces, mixed 0.046 and 0.044 but a slower step).  Once groups of 4 fill
// the FP32 solve's 4 wavefronts per SIMD, 4 faces: mixed 192x192x128 1.05 -> 0.885 ms,
// 96x96x64 0.140 -> 0.136, binary disk 120x64x160 0.343 -> 0.303; 67x45x33, which
// does not, 0.051 -> 0.057.  FP64 groups of 4 take 254 registers, two wavefronts
// per SIMD, and gain nothing (1.61 ms at 192x192x128; disk 0.67 -> 0.94).
static unsigned flux_all_faces(const Params& P, long long faces, unsigned simds) {
  if (!flux_all_multi(P)) return 1;
  if (faces <= 64ll * simds && !P.otf) return 1;
  return (P.mixed && faces >= 4 * 64ll * (4 * simds)) ? 4 : 2;
}
void launch_flux_all(const Params& P, const Ptrs& X, const double* src, hipStream_t st, const PnGrid& G, int lvl,
                     unsigned simds) {
  // Flat tiles of 256 in dispatch order: round-robin over the XCDs, so that
  // all of them work on one slab (1.62 ms a step on the 192x192x128 torus
  // against 1.70 with a contiguous range of slabs per XCD; tiles of 64 run into
  // the dispatch rate, 2.98 ms; 2D tiles of 64 x 4 take 2.34).
  LaunchShape L;
  L.remap = 0;
  long long faces = 0;
  for (int d = 0; d < 3; d++) faces += flux_box(P, d).count();
  const unsigned F = flux_all_faces(P, faces, simds);
  L.spread = F == 1;
  const FluxAll A = make_flux_all(P, F, L, simds);
  const dim3 grid(A.nblocks), blk(L.bs);
  if (F > 1) {
    if (P.otf) {
      if (P.mixed && F == 4) hipLaunchKernelGGL((k_flux_all<4, 3, true, GK_GEN, true>), grid, blk, 0, st, P, X, src, A, G, lvl);
      else if (P.mixed) hipLaunchKernelGGL((k_flux_all<2, 3, true, GK_GEN, true>), grid, blk, 0, st, P, X, src, A, G, lvl);
      else hipLaunchKernelGGL((k_flux_all<2, 1, false, GK_GEN, true>), grid, blk, 0, st, P, X, src, A, G, lvl);
      return;
    }
    const auto go = [&](auto K) {
      constexpr int k = decltype(K)::value;
      if (P.mixed && F == 4) hipLaunchKernelGGL((k_flux_all<4, 4, true, k, false>), grid, blk, 0, st, P, X, src, A, G, lvl);
      else if (P.mixed) hipLaunchKernelGGL((k_flux_all<2, 4, true, k, false>), grid, blk, 0, st, P, X, src, A, G, lvl);
      else hipLaunchKernelGGL((k_flux_all<2, 3, false, k, false>), grid, blk, 0, st, P, X, src, A, G, lvl);
    };
    if (P.gkind == GK_KS) go(std::integral_constant<int, GK_KS>());
    else go(std::integral_constant<int, GK_GEN>());
    return;
  }
  with_kind(P.gkind, [&](auto K) {
    constexpr int k = decltype(K)::value;
    if (P.mixed) hipLaunchKernelGGL((k_flux_all_one<6, true, k>), grid, blk, 0, st, P, X, src, A);
    else hipLaunchKernelGGL((k_flux_all_one<4, false, k>), grid, blk, 0, st, P, X, src, A);
  });
}

}  // namespace hgpu
