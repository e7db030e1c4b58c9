// hgpu_launch.h -- launch shapes, the tile decomposition and the workgroup
// reductions shared by the device translation units of the advance
// (hgpu_kernels.hip, hgpu_flux.hip).
#pragma once
#include "hgpu_core.h"
#include <hip/hip_runtime.h>
#include <algorithm>
#include <type_traits>

namespace hgpu {

constexpr int BLOCK = 256;

// Launch shape of a stencil-kernel family (tile decomposition below).
struct LaunchShape {
  unsigned bs = 256;     // threads per workgroup: 64, 128 or 256
  unsigned kc = 0;       // k-extent of a 2D tile, dividing bs; 0 = flat tiles
  unsigned remap = 1;    // XCD-contiguous tile order
  unsigned order = 0;    // 0: plane after plane; 1: x1 fastest (one (j,k) tile through consecutive planes)
  unsigned occ = 0;      // 1: the register-capped kernel variant (flux, conserved update)
  unsigned fused = 0;    // conserved update only: 1 = update and inversion in one kernel
  unsigned fpt = 1;      // face fluxes only: faces per thread along the direction (1, 2, 4)
  unsigned stage = 0;    // x3 face fluxes (FP64, PPM, fpt > 1): reconstruction from LDS-staged pencils
  unsigned all = 0;      // face fluxes: 1: in one launch with the other directions, while they have it too
  unsigned spread = 0;   // 1: small grids are spread over more wavefronts (spread_shape)
  unsigned sp = 0;       // only the first 64 >> sp lanes of a wavefront take a point
};
enum { FAM_FLUX1 = 0, FAM_FLUX2, FAM_FLUX3, FAM_EMF, FAM_CONS, FAM_INV, N_FAM };


// --------------------------------------------------------------------------
__device__ __forceinline__ int wave_sum(int v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

__device__ __forceinline__ unsigned long long wave_max_u64(unsigned long long v) {
  for (int off = 32; off > 0; off >>= 1) {
    const unsigned long long o = __shfl_xor(v, off, 64);
    v = (o > v) ? o : v;
  }
  return v;
}

// Writes the fail() tallies of a workgroup: per-zone nfail, and block totals of
// nfailtot and the failure words, reduced in LDS so each status word receives
// at most one atomic per workgroup.  Every thread of the block must call it.
// The LDS addresses carry a zero that the compiler cannot see through: it turns
// atomics of a wavefront on one address into a loop over its lanes on the
// scalar unit (most zones count USE_FULL_INV), the LDS unit adds them faster.
// Corrector update of 24x24x16: 0.9 us of 13; k_recover on the 192x192x128 torus
// 68 -> 65 us.
__device__ __forceinline__ void commit_fail(const Params& P, const Ptrs& X, const FailRec& fr,
                                            bool active, long long c, unsigned mask) {
  __shared__ unsigned s_cnt[N_NFAIL];
  __shared__ unsigned s_flags;
  const long long NT = P.nt;
  const int tid = threadIdx.x;
  if (tid < N_NFAIL) s_cnt[tid] = 0;
  if (tid == 0) s_flags = 0;
  __syncthreads();
  if (active) {
    unsigned z;
    asm("v_mov_b32 %0, 0" : "=v"(z));
    for (int l = 0; l < N_NFAIL; l++) {
      if (!(mask & (1u << l))) continue;
      const int v = fr.nf[l];
      if (v) {
        if (P.track_nfail) X.nfail[l*NT + c] += v;
        atomicAdd(&s_cnt[l + z], (unsigned)v);
      }
    }
    if (fr.pflag) {
      unsigned f = 1u | ((fr.pflag == PFLAG_INTERP_PRIM) ? 2u : 4u) | ((fr.boundary & 1) ? 8u : 0u) |
                   ((fr.boundary & 2) ? 16u : 0u);
      atomicOr(&s_flags + z, f);
    }
  }
  __syncthreads();
  if (tid < N_NFAIL && s_cnt[tid]) atomicAdd(&X.status[ST_NFAILTOT + tid], (unsigned long long)s_cnt[tid]);
  if (tid == 0) {
    const unsigned f = s_flags;
    if (f) {
      atomicOr(&X.status[ST_FAILURE_EXISTS], 1ull);
      atomicOr(&X.status[ST_PFDIRTY], 1ull);
      if (f & 2u) atomicOr(&X.status[ST_FAILTYPE_PRIM], 1ull);
      if (f & 4u) atomicOr(&X.status[ST_FAILTYPE_V], 1ull);
      if (f & 8u) atomicOr(&X.status[ST_BOUNDARY_PHYS], 1ull);
      if (f & 16u) atomicOr(&X.status[ST_BOUNDARY_MPI], 1ull);
    }
  }
}

// The face fluxes' tallies, wavefront by wavefront without a barrier: the
// GAMMA_CALC failures (rare) and the fastest face speed, into the workgroup's line.
__device__ __forceinline__ void commit_flux(const Ptrs& X, const FailRec& fr, bool active, int vmax_slot) {
  const int v = active ? fr.nf[NFAIL_GAMMA_CALC] : 0;
  const bool first = (threadIdx.x & 63) == 0;
  if (__ballot(v != 0)) {
    const int n = wave_sum(v);
    if (first) atomicAdd(&X.status[ST_NFAILTOT + NFAIL_GAMMA_CALC], (unsigned long long)n);
  }
  const unsigned long long m = wave_max_u64(active ? dbl_bits(fr.vmax) : 0ull);
  if (first && m) atomicMax(&X.status[VS_FIRST + VS_LINE * (blockIdx.x & (N_VSLOT - 1)) + vmax_slot], m);
}

// ST_VMAX of the stage from the workgroups' lines, by one wavefront; the
// failure words' dirty mark goes down here too, after k_begin_stage's use.
__device__ __forceinline__ void fold_flux_words(const Ptrs& X) {
  if (threadIdx.x >= 64) return;
  unsigned long long m[3] = {0, 0, 0};
  for (int s = threadIdx.x; s < N_VSLOT; s += 64)
    for (int d = 0; d < 3; d++) {
      const unsigned long long o = X.status[VS_FIRST + VS_LINE * s + 1 + d];
      m[d] = o > m[d] ? o : m[d];
    }
  for (int d = 0; d < 3; d++) m[d] = wave_max_u64(m[d]);
  if (threadIdx.x == 0) {
    for (int d = 0; d < 3; d++) X.status[ST_VMAX + 1 + d] = m[d];
    X.status[ST_PFDIRTY] = 0;
  }
}

// Work decomposition of the stencil kernels.  The index box is cut into
// x1-planes of (j,k) and each plane into tiles of one workgroup: either bs
// consecutive (j,k) points (k fastest; kc = 0), or kc k-points x bs/kc j-rows
// (kc > 0).  Hardware dispatches workgroup p to XCD p % 8, and each XCD has its
// own L2; with remap set, the logical tile of workgroup p is chosen so that
// every XCD gets one contiguous range of tiles (whole x1-slabs), processed in
// order, so the +-3-zone stencils of neighbouring tiles hit the same L2.  With
// order = 1 consecutive workgroups take one (j,k) tile through consecutive
// x1-planes, so an x1 stencil finds the planes it shares with the previous
// workgroup in L2.  The shape of each kernel family is picked by the autotuner
// (or set by the caller).
struct Tiling {
  unsigned ni, nj, nk;  // box extents (ni: rows of tiles, i.e. x1-planes, or groups of pp of them)
  unsigned bs, kc, jr;  // threads; tile: kc x jr (kc > 0) or bs >> sp consecutive points (kc = 0)
  unsigned sp;          // only the first 64 >> sp lanes of a wavefront take a point
  unsigned nkt;         // tiles along k (2D tiles)
  unsigned pp, np;      // x1-planes per flat tile (small planes), x1-planes in all
  unsigned X;           // tiles per plane
  unsigned nblocks;     // X * ni, rounded up to a multiple of 8 when remapped
  unsigned remap;
  unsigned order;
};

// Small grids whose rows along x3 are shorter than a cache line (1D grids, 2D
// ones in x1 and x2): the 64 lanes of a wavefront touch a line each with every
// load, about 60 loads one after the other on one compute unit, and most compute
// units have no wavefront at all.  Workgroups of one wavefront with 64 >> sp
// points each spread them, as long as that makes no more than one wavefront for
// two SIMDs (512 on the 256-CU part).  1024-zone shock tube: update 21 -> 10 us a launch, step 0.097 ->
// 0.074 ms (0.075 up to 1024 wavefronts, 0.081 up to 2048, where the dispatch of
// the workgroups takes over).  Longer rows share their lines between lanes and lose:
// 24x24x16, spread twofold 0.170 -> 0.172 ms, fourfold 0.187.
static inline LaunchShape spread_shape(LaunchShape L, const Box& b, long long points, unsigned simds) {
  if (!L.spread || L.kc || b.hi[2] - b.lo[2] + 1 >= 8) return L;
  const long long waves = (points + 63) / 64;
  while (L.sp < 4 && (waves << (L.sp + 1)) <= simds / 2) L.sp++;
  if (L.sp) L.bs = 64;
  return L;
}

static inline Tiling make_tiling(const Box& b, const LaunchShape& L = LaunchShape()) {
  Tiling T;
  T.nk = (unsigned)(b.hi[2] - b.lo[2] + 1);
  T.nj = (unsigned)(b.hi[1] - b.lo[1] + 1);
  T.ni = T.np = (unsigned)(b.hi[0] - b.lo[0] + 1);
  T.pp = 1;
  T.bs = L.bs;
  T.sp = L.sp;
  const unsigned pts = L.bs >> L.sp;
  T.remap = L.remap;
  T.order = L.order;
  if (L.kc > 0 && L.kc < T.nk && L.bs % L.kc == 0 && L.sp == 0) {
    T.kc = L.kc;
    T.jr = L.bs / L.kc;
    T.nkt = (T.nk + T.kc - 1) / T.kc;
    T.X = T.nkt * ((T.nj + T.jr - 1) / T.jr);
  } else {
    T.kc = 0;
    T.jr = 0;
    T.nkt = 0;
    T.X = (T.nj * T.nk + pts - 1) / pts;
    // planes smaller than a tile: several to a tile (a 1D grid's planes hold a
    // handful of points, and a workgroup per plane left 250 of 256 threads idle)
    T.pp = std::max(1u, pts / (T.nj * T.nk));
    T.ni = (T.np + T.pp - 1) / T.pp;
  }
  T.nblocks = T.X * T.ni;
  if (T.remap) T.nblocks = ((T.nblocks + 7u) / 8u) * 8u;
  return T;
}

// point (i, j, k) of this thread in tile t of tile row ii.  SP: the kernel may be
// launched with spread tiles.
template <bool SP = false>
__device__ __forceinline__ bool tile_point(const Box& b, const Tiling& T, unsigned ii, unsigned t, int& i, int& j,
                                           int& k) {
  unsigned jj, kk, r0 = threadIdx.x;
  if (SP && T.sp) {
    const unsigned lanes = 64u >> T.sp, lane = r0 & 63u;
    if (lane >= lanes) return false;
    r0 = (r0 >> 6) * lanes + lane;
  }
  if (T.pp > 1) {        // X = 1
    const unsigned np = T.nj * T.nk, di = r0 / np, q = r0 - di * np;
    ii = ii * T.pp + di;
    if (di >= T.pp || ii >= T.np) return false;
    jj = q / T.nk;
    kk = q - jj * T.nk;
  } else if (T.kc == 0) {
    const unsigned q = t * (SP ? T.bs >> T.sp : T.bs) + r0;
    jj = q / T.nk;
    kk = q - jj * T.nk;
    if (jj >= T.nj) return false;
  } else {
    const unsigned tj = t / T.nkt;
    const unsigned tk = t - tj * T.nkt;
    const unsigned r = threadIdx.x / T.kc;
    kk = tk * T.kc + (threadIdx.x - r * T.kc);
    jj = tj * T.jr + r;
    if (kk >= T.nk || jj >= T.nj) return false;
  }
  i = b.lo[0] + (int)ii;
  j = b.lo[1] + (int)jj;
  k = b.lo[2] + (int)kk;
  return true;
}

template <bool SP = false>
__device__ __forceinline__ bool tile_index(const Box& b, const Tiling& T, int& i, int& j, int& k) {
  const unsigned p = blockIdx.x;
  const unsigned L = T.remap ? (p & 7u) * (T.nblocks >> 3) + (p >> 3) : p;
  unsigned ii, t;
  if (T.order == 0) {
    ii = L / T.X;
    t = L - ii * T.X;
  } else {
    t = L / T.ni;
    ii = L - t * T.ni;
    if (t >= T.X) return false;
  }
  if (ii >= T.ni) return false;
  return tile_point<SP>(b, T, ii, t, i, j, k);
}

constexpr unsigned MASK_GAMMA = 1u << NFAIL_GAMMA_CALC;
constexpr unsigned MASK_ALL = (1u << N_NFAIL) - 1u;

// Positions and velocities of a level's orbit record (the 12 values the
// metric records read; not the time derivatives, which only the metric
// derivatives need): the same address in every lane, read through the
// scalar cache (constant address space) so they sit in SGPRs.
__device__ __forceinline__ PnOrbit orbit_load(const PnOrbit* p) {
  const __attribute__((address_space(4))) double* q = (const __attribute__((address_space(4))) double*)p;
  PnOrbit o;
  double* d = &o.y[0][0];
#pragma unroll
  for (int m = 0; m < 12; m++) d[m] = q[m];
  return o;
}


// hgpu_flux.hip: face fluxes of direction d with launch shape L
void launch_flux_dir(int d, const Params& P, const Ptrs& X, const LaunchShape& L, const double* src, hipStream_t st,
                     const PnGrid& G, int lvl);
// The three directions in one launch (flux_all_possible()), 1, 2 or 4 faces per
// thread by the grid's size and the device's SIMDs
bool flux_all_possible(const Params& P);
void launch_flux_all(const Params& P, const Ptrs& X, const double* src, hipStream_t st, const PnGrid& G, int lvl,
                     unsigned simds);

}  // namespace hgpu
