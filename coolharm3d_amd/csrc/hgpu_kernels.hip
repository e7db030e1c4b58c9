// hgpu_kernels.hip -- MI355X (gfx950) backend of the per-substep GRMHD advance.
//
// Kernels are thin wrappers over the per-thread bodies of hgpu_bodies.h.  The
// 64 lanes of a wavefront walk contiguous zones of one x3 pencil (k fastest:
// coalesced SoA loads; the 2D geometry record is a wavefront-wide broadcast);
// the stencil kernels map workgroups to tiles XCD by XCD (Tiling in hgpu_launch.h).
// Failure counters are summed in LDS before one atomic per workgroup and word
// (commit_fail()); the face fluxes, which rarely fail, add theirs per wavefront.
#include "hgpu_launch.h"
#include "hgpu_xfer.h"
#include <cstdlib>

namespace hgpu {

struct ProfEvent { std::string name; hipEvent_t a, b; };

struct GpuPriv {
  hipStream_t stream = nullptr;
  unsigned simds = 1024;               // SIMDs of the device
  unsigned flag_grid = 1024;           // workgroups of the kernels that mostly find nothing to do
  bool prof = false;
  bool graph = false;                  // replay captured steps
  hipGraphExec_t step_exec = nullptr;  // one step_ch(), captured on first use
  LaunchShape shape[N_FAM];            // per kernel family
  std::vector<ProfEvent> pending;
  std::vector<hipEvent_t> pool;
  std::map<std::string, std::pair<double, long long>> acc;
  std::map<std::string, hipEvent_t> open;   // mark() begin events
  void* box_stage = nullptr;           // staging of hgpu_download_box / hgpu_upload_box
  size_t box_bytes = 0;
  XferRing ring;                       // pinned chunks of the copies to and from the host
};

static inline GpuPriv* priv(hgpu_ctx* c) { return static_cast<GpuPriv*>(c->be); }

static int hip_check(hipError_t e, const char* what) {
  if (e == hipSuccess) return 0;
  return set_error(-4, std::string(what) + ": " + hipGetErrorString(e));
}

// The holes' positions and velocities at the step's three levels
__global__ __launch_bounds__(64) void k_orbit(Ptrs X, PnBinary B, PnOrbit* out) {
  const int l = threadIdx.x;
  if (l < 3) pn_orbit_at(B, level_time(X, l), &out[l]);
}

template <bool BR>
__global__ __launch_bounds__(BLOCK) void k_emf(Params P, Ptrs X, Box b, Tiling T) {
  if (blockIdx.x == T.nblocks) { fold_flux_words(X); return; }   // a workgroup of its own, beside the edges'
  int i, j, k;
  if (!tile_index<true>(b, T, i, j, k)) return;
  emf_edge<BR>(P, X, i, j, k);
}

__global__ __launch_bounds__(BLOCK) void k_emf_mixed(Params P, Ptrs X, Box b, Tiling T) {
  if (blockIdx.x == T.nblocks) { fold_flux_words(X); return; }
  int i, j, k;
  if (!tile_index<true>(b, T, i, j, k)) return;
  emf_edge_mixed(P, X, i, j, k);
}

// M_tot of advance() (src/step_ch.c:309, :389): the sum of U^{n+1}[RHO] over
// the stage's zones, in three fixed-order levels so that the result does not
// depend on scheduling (it differs from the reference's serial loop only in
// the order of the additions):
//  1. the update: each wavefront's sum (a butterfly over the lanes), one part
//     per wavefront, no barrier;
//  2. k_recover (which follows every update): thread g of the grid adds the
//     parts g, g + G, g + 2G ... (G threads), each workgroup sums its threads;
//  3. the first boundary kernel of the stage: its first workgroup adds the
//     second-level parts.
// The kernel boundaries order each level's stores before the next's reads.
// The sum of a wavefront's 64 values, the same bits in every lane and on every
// run: within each row of 16 lanes, pairs, quads, halves and the row by DPP
// permutations (a + b == b + a exactly, so every lane of a row ends with the
// same row sum); then (row0 + row1) + (row2 + row3).  Every lane active.
__device__ __forceinline__ double dpp_f64(double v, int ctrl_sel) {
  const unsigned long long u = __double_as_longlong(v);
  int lo = (int)(unsigned)u, hi = (int)(unsigned)(u >> 32);
  switch (ctrl_sel) {   // the DPP control must be a constant
    case 0: lo = __builtin_amdgcn_mov_dpp(lo, 0xB1, 0xF, 0xF, false); hi = __builtin_amdgcn_mov_dpp(hi, 0xB1, 0xF, 0xF, false); break;
    case 1: lo = __builtin_amdgcn_mov_dpp(lo, 0x4E, 0xF, 0xF, false); hi = __builtin_amdgcn_mov_dpp(hi, 0x4E, 0xF, 0xF, false); break;
    case 2: lo = __builtin_amdgcn_mov_dpp(lo, 0x141, 0xF, 0xF, false); hi = __builtin_amdgcn_mov_dpp(hi, 0x141, 0xF, 0xF, false); break;
    default: lo = __builtin_amdgcn_mov_dpp(lo, 0x140, 0xF, 0xF, false); hi = __builtin_amdgcn_mov_dpp(hi, 0x140, 0xF, 0xF, false); break;
  }
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
__device__ __forceinline__ double lane_f64(double v, int lane) {
  const unsigned long long u = __double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)u, lane);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), lane);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ double wave_sum_fixed(double v) {
  v += dpp_f64(v, 0);   // quad_perm [1,0,3,2]: pairs
  v += dpp_f64(v, 1);   // quad_perm [2,3,0,1]: quads
  v += dpp_f64(v, 2);   // row_half_mirror: eights
  v += dpp_f64(v, 3);   // row_mirror: rows of 16
  return (lane_f64(v, 0) + lane_f64(v, 16)) + (lane_f64(v, 32) + lane_f64(v, 48));
}
__device__ __forceinline__ double block_sum_fixed(double v, double* s_w) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  v = wave_sum_fixed(v);
  if (lane == 0) s_w[wv] = v;
  __syncthreads();
  double b = 0.;
  for (int q = 0; q < nw; q++) b += s_w[q];
  __syncthreads();
  return b;
}
__device__ __forceinline__ void mtot_wave_part(const Ptrs& X, double v) {
  v = wave_sum_fixed(v);
  const unsigned nw = blockDim.x >> 6;
  if ((threadIdx.x & 63) == 0) X.mpart[blockIdx.x * nw + (threadIdx.x >> 6)] = v;
  if (blockIdx.x == 0 && threadIdx.x == 0) X.status[ST_MPARTS] = (unsigned long long)gridDim.x * nw;
}
// every thread of every workgroup of the grid
__device__ __forceinline__ void mtot_level2(const Ptrs& X) {
  __shared__ double s_w[16];
  const unsigned n = (unsigned)X.status[ST_MPARTS];
  const unsigned G = gridDim.x * blockDim.x;
  double s = 0.;
  for (unsigned q = blockIdx.x * blockDim.x + threadIdx.x; q < n; q += G) s += X.mpart[q];
  const double b = block_sum_fixed(s, s_w);
  if (threadIdx.x == 0) X.mpart2[blockIdx.x] = b;
  if (blockIdx.x == 0 && threadIdx.x == 0) X.status[ST_MPARTS2] = gridDim.x;
}
// every thread of one workgroup
__device__ __forceinline__ void mtot_level3(const Ptrs& X) {
  __shared__ double s_w[BLOCK / 64];
  const unsigned n = (unsigned)X.status[ST_MPARTS2];
  double s = 0.;
  for (unsigned q = threadIdx.x; q < n; q += blockDim.x) s += X.mpart2[q];
  const double tot = block_sum_fixed(s, s_w);
  if (threadIdx.x == 0) X.scal[SC_MTOT] = tot;
}

// Conserved update U^{n+1} of every interior zone into the U buffer
// ([8][NT], indexed like the state).
template <bool MIXED, int W>
__global__ __launch_bounds__(BLOCK, W) void k_conserved(Params P, Ptrs X, int stage, Box b, Tiling T) {
  int i, j, k;
  const bool active = tile_index(b, T, i, j, k);
  FailRec fr; fr.clear();
  long long c = 0;
  double urho = 0.;
  if (active) {
    const double dt = X.scal[SC_DT];
    const double Dt = (stage == 0) ? 0.5*dt : dt;
    c = cidx(P, i, j, k);
    double U[NP];
    const int gid = geom_id(P, i, j, k, CENT);
    zone_conserved<MIXED>(P, X, stage, Dt, i, j, k, X.geom_n + gid, X.geom + gid, fr, U);
#pragma unroll
    for (int l = 0; l < NP; l++) X.Uslow[l*P.nt + c] = U[l];
    urho = U[RHO];
  }
  commit_fail(P, X, fr, active, c, MASK_GAMMA);
  mtot_wave_part(X, urho);
}

// The common con-to-prim branch; zones that need the full recover_primitives()
// tree are queued (wave-aggregated slot allocation) for k_recover.
__global__ __launch_bounds__(BLOCK) void k_invert(Params P, Ptrs X, int stage, Box b, Tiling T) {
  int i, j, k;
  const bool active = tile_index(b, T, i, j, k);
  FailRec fr; fr.clear();
  long long c = 0;
  bool queue = false;
  if (active) {
    c = cidx(P, i, j, k);
    double U[NP], pf[NP];
#pragma unroll
    for (int l = 0; l < NP; l++) U[l] = X.Uslow[l*P.nt + c];
    zone_guess(P, X, stage, i, c, pf);
    double pgam = 1.;
    if (recover_fast(P, X, i, j, k, pf, U, geom_at(P, X, i, j, k, CENT), floor_rho(P, X, i, c),
                     floor_uu(P, X, i, c), &pgam, fr))
      store_zone(P, X, stage, c, pf, pgam, fr);
    else
      queue = true;
  }
  const unsigned long long ballot = __ballot(queue);
  if (ballot) {
    const int lane = threadIdx.x & 63;
    const int leader = __ffsll((long long)ballot) - 1;
    unsigned base = 0;
    if (lane == leader) base = (unsigned)atomicAdd(&X.status[ST_SLOW], (unsigned long long)__popcll(ballot));
    base = __shfl(base, leader, 64);
    if (queue) X.slow_idx[base + (unsigned)__popcll(ballot & ((1ull << lane) - 1ull))] = (unsigned)c;
  }
  commit_fail(P, X, fr, active, c, MASK_ALL);
}

// Conserved update and the common con-to-prim branch in one pass: U^{n+1}
// stays in registers; only the zones queued for k_recover store it.
// OTF: the zone records at the stage's level (lvl, also U^n's in the
// predictor) and the result's (lvl + 1) are evaluated from the orbit.
// MET: 0 static metric, 1 binary metric (stored levels or, with OTF,
// evaluated records); each kernel carries only its metric's source branch.
// UNI: row-aligned tiles (each wavefront in one (i, j) column of a 2D static
// metric): the connection records are read through the scalar cache.
// K: structure of the static metric's records (GK_*).
template <bool MIXED, int W, bool OTF = false, int MET = 0, bool UNI = false, int K = GK_GEN>
__global__ __launch_bounds__(BLOCK, W) void k_update(Params P, Ptrs X, int stage, Box b, Tiling T, PnGrid G,
                                                     int lvl) {
  int i, j, k;
  const bool active = tile_index<true>(b, T, i, j, k);
  FailRec fr; fr.clear();
  long long c = 0;
  bool queue = false;
  double urho = 0.;
  if (active) {
    const double dt = X.scal[SC_DT];
    c = cidx(P, i, j, k);
    double U[NP];
    bool done;
    if constexpr (OTF) {
      // the stage's record for U^n in the predictor (the corrector reads U^n,
      // and the source terms come precomputed by k_source_otf: evaluating the
      // metric derivatives here needs their registers on top of the update's), then the result's record for the
      // inversion
      {
        Geom gs;
        if (stage == 0) pn_zone_geom(P, G, orbit_load(X.orbit + lvl), i, j, k, CENT, &gs);
        const GeomView<GK_DIAG, const Geom*> gv{&gs};
        zone_conserved<MIXED, 2>(P, X, stage, (stage == 0) ? 0.5*dt : dt, i, j, k, gv, gv, fr, U);
      }
      Geom gnew;
      pn_zone_geom(P, G, orbit_load(X.orbit + lvl + 1), i, j, k, CENT, &gnew);
      double pf[NP];
      zone_guess(P, X, stage, i, c, pf);
      double pgam = 1.;
      done = recover_fast(P, X, i, j, k, pf, U, GeomView<GK_DIAG, const Geom*>{&gnew}, floor_rho(P, X, i, c), floor_uu(P, X, i, c), &pgam, fr);
      if (done) store_zone(P, X, stage, c, pf, pgam, fr);
    } else {
      done = update_zone_fast<MIXED, MET, UNI, K>(P, X, stage, dt, i, j, k, fr, U);
    }
    urho = U[RHO];
    if (!done) {
      queue = true;
#pragma unroll
      for (int l = 0; l < NP; l++) X.Uslow[l*P.nt + c] = U[l];
    }
  }
  const unsigned long long ballot = __ballot(queue);
  if (ballot) {
    const int lane = threadIdx.x & 63;
    const int leader = __ffsll((long long)ballot) - 1;
    unsigned base = 0;
    if (lane == leader) base = (unsigned)atomicAdd(&X.status[ST_SLOW], (unsigned long long)__popcll(ballot));
    base = __shfl(base, leader, 64);
    if (queue) X.slow_idx[base + (unsigned)__popcll(ballot & ((1ull << lane) - 1ull))] = (unsigned)c;
  }
  commit_fail(P, X, fr, active, c, MASK_ALL);
  mtot_wave_part(X, urho);
}

// Full con-to-prim tree for the queued zones: a fixed grid strides over the
// queue, 64 zones to a workgroup of 8 wavefronts.  Few zones take the tree (a
// few thousandths of a torus), so the launch lasts as long as one zone's serial
// chain, and the chain is cut by what can run side by side: wavefronts 0-5 form
// the zones' six entropy face fluxes (one face each: reconstruction and two
// face states), wavefront 6 runs the 2D inversion and wavefront 7 the 1D one
// (used where the 2D one fails); then wavefront 6 goes on to the entropy solve
// with their results from LDS.  One thread per zone took 0.10 ms a stage on every
// torus (0.20 ms a step at 192x192x128, 0.19 at 67x45x33); this takes 0.14 and
// 0.08 ms a step, a launch being as long as its slowest zone.
// G, lvl: with OTF, the entropy fix's face records are evaluated from the
// orbit of level lvl.
constexpr int REC_Z = 64, REC_T = 8 * REC_Z;
template <bool MIXED, int OTF>
__global__ __launch_bounds__(REC_T) void k_recover(Params P, Ptrs X, int stage, PnGrid G, int lvl) {
  __shared__ double sF[6 * REC_Z];
  __shared__ double s1[(NP + 2) * REC_Z];
  __shared__ int sR[REC_Z];
  mtot_level2(X);   // the update's M_tot parts
  const unsigned n = (unsigned)X.status[ST_SLOW];
  const unsigned stride = gridDim.x * REC_Z;
  const unsigned rounds = (n + stride - 1) / stride;
  const double dt = X.scal[SC_DT];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (unsigned r = 0; r < rounds; r++) {
    const unsigned slot = r * stride + blockIdx.x * REC_Z + lane;
    const bool active = slot < n;
    FailRec fr; fr.clear();
    RecoverState rs;
    double U[NP];
    long long c = 0;
    int i = 0, j = 0, k = 0;
    FaceOtf fo;
    if constexpr (OTF) { fo.G = G; fo.o = X.orbit + lvl; }
    if (active) {
      c = X.slow_idx[slot];
      k = (int)(c % P.n3t);
      j = (int)((c / P.n3t) % P.n2t);
      i = (int)(c / ((long long)P.n3t * P.n2t));
      if (wv < 6) {
        sF[wv*REC_Z + lane] = entropy_face<MIXED>(P, X, (stage == 0) ? X.p : X.ph, wv, i, j, k, OTF ? &fo : nullptr);
      } else {
        Geom gb;
        const Geom* g = cent_rec<OTF>(P, X, i, j, k, gb);
#pragma unroll
        for (int l = 0; l < NP; l++) U[l] = X.Uslow[l*P.nt + c];
        zone_guess(P, X, stage, i, c, rs.pf);
        if (wv == 6) {
          recover_2d(P, U, g, rs);
        } else {
          Recover1d r1;
          recover_1d(P, U, g, rs.pf, r1);
#pragma unroll
          for (int l = 0; l < NP; l++) s1[l*REC_Z + lane] = r1.pf[l];
          s1[NP*REC_Z + lane] = r1.gamma;
          s1[(NP + 1)*REC_Z + lane] = r1.bsq;
          sR[lane] = r1.ret;
        }
      }
    }
    __syncthreads();
    const bool finish = active && wv == 6;
    if (finish) {
      if (rs.ret) {
        Recover1d r1;
#pragma unroll
        for (int l = 0; l < NP; l++) r1.pf[l] = s1[l*REC_Z + lane];
        r1.gamma = s1[NP*REC_Z + lane];
        r1.bsq = s1[(NP + 1)*REC_Z + lane];
        r1.ret = sR[lane];
        recover_take_1d(r1, rs);
      }
      recover_zone_end<MIXED, OTF>(P, X, stage, dt, i, j, k, U, rs, fr, OTF ? &fo : nullptr, sF + lane, REC_Z);
    }
    commit_fail(P, X, fr, finish, c, MASK_ALL);   // its barriers also keep the LDS until every zone has read it
  }
}

// bounds(): every ghost zone in one launch (bound_zone()).  Both of a stage's
// bounds, three launches each before: 0.135 -> 0.081 ms a step at 192x192x128,
// 0.079 -> 0.030 on small grids, where a launch costs more than its zones.
// mtot: after an update, whose M_tot the first workgroup completes.
// tstep: the step's last launch, whose first thread also takes the new time step
// (it needs the fluxes' speeds and the fixups' counters, not the ghosts).
template <int OTF>
__global__ __launch_bounds__(BLOCK) void k_bounds(Params P, Ptrs X, double* S, int skip_mpi, long long n, int mtot,
                                                  int tstep) {
  if (mtot && blockIdx.x == 0) mtot_level3(X);
  if (tstep && blockIdx.x == 0 && threadIdx.x == 0) timestep_update(P, X);
  if (skip_mpi && !X.status[ST_BOUNDARY_PHYS]) return;
  const int do_pflag = X.status[ST_FAILURE_EXISTS] ? 1 : 0;
  const long long stride = (long long)gridDim.x * BLOCK;
  const long long rounds = (n + stride - 1) / stride;   // the same in every workgroup (barriers)
  for (long long rd = 0; rd < rounds; rd++) {
    const long long t = rd * stride + (long long)blockIdx.x * BLOCK + threadIdx.x;
    const bool active = t < n;
    FailRec fr; fr.clear();
    long long c = 0;
    if (active) {
      int i, j, k;
      ghost_at(P, t, i, j, k);
      bound_zone<OTF>(P, X, S, i, j, k, do_pflag, fr);
      c = cidx(P, i, j, k);   // nfail of inflow_check() belongs to the ghost zone
    }
    commit_fail(P, X, fr, active, c, MASK_GAMMA);
  }
}

// Both interpolating fixups in one pass: a zone flagged for one of them reads
// only unflagged neighbours and writes only itself, so the velocity and the
// primitive fixups are independent and equal the reference's two sweeps.
__global__ __launch_bounds__(BLOCK) void k_fixup_interp(Params P, Ptrs X, double* S, Box b) {
  if (!X.status[ST_FAILURE_EXISTS]) return;
  if (!X.status[ST_FAILTYPE_PRIM] && !X.status[ST_FAILTYPE_V]) return;
  const long long n = b.count(), stride = (long long)gridDim.x * BLOCK;
  const long long rounds = (n + stride - 1) / stride;   // the same in every workgroup (barriers)
  for (long long rd = 0; rd < rounds; rd++) {
    const long long t = rd * stride + (long long)blockIdx.x * BLOCK + threadIdx.x;
    const bool active = t < n;
    FailRec fr; fr.clear();
    long long c = 0;
    if (active) {
      int i, j, k;
      b.at(t, i, j, k);
      c = cidx(P, i, j, k);
      const int which = X.pflag[c];
      if (which == PFLAG_INTERP_V || which == PFLAG_INTERP_PRIM) fixup_interp_zone(P, X, S, which, i, j, k, fr);
    }
    commit_fail(P, X, fr, active, c, MASK_ALL);
  }
}

__global__ __launch_bounds__(BLOCK) void k_fixup_init(Params P, Ptrs X, Box b) {
  long long t = (long long)blockIdx.x * BLOCK + threadIdx.x;
  const bool active = t < b.count();
  FailRec fr; fr.clear();
  long long c = 0;
  if (active) {
    int i, j, k;
    b.at(t, i, j, k);
    fixup_init_zone(P, X, i, j, k, fr);
    c = cidx(P, i, j, k);
  }
  commit_fail(P, X, fr, active, c, MASK_ALL);
}

// Start of a stage, one launch: the flag map cleared if a zone was flagged
// since it last was (a word of its own says so: the first workgroup may reset
// the others before the last one has started; k_emf clears it, after this
// kernel and before anything can flag a zone again), and the words a stage
// starts from: failure words, boundary flags, fastest speeds, an empty
// slow-zone queue.
__global__ __launch_bounds__(BLOCK) void k_begin_stage(Ptrs X, long long nt) {
  if (blockIdx.x == 0) {
    if (threadIdx.x == 0) {
      X.status[ST_FAILURE_EXISTS] = 0;
      X.status[ST_FAILTYPE_V] = 0;
      X.status[ST_FAILTYPE_PRIM] = 0;
      X.status[ST_BOUNDARY_PHYS] = 0;
      X.status[ST_BOUNDARY_MPI] = 0;
      X.status[ST_SLOW] = 0;
    }
    if (threadIdx.x < 4) X.status[ST_VMAX + threadIdx.x] = 0;
    for (int w = threadIdx.x; w < VS_LINE * N_VSLOT; w += BLOCK) X.status[VS_FIRST + w] = 0;
  }
  if (!X.status[ST_PFDIRTY]) return;
  const long long stride = (long long)gridDim.x * BLOCK;
  for (long long t = (long long)blockIdx.x * BLOCK + threadIdx.x; t < nt; t += stride) X.pflag[t] = 0;
}

__global__ void k_reset_words(Ptrs X, int first, int n) {
  if ((int)threadIdx.x < n) X.status[first + threadIdx.x] = 0;
}

// boundary_phys_pflag / boundary_mpi_pflag: set to given values (set = 1) or cleared
__global__ void k_boundary_words(Ptrs X, int set, int phys, int mpi) {
  if (threadIdx.x == 0) {
    X.status[ST_BOUNDARY_PHYS] = set ? (unsigned long long)(phys != 0) : 0ull;
    X.status[ST_BOUNDARY_MPI] = set ? (unsigned long long)(mpi != 0) : 0ull;
  }
}

// A box of zones of S (and pflag) to (to_box) or from a contiguous staging
// buffer: prims [t][8] then pflag [t], t the zone's position in the box.
__global__ __launch_bounds__(BLOCK) void k_box_copy(Params P, Ptrs X, double* S, Box b, double* stage,
                                                    int* pstage, int to_box) {
  const long long t = (long long)blockIdx.x * BLOCK + threadIdx.x;
  if (t >= b.count()) return;
  int i, j, k;
  b.at(t, i, j, k);
  const long long c = cidx(P, i, j, k);
  if (stage) {
    for (int v = 0; v < NP; v++) {
      if (to_box) stage[t*NP + v] = S[v*P.nt + c];
      else S[v*P.nt + c] = stage[t*NP + v];
    }
  }
  if (pstage) {
    if (to_box) pstage[t] = X.pflag[c];
    else X.pflag[c] = pstage[t];
  }
}

__global__ void k_timestep(Params P, Ptrs X) {
  if (threadIdx.x == 0) timestep_update(P, X);
}

__global__ __launch_bounds__(BLOCK) void k_zero(unsigned int* p, long long n) {
  long long t = (long long)blockIdx.x * BLOCK + threadIdx.x;
  if (t < n) p[t] = 0u;
}

__global__ __launch_bounds__(BLOCK) void k_divb(Params P, Ptrs X, Box b, unsigned long long* out) {
  long long t = (long long)blockIdx.x * BLOCK + threadIdx.x;
  if (t >= b.count()) return;
  int i, j, k;
  b.at(t, i, j, k);
  double v = divb_corner(P, X, X.p, i, j, k);
  if (v == v) atomicMax(out, dbl_bits(v));
}

// Time-dependent metric: geometry records of position pos of every zone at
// time level tsel, recomputed per zone, in FP64 (dst) and/or FP32 (dstf).  One
// wavefront computes 64 consecutive records, stages them in LDS and stores
// them as one contiguous, coalesced run.
constexpr int FILL_B = 64;
constexpr int GEOMF_FLOATS = (int)(sizeof(GeomF) / sizeof(float));
__global__ __launch_bounds__(FILL_B) void k_fill_geom(Params P, Ptrs X, PnGrid G, int tsel, int pos, Geom* dst,
                                                     GeomF* dstf) {
  __shared__ double sbuf[FILL_B * GEOM_DOUBLES];   // one staging buffer, FP64 or FP32 records
  const long long nt = P.nt;
  const long long z0 = (long long)blockIdx.x * FILL_B;
  const long long z = z0 + threadIdx.x;
  const long long nrec = (nt - z0 < FILL_B) ? nt - z0 : FILL_B;
  const int k = (int)(z % P.n3t);
  const int j = (int)((z / P.n3t) % P.n2t);
  const int i = (int)(z / ((long long)P.n3t * P.n2t));
  Geom g;
  if (z < nt && dst) pn_zone_geom(P, G, X.orbit[tsel], i, j, k, pos, &g);
  // records of position pos are contiguous: geom_id = pos * NT + zone index
  if (dst) {
    if (z < nt) {
      const double* gp = reinterpret_cast<const double*>(&g);
      for (int l = 0; l < GEOM_DOUBLES; l++) sbuf[threadIdx.x * GEOM_DOUBLES + l] = gp[l];
    }
    __syncthreads();
    double* out = reinterpret_cast<double*>(dst + (long long)pos * nt + z0);
    for (long long m = threadIdx.x; m < nrec * GEOM_DOUBLES; m += FILL_B) out[m] = sbuf[m];
    __syncthreads();
  }
  if (dstf) {
    float* sf = reinterpret_cast<float*>(sbuf);
    if (z < nt) {
      GeomF f;
      pn_zone_geomf(P, G, X.orbit[tsel], i, j, k, pos, &f);   // the FP32 face solve's own records
      const float* fp = reinterpret_cast<const float*>(&f);
      for (int l = 0; l < GEOMF_FLOATS; l++) sf[threadIdx.x * GEOMF_FLOATS + l] = fp[l];
    }
    __syncthreads();
    float* outf = reinterpret_cast<float*>(dstf + (long long)pos * nt + z0);
    for (long long m = threadIdx.x; m < nrec * GEOMF_FLOATS; m += FILL_B) outf[m] = sf[m];
  }
}

// Connection at the interior zone centres at time level tsel.
__global__ __launch_bounds__(BLOCK) void k_fill_conn(Params P, Ptrs X, PnGrid G, int tsel, double* dst) {
  const long long z = (long long)blockIdx.x * BLOCK + threadIdx.x;
  if (z >= (long long)P.n1 * P.n2 * P.n3) return;
  const int k = NG + (int)(z % P.n3);
  const int j = NG + (int)((z / P.n3) % P.n2);
  const int i = NG + (int)(z / ((long long)P.n3 * P.n2));
  double dg[PN_NDG];
  pn_zone_dg(P, G, X.orbit[tsel], i, j, k, dg);
  const long long cid = conn_id(P, i, j, k);
  for (int l = 0; l < PN_NDG; l++) dst[l * P.nconn + cid] = dg[l];   // structure-of-arrays levels
}

// Source terms of a stage on the binary metric evaluated in the kernels: the
// metric derivatives at the zone and the stage's level (as k_fill_conn) and
// the stage's zone record (as the update evaluates it), contracted with the
// stage's state at once as source() forms them (src/phys.c:121-187); the update reads
// the 4 terms (UU..U3, [4][nconn] in dst) instead of the 28 derivatives.
// Failures of get_state() are counted here (the update counts none for the
// source).
__global__ __launch_bounds__(BLOCK, 2) void k_source_otf(Params P, Ptrs X, PnGrid G, int stage, double* dst) {
  const long long z = (long long)blockIdx.x * BLOCK + threadIdx.x;
  const bool active = z < (long long)P.n1 * P.n2 * P.n3;
  FailRec fr; fr.clear();
  long long c = 0;
  if (active) {
    const int k = NG + (int)(z % P.n3);
    const int j = NG + (int)((z / P.n3) % P.n2);
    const int i = NG + (int)(z / ((long long)P.n3 * P.n2));
    const PnOrbit& o = X.orbit[stage];   // all of it: the derivatives read the time derivatives too
    c = cidx(P, i, j, k);
    // the state's part first (the zone record is then dead but for sqrt(-g)),
    // the metric derivatives last, so their evaluation holds few live values
    SrcDyn sd;
    double gdet;
    {
      Geom gs;
      pn_zone_geom(P, G, o, i, j, k, CENT, &gs);
      const double* src = (stage == 0) ? X.p : X.ph;
      double phz[NP];
#pragma unroll
      for (int v = 0; v < NP; v++) phz[v] = rt_val(P, X, v, i, src[v*P.nt + c]);
      source_dyn_state(P, X, phz, GeomView<GK_DIAG, const Geom*>{&gs}, i, sd);
      gdet = gs.g;
    }
    double dg[PN_NDG], dU[NP];
    pn_zone_dg(P, G, o, i, j, k, dg);
    source_dyn_finish(P, sd, dg, 1, gdet, dU);
    fr.nf[NFAIL_GAMMA_CALC] += sd.gfail;
    const long long cid = conn_id(P, i, j, k);
#pragma unroll
    for (int m = 0; m < 4; m++) dst[m*P.nconn + cid] = dU[UU + m];
  }
  commit_fail(P, X, fr, active, c, MASK_GAMMA);
}

// Batched Utoprim_2d_fast() on independent zones (SoA buffers).
__global__ __launch_bounds__(BLOCK) void k_con2prim(Params P, long long n, const double* __restrict__ U,
                                                   const Geom* __restrict__ geom, double* prim,
                                                   double* gamma, int* code, int* iters) {
  long long t = (long long)blockIdx.x * BLOCK + threadIdx.x;
  if (t >= n) return;
  double u[NP], pr[NP];
  for (int l = 0; l < NP; l++) { u[l] = U[l*n + t]; pr[l] = prim[l*n + t]; }
  double gm = 1., bsq = 0.;
  int it = 0;
  int ret = utoprim_2d_fast(u, &geom[t], P.gam, P.gam_m1_o_gam, pr, &gm, &bsq, &it);
  for (int l = 0; l < NP; l++) prim[l*n + t] = pr[l];
  gamma[t] = gm;
  code[t] = ret;
  if (iters) iters[t] = it;
}

// --------------------------------------------------------------------------
struct GpuBE {
  static int init(hgpu_ctx* c) {
    int ndev = 0;
    hipError_t e = hipGetDeviceCount(&ndev);
    if (e != hipSuccess || ndev < 1)
      return set_error(-5, "no HIP device available (the hgpu library runs only on a GPU)");
    GpuPriv* g = new GpuPriv();
    c->be = g;
    // Untuned defaults: the autotuner's picks on the 192x192x128 torus.  The
    // face fluxes run 2 faces per thread, FP64 in the kernels capped at 3
    // waves per SIMD, FP32 uncapped (3 waves) but along x2 (capped at 4); the
    // update is the fused kernel, register-capped (3 waves per SIMD; the
    // mixed-precision row-aligned variant 4).
    const bool mixed = c->P.mixed != 0;
    for (int f = FAM_FLUX1; f <= FAM_FLUX3; f++) {
      g->shape[f].fpt = 2;
      g->shape[f].occ = mixed ? 0u : 1u;
      g->shape[f].remap = 0;
      g->shape[f].all = 1;
    }
    // x2 stencils share rows with the neighbouring tiles: XCD-contiguous
    // tiles keep those in one L2 (half the HBM reads of round-robin tiles)
    g->shape[FAM_FLUX2].occ = 1;
    g->shape[FAM_FLUX2].remap = 1;
    g->shape[FAM_EMF].order = mixed ? 1u : 0u;
    g->shape[FAM_EMF].spread = g->shape[FAM_CONS].spread = 1;
    g->shape[FAM_CONS].fused = 1;
    g->shape[FAM_CONS].remap = 0;
    g->shape[FAM_CONS].occ = 1;
    // Kernels gated by a device flag (fixups, flag clears, the boundaries of
    // bounds(prim,1)) stride over their zones with 4 workgroups per CU: a
    // full grid of workgroups that find the flag clear costs several
    // microseconds just to dispatch.
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) == hipSuccess) {
      g->ring.device = dev;
      if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && cus > 0)
        g->flag_grid = g->simds = 4u * (unsigned)cus;
    }
    if (const char* n = std::getenv("HGPU_PINNED_CHUNKS"))
      g->ring.cap = std::max(0, std::min(std::atoi(n), XferRing::SLOTS));
    return hip_check(hipStreamCreateWithFlags(&g->stream, hipStreamNonBlocking), "hipStreamCreate");
  }
  static void fini(hgpu_ctx* c) {
    GpuPriv* g = priv(c);
    if (!g) return;
    if (g->stream) (void)hipStreamSynchronize(g->stream);
    if (g->step_exec) (void)hipGraphExecDestroy(g->step_exec);
    g->ring.release();
    if (g->box_stage) (void)hipFree(g->box_stage);
    if (g->stream) (void)hipStreamDestroy(g->stream);
    for (auto& pe : g->pending) { (void)hipEventDestroy(pe.a); (void)hipEventDestroy(pe.b); }
    for (auto ev : g->pool) (void)hipEventDestroy(ev);
    for (auto& kv : g->open) (void)hipEventDestroy(kv.second);
    delete g;
    c->be = nullptr;
  }
  static int alloc(hgpu_ctx*, void** p, size_t bytes) {
    *p = nullptr;
    if (bytes == 0) bytes = 8;
    return hip_check(hipMalloc(p, bytes), "hipMalloc");
  }
  static void release(hgpu_ctx*, void* p) { (void)hipFree(p); }
  static int h2d(hgpu_ctx* c, void* d, const void* h, size_t bytes) {
    return hip_check(hipMemcpyAsync(d, h, bytes, hipMemcpyHostToDevice, priv(c)->stream), "hipMemcpy H2D") |
           hip_check(hipStreamSynchronize(priv(c)->stream), "hipStreamSynchronize");
  }
  static int d2h(hgpu_ctx* c, void* h, const void* d, size_t bytes) {
    GpuPriv* g = priv(c);
    if (bytes >= 4 && bytes % 4 == 0 && reinterpret_cast<uintptr_t>(d) % 16 == 0) {
      const char* src = static_cast<const char*>(d);
      return hip_check(xfer_to_host(g->ring, g->stream, h, bytes, [&](size_t off, size_t len, char* chunk) {
        const long long n32 = (long long)(len / 4);
        const unsigned nb = (unsigned)std::min<long long>((n32 / 4 + XFER_B - 1) / XFER_B + 1, 512);
        hipLaunchKernelGGL(k_copy_words, dim3(nb), dim3(XFER_B), 0, g->stream,
                           reinterpret_cast<const unsigned*>(src + off), n32, reinterpret_cast<unsigned*>(chunk));
      }, [&]() { return plain_to_host(g->stream, h, d, bytes); }), "copy to host");
    }
    return hip_check(plain_to_host(g->stream, h, d, bytes), "copy to host");
  }
  // a state array S ([8][nt]) to or from the host's [nt][8]
  static int download_state(hgpu_ctx* c, double* h, const double* S, long long nt) {
    GpuPriv* g = priv(c);
    return hip_check(xfer_to_host(g->ring, g->stream, h, sizeof(double) * NP * nt, [&](size_t off, size_t len, char* chunk) {
      const long long z0 = (long long)(off / (sizeof(double) * NP)), nz = (long long)(len / (sizeof(double) * NP));
      hipLaunchKernelGGL(k_soa_to_aos, dim3((unsigned)((nz + XFER_B - 1) / XFER_B)), dim3(XFER_B), 0, g->stream, S, nt,
                         z0, nz, reinterpret_cast<double*>(chunk));
    }, [&]() { return plain_state_to_host(g->stream, h, S, nt, NP); }), "state to host");
  }
  static int upload_state(hgpu_ctx* c, double* S, const double* h, long long nt) {
    GpuPriv* g = priv(c);
    return hip_check(xfer_to_device(g->ring, g->stream, h, sizeof(double) * NP * nt, [&](size_t off, size_t len, const char* chunk) {
      const long long z0 = (long long)(off / (sizeof(double) * NP)), nz = (long long)(len / (sizeof(double) * NP));
      hipLaunchKernelGGL(k_aos_to_soa, dim3((unsigned)((nz + XFER_B - 1) / XFER_B)), dim3(XFER_B), 0, g->stream,
                         reinterpret_cast<const double*>(chunk), nt, z0, nz, S);
    }, [&]() { return plain_state_to_device(g->stream, S, h, nt, NP); }), "state to device");
  }
  // zero fill with a kernel (no memset nodes on the stream)
  static int zero(hgpu_ctx* c, void* p, size_t bytes) {
    if (bytes % 4) return set_error(-2, "zero(): size not a multiple of 4");
    long long n = (long long)(bytes / 4);
    long long nb = (n + BLOCK - 1) / BLOCK;
    if (nb > 0) hipLaunchKernelGGL(k_zero, dim3((unsigned)nb), dim3(BLOCK), 0, priv(c)->stream, (unsigned int*)p, n);
    return hip_check(hipGetLastError(), "k_zero");
  }
  static int sync(hgpu_ctx* c) { return hip_check(hipStreamSynchronize(priv(c)->stream), "hipStreamSynchronize"); }

  // profiling ---------------------------------------------------------------
  static hipEvent_t ev(GpuPriv* g) {
    if (!g->pool.empty()) { hipEvent_t e = g->pool.back(); g->pool.pop_back(); return e; }
    hipEvent_t e;
    (void)hipEventCreate(&e);
    return e;
  }
  struct Scope {
    GpuPriv* g; const char* name; hipEvent_t a = nullptr;
    Scope(hgpu_ctx* c, const char* n) : g(priv(c)), name(n) {
      if (g->prof) { a = ev(g); (void)hipEventRecord(a, g->stream); }
    }
    ~Scope() {
      if (g->prof) { hipEvent_t b = ev(g); (void)hipEventRecord(b, g->stream); g->pending.push_back({name, a, b}); }
    }
  };
  static int mark(hgpu_ctx* c, const char* name, int end) {
    GpuPriv* g = priv(c);
    if (!g->prof) return 0;
    if (!end) { hipEvent_t a = ev(g); (void)hipEventRecord(a, g->stream); g->open[name] = a; }
    else {
      auto it = g->open.find(name);
      if (it == g->open.end()) return 0;
      hipEvent_t b = ev(g);
      (void)hipEventRecord(b, g->stream);
      g->pending.push_back({name, it->second, b});
      g->open.erase(it);
    }
    return 0;
  }
  static int profile_enable(hgpu_ctx* c, int on) {
    GpuPriv* g = priv(c);
    int rc = sync(c);
    drain(g);
    g->acc.clear();
    g->prof = on != 0;
    return rc;
  }
  static void drain(GpuPriv* g) {
    for (auto& pe : g->pending) {
      float ms = 0.f;
      if (hipEventElapsedTime(&ms, pe.a, pe.b) == hipSuccess) {
        auto& a = g->acc[pe.name];
        a.first += ms;
        a.second += 1;
      }
      g->pool.push_back(pe.a);
      g->pool.push_back(pe.b);
    }
    g->pending.clear();
  }
  // Step replay from a captured graph.  Every launch of a step is enqueued on
  // the library stream with arguments fixed at context creation (state lives
  // in device memory), and the step path records no memset or copy nodes, so
  // one captured step_ch() replays any number of steps.  Kernel scopes are not
  // recorded inside the capture; "step" times whole replays.
  static int set_graph(hgpu_ctx* c, int on) {
    GpuPriv* g = priv(c);
    int rc = sync(c);
    g->graph = on != 0;
    return rc;
  }
  static bool graph_enabled(hgpu_ctx* c) { return priv(c)->graph; }
  static int invalidate_graph(hgpu_ctx* c) {
    GpuPriv* g = priv(c);
    int rc = 0;
    if (g->step_exec) {
      rc = sync(c);
      rc |= hip_check(hipGraphExecDestroy(g->step_exec), "hipGraphExecDestroy");
      g->step_exec = nullptr;
    }
    return rc;
  }
  template <class F>
  static int graph_steps(hgpu_ctx* c, int nsteps, F&& one_step) {
    GpuPriv* g = priv(c);
    if (!g->step_exec) {
      const bool prof = g->prof;
      g->prof = false;
      int rc = hip_check(hipStreamBeginCapture(g->stream, hipStreamCaptureModeThreadLocal), "hipStreamBeginCapture");
      if (rc) { g->prof = prof; return rc; }
      rc = one_step();
      hipGraph_t graph = nullptr;
      const int rc_end = hip_check(hipStreamEndCapture(g->stream, &graph), "hipStreamEndCapture");
      g->prof = prof;
      if (rc || rc_end) {
        if (graph) (void)hipGraphDestroy(graph);
        return rc ? rc : rc_end;
      }
      rc = hip_check(hipGraphInstantiate(&g->step_exec, graph, nullptr, nullptr, 0), "hipGraphInstantiate");
      (void)hipGraphDestroy(graph);
      if (rc) { g->step_exec = nullptr; return rc; }
    }
    int rc = 0;
    for (int s = 0; s < nsteps && !rc; s++) {
      rc |= mark(c, "step", 0);
      rc |= hip_check(hipGraphLaunch(g->step_exec, g->stream), "hipGraphLaunch");
      rc |= mark(c, "step", 1);
    }
    return rc;
  }

  // Launch-shape autotuner.  For each stencil family (flux in x1, x2, x3, EMF,
  // conserved update) every candidate shape -- workgroup size 64/128/256, flat
  // or kc x (bs/kc) tiles with kc in {16, 32, 64}, XCD remap on/off, plane-major
  // or x1-fastest tile order -- is timed
  // with HIP events over `reps` launches on the current state, and the fastest
  // kept.  These kernels write only face fluxes, EMFs and the conserved
  // scratch, which every substep recomputes before use; the failure words and
  // counters they also touch are saved before and restored after.  The
  // inversion keeps its own shape (it rewrites the state) unless set.
  static unsigned fpt_code(unsigned fpt) { return fpt == 4 ? 2u : (fpt == 2 ? 1u : 0u); }
  static unsigned shape_flags(const LaunchShape& L) {
    return L.remap | (L.order << 1) | (L.occ << 2) | (L.fused << 3) | (fpt_code(L.fpt) << 4) | (L.stage << 6) |
           (L.all << 7) | (L.spread << 8);
  }
  // the flags as a caller sees them: bit 7 only where the directions can share a launch
  static unsigned shown_flags(hgpu_ctx* c, int fam) {
    LaunchShape L = priv(c)->shape[fam];
    if (!flux_all_possible(c->P)) L.all = 0;
    return shape_flags(L);
  }
  static bool flux_in_one(hgpu_ctx* c) {
    const LaunchShape* s = priv(c)->shape;
    return s[FAM_FLUX1].all && s[FAM_FLUX2].all && s[FAM_FLUX3].all && flux_all_possible(c->P);
  }
  static int check_shape(const LaunchShape& L) {
    if (L.bs != 64 && L.bs != 128 && L.bs != 256) return set_error(-2, "workgroup size must be 64, 128 or 256");
    if (L.kc != 0 && (L.kc > L.bs || L.bs % L.kc != 0)) return set_error(-2, "tile k-extent must divide the workgroup size");
    if (L.remap > 1 || L.order > 1 || L.occ > 1 || L.fused > 1 || L.stage > 1)
      return set_error(-2, "remap, order, occ, fused and stage must be 0 or 1");
    if (L.stage && L.fpt == 1) return set_error(-2, "staged pencils need 2 or 4 faces per thread");
    if (L.fpt != 1 && L.fpt != 2 && L.fpt != 4) return set_error(-2, "faces per thread must be 1, 2 or 4");
    return 0;
  }
  static int set_shape(hgpu_ctx* c, int fam, int bs, int kc, int flags) {
    if (fam < 0 || fam >= N_FAM) return set_error(-2, "kernel family out of range");
    LaunchShape L;
    L.bs = (unsigned)bs; L.kc = (unsigned)kc; L.remap = (unsigned)flags & 1u; L.order = ((unsigned)flags >> 1) & 1u;
    L.occ = ((unsigned)flags >> 2) & 1u;
    L.fused = ((unsigned)flags >> 3) & 1u;
    const unsigned fcode = ((unsigned)flags >> 4) & 3u;
    L.fpt = 1u << fcode;
    L.stage = ((unsigned)flags >> 6) & 1u;
    L.all = ((unsigned)flags >> 7) & 1u;
    L.spread = ((unsigned)flags >> 8) & 1u;
    if (bs < 0 || kc < 0 || flags < 0 || flags > 511 || fcode > 2) return set_error(-2, "bad launch-shape field");
    if (L.stage && fam != FAM_FLUX3) return set_error(-2, "flag bit 6 (staged pencils) applies to the x3 face fluxes only");
    if (L.fused && fam != FAM_CONS) return set_error(-2, "flag bit 3 (fused update) applies to the conserved update only");
    if (L.fpt > 1 && fam > FAM_FLUX3) return set_error(-2, "flag bits 4-5 (faces per thread) apply to the face fluxes only");
    if (L.all && fam > FAM_FLUX3) return set_error(-2, "flag bit 7 (one launch over the directions) applies to the face fluxes only");
    if (L.spread && fam != FAM_EMF && fam != FAM_CONS) return set_error(-2, "flag bit 8 (small grids spread) applies to the EMFs and the conserved update only");
    if (int rc = check_shape(L)) return rc;
    int rc = invalidate_graph(c);
    priv(c)->shape[fam] = L;
    return rc;
  }
  static int get_shape(hgpu_ctx* c, int fam, int* bs, int* kc, int* remap) {
    if (fam < 0 || fam >= N_FAM) return set_error(-2, "kernel family out of range");
    const LaunchShape& L = priv(c)->shape[fam];
    if (bs) *bs = (int)L.bs;
    if (kc) *kc = (int)L.kc;
    if (remap) *remap = (int)shown_flags(c, fam);
    return 0;
  }
  static void launch_conserved(hgpu_ctx* c, const LaunchShape& L, const Tiling& T, const Box& b, const Ptrs& X,
                               int stage) {
    hipStream_t st = priv(c)->stream;
    const dim3 grid(T.nblocks), blk(T.bs);
    if (c->P.mixed) {
      if (L.occ) hipLaunchKernelGGL((k_conserved<true, 4>), grid, blk, 0, st, c->P, X, stage, b, T);
      else hipLaunchKernelGGL((k_conserved<true, 1>), grid, blk, 0, st, c->P, X, stage, b, T);
    } else {
      if (L.occ) hipLaunchKernelGGL((k_conserved<false, 4>), grid, blk, 0, st, c->P, X, stage, b, T);
      else hipLaunchKernelGGL((k_conserved<false, 1>), grid, blk, 0, st, c->P, X, stage, b, T);
    }
  }
  static void launch_fused(hgpu_ctx* c, const LaunchShape& L, const Tiling& T, const Box& b, int stage) {
    hipStream_t st = priv(c)->stream;
    const dim3 grid(T.nblocks), blk(T.bs);
    const PnGrid& G = c->pn;
    const int lvl = c->otf_stage;
    if (c->P.otf) {   // three waves per SIMD fit the FP32-face variant without spilling
      if (c->P.mixed) hipLaunchKernelGGL((k_update<true, 3, true, 1>), grid, blk, 0, st, c->P, c->X, stage, b, T, G, lvl);
      else hipLaunchKernelGGL((k_update<false, 1, true, 1>), grid, blk, 0, st, c->P, c->X, stage, b, T, G, lvl);
      return;
    }
    if (c->P.dyn) {
      if (c->P.mixed) hipLaunchKernelGGL((k_update<true, 1, false, 1>), grid, blk, 0, st, c->P, c->X, stage, b, T, G, lvl);
      else hipLaunchKernelGGL((k_update<false, 1, false, 1>), grid, blk, 0, st, c->P, c->X, stage, b, T, G, lvl);
      return;
    }
    // row-aligned flat tiles: every wavefront's 64 zones share one (i, j)
    const bool uni = c->P.metric_dim == 2 && !c->P.flat && T.kc == 0 && T.nk % 64 == 0 && T.bs % 64 == 0;
    // capped variants: 3 waves per SIMD; the mixed-precision row-aligned one 4
    // (some registers spilled), which on the 192x192x128 torus is within 1 % of 3
    // (0.824 and 0.821 ms a step)
    const auto go = [&](auto M, auto K) {
      constexpr bool m = decltype(M)::value;
      constexpr int k = decltype(K)::value;
      if constexpr (k != GK_FLAT) {
        if (uni) {
          if (L.occ) hipLaunchKernelGGL((k_update<m, m ? 4 : 3, false, 0, true, k>), grid, blk, 0, st, c->P, c->X, stage, b, T, G, lvl);
          else hipLaunchKernelGGL((k_update<m, 1, false, 0, true, k>), grid, blk, 0, st, c->P, c->X, stage, b, T, G, lvl);
          return;
        }
      }
      if (L.occ) hipLaunchKernelGGL((k_update<m, 3, false, 0, false, k>), grid, blk, 0, st, c->P, c->X, stage, b, T, G, lvl);
      else hipLaunchKernelGGL((k_update<m, 1, false, 0, false, k>), grid, blk, 0, st, c->P, c->X, stage, b, T, G, lvl);
    };
    const auto kind = [&](auto M) {
      if (c->P.gkind == GK_FLAT) go(M, std::integral_constant<int, GK_FLAT>());
      else if (c->P.gkind == GK_KS) go(M, std::integral_constant<int, GK_KS>());
      else go(M, std::integral_constant<int, GK_GEN>());
    };
    if (c->P.mixed) kind(std::true_type());
    else kind(std::false_type());
  }
  // The autotuner times the conserved-update family as the whole predictor
  // update (split pair or fused kernel), which writes only arrays that the
  // next step rewrites before reading (ph, U^n, gamma, the slow-zone queue).
  static int launch_family(hgpu_ctx* c, int fam) {
    if (fam <= FAM_FLUX3) return flux(c, c->X.p, fam - FAM_FLUX1);
    if (fam == FAM_EMF) return emf(c);
    return update(c, 0);
  }
  static int autotune(hgpu_ctx* c, int reps, double* report) {
    GpuPriv* g = priv(c);
    if (reps < 1) reps = 1;
    int rc = invalidate_graph(c);
    const long long NT = c->P.nt;
    const size_t st_bytes = sizeof(unsigned long long) * ST_WORDS;
    const size_t nf_bytes = c->P.track_nfail ? sizeof(int) * N_NFAIL * NT : 0;
    const size_t pf_bytes = sizeof(int) * NT;
    // the update candidates run the predictor, which writes ph and p_gamma:
    // both are saved and restored with the flags and counters
    const size_t gm_bytes = sizeof(double) * NT, ph_bytes = sizeof(double) * NP * NT;
    const size_t o_nf = st_bytes, o_pf = o_nf + nf_bytes, o_gm = o_pf + pf_bytes, o_ph = o_gm + gm_bytes;
    void* save = nullptr;
    rc |= alloc(c, &save, o_ph + ph_bytes);
    if (rc) return rc;
    char* sv = static_cast<char*>(save);
    hipStream_t st = g->stream;
    rc |= hip_check(hipMemcpyAsync(sv, c->X.status, st_bytes, hipMemcpyDeviceToDevice, st), "save");
    if (nf_bytes) rc |= hip_check(hipMemcpyAsync(sv + o_nf, c->X.nfail, nf_bytes, hipMemcpyDeviceToDevice, st), "save");
    rc |= hip_check(hipMemcpyAsync(sv + o_pf, c->X.pflag, pf_bytes, hipMemcpyDeviceToDevice, st), "save");
    rc |= hip_check(hipMemcpyAsync(sv + o_gm, c->X.gamma, gm_bytes, hipMemcpyDeviceToDevice, st), "save");
    rc |= hip_check(hipMemcpyAsync(sv + o_ph, c->X.ph, ph_bytes, hipMemcpyDeviceToDevice, st), "save");
    const bool prof = g->prof;
    g->prof = false;
    hipEvent_t e0 = ev(g), e1 = ev(g);
    const auto set_all = [&](const unsigned* all) { for (int d = 0; d < 3; d++) g->shape[FAM_FLUX1 + d].all = all[d]; };
    unsigned all_was[3];
    for (int d = 0; d < 3; d++) all_was[d] = g->shape[FAM_FLUX1 + d].all;
    // fluxes first, so the EMF and update candidates read current face values
    for (int d = 0; d < 3 && !rc; d++) rc |= flux(c, c->X.p, d);
    const unsigned bss[3] = {64, 128, 256}, kcs[4] = {0, 16, 32, 64};
    for (int fam = FAM_FLUX1; fam <= FAM_CONS && !rc; fam++) {
      LaunchShape incumbent = g->shape[fam];
      incumbent.all = 0;   // a launch per direction is timed here, against the one launch below
      LaunchShape best = incumbent;
      float best_ms = 1e30f;
      auto time_shape_n = [&](const LaunchShape& L, int n) -> float {
        g->shape[fam] = L;
        rc |= launch_family(c, fam);   // warm-up
        rc |= hip_check(hipEventRecord(e0, st), "hipEventRecord");
        for (int r = 0; r < n; r++) rc |= launch_family(c, fam);
        rc |= hip_check(hipEventRecord(e1, st), "hipEventRecord");
        rc |= hip_check(hipEventSynchronize(e1), "hipEventSynchronize");
        float ms = 0.f;
        rc |= hip_check(hipEventElapsedTime(&ms, e0, e1), "hipEventElapsedTime");
        return rc ? 1e30f : ms / (float)n;
      };
      auto time_shape = [&](const LaunchShape& L) -> float { return time_shape_n(L, reps); };
      const bool multi = fam <= FAM_FLUX3 && c->P.recon == RECON_PPM_MC && !c->P.degen[fam - FAM_FLUX1];
      const unsigned nfpt = multi ? 3u : 1u;
      // face groups: every group size with and without the register cap
      // (which size wins depends on the occupancy the cap buys)
      const unsigned nocc = multi ? 2u : 1u;
      for (unsigned fc = 0; fc < nfpt; fc++)
      for (unsigned oc = 0; oc < nocc; oc++)
      for (unsigned bs : bss) for (unsigned kc : kcs) for (unsigned flags = 0; flags < 4; flags++) {
        LaunchShape L;
        L.bs = bs; L.kc = kc; L.remap = flags & 1u; L.order = flags >> 1; L.fpt = 1u << fc;
        L.occ = (fc > 0) ? oc : 0u;
        L.spread = incumbent.spread;
        if (fc == 0 && oc == 1) continue;
        if (check_shape(L)) { g_last_error.clear(); continue; }
        const float ms = time_shape(L);
        if (rc) break;
        if (ms < best_ms) { best_ms = ms; best = L; }
      }
      if (multi && fam == FAM_FLUX3 && !c->P.mixed && !c->P.otf) {   // LDS-staged x3 pencils
        for (unsigned fc = 1; fc < nfpt && !rc; fc++)
        for (unsigned oc = 0; oc < 2; oc++)
        for (unsigned bs : bss) for (unsigned kc : kcs) for (unsigned flags = 0; flags < 4; flags++) {
          LaunchShape L;
          L.bs = bs; L.kc = kc; L.remap = flags & 1u; L.order = flags >> 1; L.fpt = 1u << fc;
          L.occ = oc; L.stage = 1;
          if (check_shape(L)) { g_last_error.clear(); continue; }
          const float ms = time_shape(L);
          if (rc) break;
          if (ms < best_ms) { best_ms = ms; best = L; }
        }
      }
      if (!rc && fam != FAM_EMF) {   // the register-capped variant of the best shape
        LaunchShape L = best;
        L.occ = 1;
        const float ms = time_shape(L);
        if (!rc && ms < best_ms) { best_ms = ms; best = L; }
      }
      if (!rc && fam == FAM_CONS) {  // the fused update over the same tile grid
        for (unsigned bs : bss) for (unsigned kc : kcs) for (unsigned flags = 0; flags < 4; flags++) {
          LaunchShape L;
          L.bs = bs; L.kc = kc; L.remap = flags & 1u; L.order = flags >> 1; L.fused = 1;
          L.spread = incumbent.spread;
          if (check_shape(L)) { g_last_error.clear(); continue; }
          const float ms = time_shape(L);
          if (rc) break;
          if (ms < best_ms) { best_ms = ms; best = L; }
        }
        if (!rc && best.fused) {
          LaunchShape L = best;
          L.occ = 1;
          const float ms = time_shape(L);
          if (!rc && ms < best_ms) { best_ms = ms; best = L; }
        }
      }
      // The winner of the sweep against the shape the family had, both timed
      // again, alternately, with more repetitions: a winner not 1 % faster
      // keeps the shape the family had (the sweep's single timings differ by
      // about that much from run to run).
      const bool moved = shape_flags(best) != shape_flags(incumbent) || best.bs != incumbent.bs ||
                         best.kc != incumbent.kc;
      if (!rc && moved) {
        float t_inc = 1e30f, t_best = 1e30f;
        for (int round = 0; round < 2 && !rc; round++) {
          t_inc = std::min(t_inc, time_shape_n(incumbent, 3 * reps));
          t_best = std::min(t_best, time_shape_n(best, 3 * reps));
        }
        if (!rc) {
          if (t_best < 0.99f * t_inc) best_ms = t_best;
          else { best = incumbent; best_ms = t_inc; }
        }
      }
      g->shape[fam] = best;
      if (report) {
        report[fam*4 + 0] = best.bs; report[fam*4 + 1] = best.kc;
        report[fam*4 + 2] = shape_flags(best);
        report[fam*4 + 3] = best_ms;
      }
    }
    // the face fluxes in one launch, or the tuned launch per direction
    if (!rc && flux_all_possible(c->P)) {
      float ms[2] = {1e30f, 1e30f};
      for (int round = 0; round < 2 && !rc; round++)
        for (int all = 0; all < 2; all++) {
          const unsigned on[3] = {(unsigned)all, (unsigned)all, (unsigned)all};
          set_all(on);
          rc |= flux_stage(c, c->X.p);
          rc |= hip_check(hipEventRecord(e0, st), "hipEventRecord");
          for (int r = 0; r < 3 * reps; r++) rc |= flux_stage(c, c->X.p);
          rc |= hip_check(hipEventRecord(e1, st), "hipEventRecord");
          rc |= hip_check(hipEventSynchronize(e1), "hipEventSynchronize");
          float t = 0.f;
          rc |= hip_check(hipEventElapsedTime(&t, e0, e1), "hipEventElapsedTime");
          ms[all] = std::min(ms[all], t);
        }
      for (unsigned& a : all_was) a = ms[1] < ms[0];
    }
    set_all(all_was);
    if (report)
      for (int fam = FAM_FLUX1; fam <= FAM_FLUX3; fam++) report[fam*4 + 2] = shown_flags(c, fam);
    g->pool.push_back(e0);
    g->pool.push_back(e1);
    g->prof = prof;
    rc |= hip_check(hipMemcpyAsync(c->X.status, sv, st_bytes, hipMemcpyDeviceToDevice, st), "restore");
    if (nf_bytes) rc |= hip_check(hipMemcpyAsync(c->X.nfail, sv + o_nf, nf_bytes, hipMemcpyDeviceToDevice, st), "restore");
    rc |= hip_check(hipMemcpyAsync(c->X.pflag, sv + o_pf, pf_bytes, hipMemcpyDeviceToDevice, st), "restore");
    rc |= hip_check(hipMemcpyAsync(c->X.gamma, sv + o_gm, gm_bytes, hipMemcpyDeviceToDevice, st), "restore");
    rc |= hip_check(hipMemcpyAsync(c->X.ph, sv + o_ph, ph_bytes, hipMemcpyDeviceToDevice, st), "restore");
    rc |= sync(c);
    release(c, save);
    return rc;
  }

  static int profile_read(hgpu_ctx* c, const char* name, double* ms, long long* cnt) {
    GpuPriv* g = priv(c);
    int rc = sync(c);
    drain(g);
    auto it = g->acc.find(name);
    if (ms) *ms = (it == g->acc.end()) ? 0. : it->second.first;
    if (cnt) *cnt = (it == g->acc.end()) ? 0 : it->second.second;
    return rc;
  }

  // launches ------------------------------------------------------------------
  static unsigned nblocks(long long n) { return (unsigned)((n + BLOCK - 1) / BLOCK); }

  static int reset_nfailtot(hgpu_ctx* c) {
    hipLaunchKernelGGL(k_reset_words, dim3(1), dim3(64), 0, priv(c)->stream, c->X, (int)ST_NFAILTOT, N_NFAIL);
    return hip_check(hipGetLastError(), "k_reset_words");
  }
  // every direction of a stage: one launch unless the caller or the autotuner
  // chose shapes per direction
  static int flux_stage(hgpu_ctx* c, const double* src) {
    GpuPriv* g = priv(c);
    if (flux_in_one(c)) {
      Scope s(c, "flux");
      launch_flux_all(c->P, c->X, src, g->stream, c->pn, c->otf_stage, g->simds);
      return hip_check(hipGetLastError(), "k_flux_all");
    }
    int rc = 0;
    for (int d = 0; d < 3; d++) rc |= flux(c, src, d);
    return rc;
  }
  static int flux(hgpu_ctx* c, const double* src, int d) {
    Scope s(c, "flux");
    launch_flux_dir(d, c->P, c->X, priv(c)->shape[FAM_FLUX1 + d], src, priv(c)->stream, c->pn, c->otf_stage);
    return hip_check(hipGetLastError(), "k_flux");
  }
  static int emf(hgpu_ctx* c) {
    Box b = edge_box(c->P);
    Scope s(c, "emf");
    const Tiling T = make_tiling(b, spread_shape(priv(c)->shape[FAM_EMF], b, b.count(), priv(c)->simds));
    if (c->P.mixed) hipLaunchKernelGGL(k_emf_mixed, dim3(T.nblocks + 1), dim3(T.bs), 0, priv(c)->stream, c->P, c->X, b, T);
    // The limiters' form: as long as the edges are one round of wavefronts (5 per
    // SIMD) the launch is one wavefront's chain, shorter by selects (24x24x16: 7.0
    // us against 8.6); from there on the issue of the sides that branches skip
    // counts (192x192x128: 137 us by branches, 143 by selects).
    else if (b.count() <= 64ll * 5 * priv(c)->simds) hipLaunchKernelGGL(k_emf<false>, dim3(T.nblocks + 1), dim3(T.bs), 0, priv(c)->stream, c->P, c->X, b, T);
    else hipLaunchKernelGGL(k_emf<true>, dim3(T.nblocks + 1), dim3(T.bs), 0, priv(c)->stream, c->P, c->X, b, T);
    return hip_check(hipGetLastError(), "k_emf");
  }
  // reset_slow: empty the slow-zone queue first (the stage's update finds it
  // emptied by begin_stage(); the autotuner's repeated updates do not)
  static int update(hgpu_ctx* c, int stage, bool reset_slow = true) {
    if (c->P.otf) {   // the stage's source terms, into the buffer the update reads (the stage's level)
      Scope sm(c, "metric");
      const long long n = (long long)c->P.n1 * c->P.n2 * c->P.n3;
      hipLaunchKernelGGL(k_source_otf, dim3(nblocks(n)), dim3(BLOCK), 0, priv(c)->stream, c->P, c->X, c->pn, stage,
                         const_cast<double*>(c->X.conn));
      int rc = hip_check(hipGetLastError(), "k_source_otf");
      if (rc) return rc;
    }
    Box b = interior_box(c->P);
    Scope s(c, "update");
    LaunchShape L = priv(c)->shape[FAM_CONS];
    if (L.fused || c->P.otf) L = spread_shape(L, b, b.count(), priv(c)->simds);
    const Tiling T = make_tiling(b, L);
    const Tiling T2 = make_tiling(b, priv(c)->shape[FAM_INV]);
    if ((long long)T.nblocks * (T.bs / 64) > c->mpart_cap) return set_error(-3, "update grid exceeds the M_tot parts buffer");
    if (reset_slow) hipLaunchKernelGGL(k_reset_words, dim3(1), dim3(64), 0, priv(c)->stream, c->X, (int)ST_SLOW, 1);
    hipStream_t st = priv(c)->stream;
    if (priv(c)->shape[FAM_CONS].fused || c->P.otf) {   // the evaluated metric has the fused kernel only
      launch_fused(c, priv(c)->shape[FAM_CONS], T, b, stage);
      return hip_check(hipGetLastError(), "k_update");
    }
    launch_conserved(c, priv(c)->shape[FAM_CONS], T, b, c->X, stage);
    Ptrs Xn = c->X;
    Xn.geom = c->X.geom_new;   // inversion at the result's time level
    hipLaunchKernelGGL(k_invert, dim3(T2.nblocks), dim3(T2.bs), 0, st, c->P, Xn, stage, b, T2);
    return hip_check(hipGetLastError(), "k_update");
  }
  static int recover_queued(hgpu_ctx* c, int stage) {
    Scope s(c, "recover");
    const long long nint = (long long)c->P.n1 * c->P.n2 * c->P.n3;
    const unsigned nb = (unsigned)std::min<long long>((nint + REC_Z - 1) / REC_Z, 1024);
    const auto go = [&](auto M, auto O) {
      hipLaunchKernelGGL((k_recover<decltype(M)::value, decltype(O)::value>), dim3(nb), dim3(REC_T), 0,
                         priv(c)->stream, c->P, c->X, stage, c->pn, stage);
    };
    typedef std::integral_constant<int, 0> Stored;
    typedef std::integral_constant<int, 1> Evaluated;
    if (c->P.mixed) { if (c->P.otf) go(std::true_type(), Evaluated()); else go(std::true_type(), Stored()); }
    else { if (c->P.otf) go(std::false_type(), Evaluated()); else go(std::false_type(), Stored()); }
    return hip_check(hipGetLastError(), "k_recover");
  }
  static int bounds(hgpu_ctx* c, double* S, int skip_mpi, bool mtot = false, bool tstep = false) {
    Scope s(c, "bounds");
    const long long n = ghost_count(c->P, 0) + ghost_count(c->P, 1) + ghost_count(c->P, 2);
    // bounds(prim,0) has work every time: one zone per thread; bounds(prim,1)
    // mostly finds its flag clear: a strided grid
    const unsigned nb = skip_mpi ? std::min(nblocks(n), priv(c)->flag_grid) : nblocks(n);
    if (c->P.otf)
      hipLaunchKernelGGL(k_bounds<1>, dim3(nb), dim3(BLOCK), 0, priv(c)->stream, c->P, c->X, S, skip_mpi, n, mtot, tstep);
    else
      hipLaunchKernelGGL(k_bounds<0>, dim3(nb), dim3(BLOCK), 0, priv(c)->stream, c->P, c->X, S, skip_mpi, n, mtot, tstep);
    return hip_check(hipGetLastError(), "k_bounds");
  }
  static int fixup_interp(hgpu_ctx* c, double* S) {
    Box b = interior_box(c->P);
    Scope s(c, "fixup");
    const unsigned nb = std::min(nblocks(b.count()), priv(c)->flag_grid);
    hipLaunchKernelGGL(k_fixup_interp, dim3(nb), dim3(BLOCK), 0, priv(c)->stream, c->P, c->X, S, b);
    return hip_check(hipGetLastError(), "k_fixup_interp");
  }
  static int set_boundary_flags(hgpu_ctx* c, int phys, int mpi) {
    hipLaunchKernelGGL(k_boundary_words, dim3(1), dim3(64), 0, priv(c)->stream, c->X, 1, phys, mpi);
    return hip_check(hipGetLastError(), "k_boundary_words");
  }
  static int set_vmax(hgpu_ctx* c, const double* vmax4) {
    unsigned long long w[4];
    for (int l = 0; l < 4; l++) w[l] = dbl_bits(vmax4[l]);
    return h2d(c, c->X.status + ST_VMAX, w, sizeof(w));
  }
  // a box of zones of S (and pflag) to (to_host) or from contiguous host
  // arrays [i][j][k][8] / [i][j][k], through a device staging buffer kept
  // between calls (grown when a larger box comes)
  static int box_copy(hgpu_ctx* c, double* S, const Box& b, double* prims, int* pflag, int to_host) {
    GpuPriv* g = priv(c);
    const long long n = b.count();
    const size_t need = (size_t)n * (NP * sizeof(double) + sizeof(int));
    int rc = 0;
    if (need > g->box_bytes) {
      rc |= sync(c);
      if (g->box_stage) (void)hipFree(g->box_stage);
      g->box_stage = nullptr;
      g->box_bytes = 0;
      rc |= hip_check(hipMalloc(&g->box_stage, need), "hipMalloc");
      if (rc) return rc;
      g->box_bytes = need;
    }
    double* ds = static_cast<double*>(g->box_stage);
    int* ps = reinterpret_cast<int*>(ds + n * NP);
    if (!to_host) {
      if (prims) rc |= h2d(c, ds, prims, sizeof(double) * NP * n);
      if (pflag) rc |= h2d(c, ps, pflag, sizeof(int) * n);
    }
    hipLaunchKernelGGL(k_box_copy, dim3(nblocks(n)), dim3(BLOCK), 0, g->stream, c->P, c->X, S, b,
                       prims ? ds : nullptr, pflag ? ps : nullptr, to_host);
    rc |= hip_check(hipGetLastError(), "k_box_copy");
    if (to_host) {
      if (prims) rc |= d2h(c, prims, ds, sizeof(double) * NP * n);
      if (pflag) rc |= d2h(c, pflag, ps, sizeof(int) * n);
    }
    return rc ? rc : sync(c);
  }
  // before each stage: flag map, failure words and boundary flags cleared,
  // fastest speeds reset, the slow-zone queue emptied
  static int begin_stage(hgpu_ctx* c) {
    hipLaunchKernelGGL(k_begin_stage, dim3(std::min(nblocks(c->P.nt), priv(c)->flag_grid)), dim3(BLOCK), 0,
                       priv(c)->stream, c->X, c->P.nt);
    return hip_check(hipGetLastError(), "k_begin_stage");
  }
  static int timestep(hgpu_ctx* c) {
    hipLaunchKernelGGL(k_timestep, dim3(1), dim3(64), 0, priv(c)->stream, c->P, c->X);
    return hip_check(hipGetLastError(), "k_timestep");
  }
  static int fixup_init(hgpu_ctx* c) {
    Box b = interior_box(c->P);
    hipLaunchKernelGGL(k_fixup_init, dim3(nblocks(b.count())), dim3(BLOCK), 0, priv(c)->stream, c->P, c->X, b);
    return hip_check(hipGetLastError(), "k_fixup_init");
  }
  static int divb_max(hgpu_ctx* c, double* out) {
    unsigned long long* d = nullptr;
    int rc = alloc(c, (void**)&d, 8);
    if (rc) return rc;
    rc |= zero(c, d, 8);
    Box b = divb_box(c->P);
    if (b.count() > 0)
      hipLaunchKernelGGL(k_divb, dim3(nblocks(b.count())), dim3(BLOCK), 0, priv(c)->stream, c->P, c->X, b, d);
    rc |= hip_check(hipGetLastError(), "k_divb");
    unsigned long long h = 0;
    rc |= d2h(c, &h, d, 8);
    release(c, d);
    *out = bits_dbl(h);
    return rc;
  }
  // positions in mask64 to dst (FP64), in mask32 to dstf (FP32)
  static int fill_geometry(hgpu_ctx* c, Geom* dst, GeomF* dstf, int tsel, unsigned mask64, unsigned mask32) {
    Scope s(c, "metric");
    const unsigned nb = (unsigned)((c->P.nt + FILL_B - 1) / FILL_B);
    int rc = 0;
    for (int pos = 0; pos < NPOS; pos++) {
      Geom* d64 = (mask64 >> pos) & 1u ? dst : nullptr;
      GeomF* d32 = ((mask32 >> pos) & 1u) && dstf ? dstf : nullptr;
      if (!d64 && !d32) continue;
      hipLaunchKernelGGL(k_fill_geom, dim3(nb), dim3(FILL_B), 0, priv(c)->stream, c->P, c->X, c->pn, tsel, pos, d64,
                         d32);
      rc |= hip_check(hipGetLastError(), "k_fill_geom");
    }
    return rc;
  }
  static constexpr bool HAS_METRIC_OTF = true;
  static int orbit(hgpu_ctx* c) {
    hipLaunchKernelGGL(k_orbit, dim3(1), dim3(64), 0, priv(c)->stream, c->X, c->pn.B, c->orbit);
    return hip_check(hipGetLastError(), "k_orbit");
  }
  static int fill_conn(hgpu_ctx* c, double* dst, int tsel) {
    Scope s(c, "metric");
    const long long n = (long long)c->P.n1 * c->P.n2 * c->P.n3;
    hipLaunchKernelGGL(k_fill_conn, dim3(nblocks(n)), dim3(BLOCK), 0, priv(c)->stream, c->P, c->X, c->pn, tsel, dst);
    return hip_check(hipGetLastError(), "k_fill_conn");
  }
  static int con2prim_batch(hgpu_ctx* c, long long n, const double* U, const double* geom, double* prim,
                            double* gamma, int* code, int* iters) {
    if (n == 0) return 0;
    Scope s(c, "con2prim");
    hipLaunchKernelGGL(k_con2prim, dim3(nblocks(n)), dim3(BLOCK), 0, priv(c)->stream, c->P, n, U,
                       reinterpret_cast<const Geom*>(geom), prim, gamma, code, iters);
    return hip_check(hipGetLastError(), "k_con2prim");
  }
};

}  // namespace hgpu

using BE = hgpu::GpuBE;
#include "hgpu_capi.inc"
