// pip_kernels.h -- HIP kernels of the fused two-fluid step for gfx950.
//
// Device layout (identical to the reference arrays, so uploads are memcpy):
// one buffer of NVT = nvar_m + 5 planes, plane n holding ix*jx doubles
// (x fastest); planes 0..nvar_m-1 are U_m, planes nvar_m.. are U_h.
//
// One launch of k_stage performs one SSP-RK stage for both fluids on a
// TX x TY tile of interior cells per workgroup:
//   load  : the TX x TY cells and the two-deep ring around them (no corners)
//           -> primitives in LDS (u2v_*, HLL_rot.f90:1136-1186)
//   x     : (TX+1)*TY faces: minmod MUSCL + HLLD, then minmod MUSCL + HLLC
//           (one fluid at a time, so the neutral face states are not live
//           while HLLD runs) -> flux tile in LDS
//   cell  : source_PIP + SSP blend + x flux divergence (Solver_rot.f90:464-478)
//   y     : TX*(TY+1) faces (permuted HLLD/HLLC) -> flux tile in LDS
//   cell  : y flux divergence, add_source, Dedner psi damping, then (last
//           stage of a fused step) the set_IR/cfl rewrite chain of main.f90
//           with the dt reduction, and the store of the cell and its ghost
//           images (Boundary_rot.f90:323-402 applied by index mapping).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "pip_bnd.h"
#include "pip_phys.h"
#include "pip_riemann.h"

namespace PIP_NS {

// Reduction slots (bit patterns of non-negative doubles; min/max as uint64).
enum { RED_DT = 0, RED_RHOAC = 1, RED_GMAX = 2, RED_IONPOT = 3, RED_NAN = 4, RED_N = 5 };

// The workgroups of a plain context's launch spread their reductions over up
// to kRedSlots sets of slots, one per 128-byte line (k_finalize combines
// them): atomics on one address complete one every ~9.5 ns here, so with a
// single set the stage that reduces waits for them (four atomics a workgroup
// bound stage 2 of 16x7 tiles: 360 us at 1024^2, 187 with 16 sets; 16x15
// tiles, half as many workgroups: 195 -> 185).  red_sets: one set per 16
// workgroups, whose atomics take 0.6 us (with one per 64, stage 2 of KH + IR
// 160^2, whose 230 workgroups end together, took 20.3 instead of 16.8 us);
// k_finalize pays 0.1 us a step for 16 sets.
constexpr int kRedSlots = 16;
PIP_HD int red_sets(long long workgroups) {
  int n = 1;
  while (n < kRedSlots && 16LL * n < workgroups) n *= 2;
  return n;
}
struct alignas(128) RedSlot {
  unsigned long long v[RED_N];
};
PIP_HD RedSlot red_slot_init();

struct DevScalars {
  double dt;        // dt of the current step (global dt)
  double time;
  double cmax;      // GLM ch (Scheme_rot.f90:205-211)
  double tend;
  double dt_out;    // last cfl result
  unsigned long long red[RED_N];
  long long nt;
  long long nmax;
  int active;       // 1 while time < tend and no stop condition
  int last;         // current step is the last one (skip the look-ahead rewrite)
  int status;       // stop_sim flags
  int ion_pot_valid;
  int pad[4];
};

// Stage kernel modes: a step of the time loop; a step of a frozen-dt replay
// ({dt, cmax} from StageArgs::dtc, always active, never the loop's last
// step, no dt reduction) that also writes the primitives of its input to
// Vout; a step of the time loop that writes them as well (the last segment of
// an adjoint's recording run).
enum { STAGE_PLAIN = 0, STAGE_REPLAY = 1, STAGE_SAVE = 2 };

// ---------------------------------------------------------------- step end
// What the end of a cfl (Scheme_rot.f90:183-213) and of a fused step needs
// besides the scalars and the reduction slots.  A recorded run also passes
// hist: at a step's end the next step's {dt, cmax} go to hist[2 hist_k],
// hist[2 hist_k + 1], as k_record_dt would write them.
struct FinArgs {
  DevScalars* sc;
  RedSlot* red;
  DevScalars* src;    // the step that ends
  RedSlot* src_red;
  int nred;
  int mode, into_global, flag_ir, flag_ir_type, flag_divb, pip_imp;
  double safety, dxyz_min, pip_imp_factor;
  double* hist;
  int hist_k;
};

// Boundary description: per side type (1 periodic, 2 mirror, 10 free) and
// sign masks (bit n set -> variable n flips sign), Boundary_rot.f90:239-320.
struct StageArgs {
  const double* Uin;  // stage input (stencil)
  const double* U0;   // state at run_solver entry (pointwise; may alias Uout)
  double* Uout;
  const double* ac;       // per-cell alpha_c or nullptr
  double* ac_out;         // set_collisional col_type >= 1: alpha_c of this stage (nullable)
  double* U0out;          // implicit collisions: updated stage base for the next stage (nullable)
  const double* arb_heat; // IR type 0
  double* ion_pot_out;    // nullable: ion_pot of this stage
  double* Vout;           // replay and saving kernels, nullable: primitives of Uin at the
                          // tile's cells and their ghost images
  const double* dtc;      // replay kernels: frozen {dt, cmax} of the replayed step
  DevScalars* sc;
  RedSlot* red;           // reduction slot sets, nred (a power of two) in use
  int nred;
  int fold;               // k_stage and k_stage_split, stage 1: apply the end of the step before (fin) first
  FinArgs fin;
  int ix, jx, nx, ny;
  long long N;            // plane stride ix*jx
  int istep, t_order, epi;  // epi: 0 none, 1 one cfl round, 2 two rounds + dt reduction
  int xcd_remap;          // 1: contiguous tile ranges per XCD
  double col;
  double gmin_safety;     // safety*min(dx,dy,dz)
  double dxyz_min;        // min(dx,dy,dz)
  double dx, dy;
  double db_clean;
  Phys ph;
  IRConst irc;
  Bnd bnd;
};

PIP_HD unsigned long long as_u64(double x) {
  union { double d; unsigned long long u; } c;
  c.d = x;
  return c.u;
}
PIP_HD double as_f64(unsigned long long x) {
  union { double d; unsigned long long u; } c;
  c.u = x;
  return c.d;
}

PIP_HD RedSlot red_slot_init() {
  RedSlot r;
  for (int k = 0; k < RED_N; k++) r.v[k] = 0ull;
  r.v[RED_DT] = as_u64(1.0e300);
  return r;
}

// The slot sets combined, by one wave: every lane gets the result.
struct RedVals {
  double rdt, rhoac, gmax, ratio;
  int nan;
};
__device__ __forceinline__ RedSlot load_slot(const RedSlot* red, int nred, int flag_ir) {
  const int lane = threadIdx.x & 63;
  RedSlot rs = red_slot_init();
  if (lane < nred) {
    rs.v[RED_DT] = red[lane].v[RED_DT];
    rs.v[RED_RHOAC] = red[lane].v[RED_RHOAC];
    rs.v[RED_NAN] = red[lane].v[RED_NAN];
    if (flag_ir >= 1) {
      rs.v[RED_GMAX] = red[lane].v[RED_GMAX];
      rs.v[RED_IONPOT] = red[lane].v[RED_IONPOT];
    }
  }
  return rs;
}
__device__ __forceinline__ RedVals combine_slots(RedSlot rs, int nred, int flag_ir) {
  auto lo = [](unsigned long long a, unsigned long long b) { return a < b ? a : b; };
  auto hi = [](unsigned long long a, unsigned long long b) { return a > b ? a : b; };
  for (int off = nred / 2; off > 0; off >>= 1) {  // as the slots' atomics would
    rs.v[RED_DT] = lo(rs.v[RED_DT], __shfl_xor(rs.v[RED_DT], off, 64));
    rs.v[RED_RHOAC] = hi(rs.v[RED_RHOAC], __shfl_xor(rs.v[RED_RHOAC], off, 64));
    if (flag_ir >= 1) {
      rs.v[RED_GMAX] = hi(rs.v[RED_GMAX], __shfl_xor(rs.v[RED_GMAX], off, 64));
      rs.v[RED_IONPOT] = hi(rs.v[RED_IONPOT], __shfl_xor(rs.v[RED_IONPOT], off, 64));
    }
  }
  auto first = [](unsigned long long x) {
    const unsigned l = __builtin_amdgcn_readfirstlane((unsigned)x), h = __builtin_amdgcn_readfirstlane((unsigned)(x >> 32));
    return as_f64(((unsigned long long)h << 32) | l);
  };
  return RedVals{first(rs.v[RED_DT]), first(rs.v[RED_RHOAC]), first(rs.v[RED_GMAX]), first(rs.v[RED_IONPOT]),
                 __builtin_amdgcn_ballot_w64(rs.v[RED_NAN] != 0ull) != 0ull ? 1 : 0};
}

// dt of a cfl from its reductions.
__device__ __forceinline__ double cfl_dt(const RedVals& v, int ion_pot_valid, const FinArgs& f) {
  double dttemp = dmin(10.0, v.rdt);
  // cfl_pn_col (Scheme_rot.f90:305-313)
  if (f.pip_imp == 1) dttemp = dmin(dttemp, f.pip_imp_factor / v.rhoac);
  else dttemp = dmin(dttemp, dmin(f.safety, 0.3) / v.rhoac);
  if (f.flag_ir >= 1) {
    dttemp = dmin(dttemp, dmin(f.safety, 0.1) / dmax(v.gmax, 1.0e-5));
    if (f.flag_ir_type == 0) {
      double mx = ion_pot_valid ? v.ratio : 0.0;
      dttemp = dmin(dttemp, f.safety / dmax(mx, 1.0e-5));
    }
  }
  return dttemp;
}

// The scalars a step's end reads and writes (DevScalars without its slots).
struct StepState {
  double dt, time, cmax, tend, dt_out;
  long long nt, nmax;
  int active, last, status, ion_pot_valid;
};
__device__ __forceinline__ StepState load_state(const DevScalars* p) {
  return StepState{p->dt, p->time, p->cmax, p->tend, p->dt_out, p->nt, p->nmax, p->active, p->last, p->status,
                   p->ion_pot_valid};
}
__device__ __forceinline__ void store_state(DevScalars* p, const StepState& s) {
  p->dt = s.dt;
  p->time = s.time;
  p->cmax = s.cmax;
  p->tend = s.tend;
  p->dt_out = s.dt_out;
  p->nt = s.nt;
  p->nmax = s.nmax;
  p->active = s.active;
  p->last = s.last;
  p->status = s.status;
  p->ion_pot_valid = s.ion_pot_valid;
}

__device__ __forceinline__ void record_dt(const StepState& s, double* hist, int k) {
  hist[2 * k] = s.active ? s.dt : 0.0;
  hist[2 * k + 1] = s.cmax;
}

// End of a running fused step: main.f90:58-62 (time += dt, stop_sim), then the
// next iteration's cfl(dt) and GLM speed and the activity flags.
__device__ __forceinline__ StepState step_end(StepState s, const RedVals& v, const FinArgs& f) {
  s.ion_pot_valid = 1;  // source_PIP ran in this step
  const double dttemp = cfl_dt(v, 1, f);
  s.dt_out = dttemp;
  const double dt_used = s.dt;
  s.time = s.time + dt_used;
  s.nt = s.nt + 1;
  int st = 0;
  if (dt_used <= 1.0e-12) st |= 1;
  if (v.nan) st |= 2;
  s.status = st;
  const bool more = (s.time < s.tend) && (s.nt < s.nmax) && (st == 0);
  s.active = more ? 1 : 0;
  if (more) {
    s.dt = dttemp;
    if (f.flag_divb >= 1) s.cmax = f.safety * f.dxyz_min / s.dt;
    s.last = ((s.time + s.dt >= s.tend) || (s.nt + 1 >= s.nmax) || (s.dt <= 1.0e-12)) ? 1 : 0;
  }
  return s;
}

// Store one cell value set (NVT vars) at (ci,cj) and at all its ghost images.
template <int NDIM, int NVT>
__device__ __forceinline__ void store_cell(double* U, long long N, int ix, int jx, int ci, int cj,
                                           const double* u, const Bnd& b) {
#pragma unroll
  for (int n = 0; n < NVT; n++) U[n * N + (long long)cj * ix + ci] = u[n];
  for_each_image(ci, cj, ix, (NDIM == 2) ? jx : 1, b, [&](int xi, int yj, unsigned m) {
    for (int n = 0; n < NVT; n++) U[n * N + (long long)yj * ix + xi] = ((m >> n) & 1u) ? -u[n] : u[n];
  });
}

// One round of the set_IR/cfl chain on one cell (main.f90:32-36 / :44-47):
// set_IR rewrites (+ rates), cfl rewrites and the cell's dt terms.
struct RoundOut {
  double dtc, rhoac, gmax, ratio;
};

template <int NV, bool IR>
__device__ __forceinline__ RoundOut cfl_round(double* um, double* uh, double ac, double ion_pot,
                                              const StageArgs& a) {
  RoundOut r;
  double gr = 0.0, gi = 0.0;
  if (IR) set_ir_cell<NV>(um, uh, a.ph, a.irc, gr, gi);
  r.dtc = cfl_cell<NV>(um, uh, a.gmin_safety, a.ph);
  r.rhoac = dmax(um[0] * ac, uh[0] * ac);
  r.gmax = dmax(gr, gi);
  r.ratio = 0.0;
  if (IR && a.ph.flag_ir_type == 0) {
    double pr, te;
    getpr_mhd(um, pr, te, a.ph);  // cfl_pip_ir :321
    r.ratio = qdiv(ion_pot, quo(pr, a.ph.gm - 1.0, a.ph.rgm1));
  }
  return r;
}

// The state rewrites of one round alone, for a round whose dt terms are not
// used (the first of the two rounds of a fused step): set_IR's get_Pr
// rewrites, cfl's cq2pv_mhd / cq2pv_hd and, for IR type 0, cfl_pip_ir's
// get_Pr_MHD, in the order cfl_round applies them.
template <int NV, bool IR>
__device__ __forceinline__ void cfl_rewrite(double* um, double* uh, const StageArgs& a) {
  if (IR) {
    double gr, gi;
    set_ir_cell<NV>(um, uh, a.ph, a.irc, gr, gi);
  }
  double pm[8], ph[5];
  cq2pv_mhd(um, pm, a.ph);
  cq2pv_hd(uh, ph, a.ph);
  if (IR && a.ph.flag_ir_type == 0) {
    double pr, te;
    getpr_mhd(um, pr, te, a.ph);
  }
}

// Workgroup min/max reduction of the dt terms into the slots `red`, one
// atomic per slot (IR: the rate and ion_pot slots too; they stay 0 without).
template <int NT, bool IR>
__device__ __forceinline__ void block_reduce_store(RoundOut r, int nanflag, bool valid, unsigned long long* red,
                                                   double* red_lds) {
  double v0 = valid ? r.dtc : 1.0e300;
  double v1 = valid ? r.rhoac : 0.0;
  double v2 = (IR && valid) ? r.gmax : 0.0;
  double v3 = (IR && valid) ? r.ratio : 0.0;
  int fl = valid ? nanflag : 0;
  for (int off = 32; off > 0; off >>= 1) {
    v0 = dmin(v0, __shfl_xor(v0, off, 64));
    v1 = dmax(v1, __shfl_xor(v1, off, 64));
    if (IR) {
      v2 = dmax(v2, __shfl_xor(v2, off, 64));
      v3 = dmax(v3, __shfl_xor(v3, off, 64));
    }
    fl |= __shfl_xor(fl, off, 64);
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  constexpr int NW = (NT + 63) / 64;
  __syncthreads();
  if (lane == 0) {
    red_lds[wid * 5 + 0] = v0;
    red_lds[wid * 5 + 1] = v1;
    if (IR) {
      red_lds[wid * 5 + 2] = v2;
      red_lds[wid * 5 + 3] = v3;
    }
    red_lds[wid * 5 + 4] = (double)fl;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < NW; w++) {
      v0 = dmin(v0, red_lds[w * 5 + 0]);
      v1 = dmax(v1, red_lds[w * 5 + 1]);
      if (IR) {
        v2 = dmax(v2, red_lds[w * 5 + 2]);
        v3 = dmax(v3, red_lds[w * 5 + 3]);
      }
      fl |= (int)red_lds[w * 5 + 4];
    }
    atomicMin(&red[RED_DT], as_u64(v0));
    atomicMax(&red[RED_RHOAC], as_u64(v1));
    if (IR) {
      atomicMax(&red[RED_GMAX], as_u64(v2));
      atomicMax(&red[RED_IONPOT], as_u64(v3));
    }
    if (fl) atomicOr(&red[RED_NAN], 1ull);
  }
}

// ------------------------------------------------------- start of a stage
// What a stage needs to know of its step.
struct StepNow {
  double dt, cmax;
  int epi;
  bool active;
};

// The scalars (and, with fold, slots) of a stage launch, loaded here and used
// in begin_step after the caller has issued its cells' loads.
template <bool REPLAY>
struct StepLoads {
  StepState st;
  RedSlot slot;
  __device__ __forceinline__ explicit StepLoads(const StageArgs& a) {
    if (REPLAY) return;
    st = load_state(a.fold ? a.fin.src : a.sc);
    if (a.fold) slot = load_slot(a.fin.src_red, a.nred, a.fin.flag_ir);
  }
  // The run is on (before the end of the step before: begin_step asks again).
  __device__ __forceinline__ bool running() const { return REPLAY || st.active != 0; }
  __device__ __forceinline__ StepNow begin_step(const StageArgs& a) {
    if (REPLAY) return StepNow{a.dtc[0], a.dtc[1], a.epi, true};
    if (a.fold) {
      // every workgroup works out the end of the step before; the first one
      // writes it where this step's later stages read it, with reset slots
      if (st.active) st = step_end(st, combine_slots(slot, a.nred, a.fin.flag_ir), a.fin);
      if (blockIdx.x == 0) {
        if ((int)threadIdx.x < a.nred) a.red[threadIdx.x] = red_slot_init();
        if (threadIdx.x == 0) {
          store_state(a.sc, st);
          if (a.fin.hist) record_dt(st, a.fin.hist, a.fin.hist_k);
        }
      }
    }
    return StepNow{st.dt, st.cmax, (a.epi >= 2 && st.last) ? 1 : a.epi, st.active != 0};
  }
};

// ------------------------------------------------------------ face fluxes
// Whether every cell of the tile is bounded (pip_riemann.h): the waves'
// answers side by side in shared memory, read by all after the barrier that
// follows the halo load.
template <int NT>
struct TileBounded {
  static constexpr int NW = (NT + 63) / 64;
  static __device__ __forceinline__ void post(int* slots, bool cells_bounded) {
    const bool any = wave_any(!cells_bounded);
    if ((threadIdx.x & 63) == 0) slots[threadIdx.x >> 6] = any ? 1 : 0;
  }
  static __device__ __forceinline__ bool read(const int* slots) {
    int u = 0;
#pragma unroll
    for (int w = 0; w < NW; w++) u |= slots[w];
    return __builtin_amdgcn_readfirstlane(u) == 0;
  }
};

// The flux of one fluid (FL 0: plasma, NV variables, HLLD with GLM; 1:
// neutrals, 5 variables, HLLC) through one face of the sweep in direction
// DIR: v points at the first of the stencil's four cells in the fluid's first
// plane, the cells ST apart, planes PV apart; the flux goes to f, planes PF
// apart.  y faces take the variables in the order (1,3,2,4,5,7,6,8,9) /
// (1,3,2,4,5) (HLL_rot.f90:414-434, 315-325).  Bounded tiles run
// hlld_flux_b / hllc_flux_b; the general functions take the faces these do
// not cover and the tiles that are not bounded.  Measured on faces of a smooth
// flow (1M faces, two 256-thread workgroups per CU): reconstruction 5.0 -> 4.0
// (with an fma for every half slope, see face_states), HLLD 20.6 -> 16.4, HLLC
// 11.9 -> 6.9 ps per face, the same values.
template <int FL, int NV, int DIR, int ST, int PV, int PF, bool BOUNDED = true>
__device__ __forceinline__ void face_flux(const double* v, double* f, const Phys& ph, double cmax, bool bounded) {
  constexpr int NFL = FL ? 5 : NV;
  auto perm = [](int n) {
    if (DIR == 0) return n;
    if (n == 1) return 2;
    if (n == 2) return 1;
    if (FL == 0 && n == 5) return 6;
    if (FL == 0 && n == 6) return 5;
    return n;
  };
  int done = 0;
  if (BOUNDED && bounded) {
    double vl[NFL], vr[NFL];
#pragma unroll
    for (int n = 0; n < NFL; n++) {
      const double* c = v + perm(n) * PV;
      if (n == 0 || n == 4) face_states<true>(c[0], c[ST], c[2 * ST], c[3 * ST], vl[n], vr[n]);
      else face_states(c[0], c[ST], c[2 * ST], c[3 * ST], vl[n], vr[n]);
    }
    vl[0] = dmax(vl[0], ph.ro_lim);
    vr[0] = dmax(vr[0], ph.ro_lim);
    auto put = [&](int n, double x) { f[perm(n) * PF] = x; };
    if constexpr (FL == 0) done = hlld_flux_b<NV>(vl, vr, ph.gm, ph.rgm1, cmax, put);
    else done = hllc_flux_b(vl, vr, ph.gm, ph.rgm1, put);
  }
  // Opaque, and nothing of the above kept in registers: otherwise the general
  // path is threaded into the solver's branches and the stencil stays live
  // across it (256 VGPRs and a spill instead of 239).
  if (BOUNDED) asm volatile("" : "+v"(done)::"memory");
  if (done) return;
  double vl[NFL], vr[NFL], fl[NFL];
#pragma unroll
  for (int n = 0; n < NFL; n++) {
    const double* c = v + perm(n) * PV;
    const double a0 = c[0], a1 = c[ST], a2 = c[2 * ST], a3 = c[3 * ST];
    vl[n] = a1 + 0.5 * minmod(a0, a1, a2);
    vr[n] = a2 - 0.5 * minmod(a1, a2, a3);
  }
  vl[0] = dmax(vl[0], ph.ro_lim);
  vr[0] = dmax(vr[0], ph.ro_lim);
  if constexpr (FL == 0) hlld_flux<NV>(vl, vr, ph.gm, cmax, fl);
  else hllc_flux(vl, vr, ph.gm, fl);
#pragma unroll
  for (int n = 0; n < NFL; n++) f[perm(n) * PF] = fl[n];
}

// ------------------------------------------------------------ stage tile
// LDS footprint of one tile (doubles): primitives (TX+4)x(TY+4) x NVT, then
// the face-flux tile NVT x max((TX+1)TY, TX(TY+1)).
template <int NDIM, int NV, int TX, int TY>
struct TileGeom {
  static constexpr int NVT = NV + 5;
  static constexpr int NCELL = TX * TY;
  static constexpr int HX = TX + 4;
  static constexpr int HY = (NDIM == 2) ? TY + 4 : 1;
  static constexpr int NFX = (TX + 1) * TY;
  static constexpr int NFY = (NDIM == 2) ? TX * (TY + 1) : 0;
  static constexpr int NF = (NFX > NFY) ? NFX : NFY;
  static constexpr int LDS_DOUBLES = NVT * HY * HX + NVT * NF;
};

// One SSP-RK stage on the tile of interior cells [i0,i0+TX) x [j0,j0+TY)
// (interior coordinates), executed by all NT threads of the workgroup.
// NT >= TX*TY; shapes with (TX+1)*TY <= NT and TX*(TY+1) <= NT compute every
// face phase in a single pass of the workgroup (e.g. 16x15 on 256 threads).
// Returns whether the calling thread owns a cell; r / nanflag receive the
// cell's dt terms when epi >= 1.
// step() is asked for the step's {dt, cmax, epi, active} once the cells' loads
// have been issued (its own loads then wait beside them); a tile of an inactive
// run ends there.  running false: it is known to be inactive, and nothing is
// loaded.
template <int NDIM, int NV, bool IR, bool EXT, int TX, int TY, int NT, int MODE = STAGE_PLAIN, bool BF = NDIM == 2,
          class Step>
__device__ __forceinline__ bool stage_tile(const StageArgs& a, Step step, int i0, int j0, double* smem, RoundOut& r,
                                           int& nanflag, bool running = true) {
  using G = TileGeom<NDIM, NV, TX, TY>;
  constexpr int NVT = G::NVT;
  constexpr int HX = G::HX;
  constexpr int HY = G::HY;
  constexpr int OY = (NDIM == 2) ? 2 : 0;
  constexpr int NFX = G::NFX;
  constexpr int NFY = G::NFY;
  constexpr int NF = G::NF;
  double* V = smem;                      // NVT * HY * HX
  double* F = smem + NVT * HY * HX;      // NVT * NF
  const int tid = threadIdx.x;
  const long long N = a.N;
  const int ix = a.ix;

  // ---- the tile's cells and the ring of halo cells its stencils reach (two
  // deep, no corners) -> primitives in LDS.  Each thread loads its own cell
  // and keeps it for the cell phase; the first NR threads also convert a ring
  // cell, whose loads are issued with the first ones.  The waves spend a third
  // of their cycles waiting, mostly on loads: against a loop over the (TX+4) x
  // (TY+4) cells with the own cell read again after the x faces, a step of
  // Orszag-Tang 1024^2 went from 349 to 330 us, of KH + IR 2048^2 from 1.53
  // to 1.49 ms (16x15 tiles: 364 instead of 380 cells in 6 instead of 7 waves).
  const int ti = tid % TX, tj = tid / TX;
  const int ci = i0 + ti + 2, cj = (NDIM == 2) ? j0 + tj + 2 : 0;
  const bool valid = (tid < TX * TY) && (i0 + ti < a.nx) && (j0 + tj < a.ny);
  const long long oc = (long long)cj * ix + ci;
  // 1-D tiles take the general fluxes: at the 168 registers of three
  // workgroups per CU the bounded ones spill, and few tiles are bound by their
  // latency (1024 cells: 5.63 against 5.44 ms for 256 steps),
  // unless they ask for them (k_lock_stage).
  __shared__ int unbounded[TileBounded<NT>::NW];
  bool cells_bounded = true;
  constexpr int NRX = (NDIM == 2) ? 4 * TX : 0;  // ring cells above and below
  constexpr int NR = NRX + 4 * TY;               // ... and at the sides
  // past the grid's edge a tile still needs the ghost cells there
  const bool inside = running && (tid < TX * TY) && ci < a.ix && cj < a.jx;
  // (in 2-D; 1-D tiles read it again, as the 26 registers across the solvers
  // would cost the third workgroup of a CU)
  constexpr bool KEEP = NDIM == 2;
  double raw[NVT];
  if (inside) {
#pragma unroll
    for (int n = 0; n < NVT; n++) raw[n] = a.Uin[n * N + oc];
  }
  static_assert(NR <= NT, "one pass over the ring");
  const int rk = (tid < NRX) ? tid / TX : (tid - NRX) % 4;
  const int rx = (tid < NRX) ? 2 + tid % TX : (rk < 2 ? rk : TX + rk);
  const int ry = (tid < NRX) ? (rk < 2 ? rk : TY + rk) : OY + (tid - NRX) / 4;
  const int gi = i0 + rx, gj = (NDIM == 2) ? j0 + ry : 0;
  const bool on_ring = running && tid < NR && gi < a.ix && gj < a.jx;
  double ring[NVT];
  if (on_ring) {
#pragma unroll
    for (int n = 0; n < NVT; n++) ring[n] = a.Uin[n * N + (long long)gj * ix + gi];
  }
  const StepNow now = step();
  if (!now.active) return false;
  const double dt = now.dt, cmax = now.cmax;
  const int epi = now.epi;
  double c0, c1, dt_sub;
  stage_coeffs(a.istep, a.t_order, dt, c0, c1, dt_sub);
  auto convert = [&](const double* u, int hx, int hy, double* v) {
    double um[NV], uh[5];
#pragma unroll
    for (int n = 0; n < NV; n++) um[n] = u[n];
#pragma unroll
    for (int n = 0; n < 5; n++) uh[n] = u[NV + n];
    if (EXT && col_type(a.ph) >= 1) {  // set_collisional's get_Te_* rewrite E (PIP_rot.f90:57-58)
      double pr, te;
      getpr_mhd(um, pr, te, a.ph);
      getpr_hd(uh, pr, te, a.ph);
    }
    if (IR) {  // set_IR of set_coefficients(.,1) rewrites E (Solver_rot.f90:111-113)
      double pr, te;
      getpr_hd(uh, pr, te, a.ph);
      getpr_mhd(um, pr, te, a.ph);
    }
    u2v_mhd<NV>(um, v, a.ph);
    u2v_hd(uh, v + NV, a.ph);
    if (BF) cells_bounded = cells_bounded & bounded_cell(v, NV) & bounded_cell(v + NV, 5);
#pragma unroll
    for (int n = 0; n < NVT; n++) V[(n * HY + hy) * HX + hx] = v[n];
  };
  if (on_ring) {
    double v[NVT];
    convert(ring, rx, ry, v);
  }
  if (inside) {
    double v[NVT];
    convert(raw, ti + 2, tj + OY, v);
    // the cell's primitives and their ghost images (u2v commutes with the
    // boundary sign maps: v = m / rho, the pressure takes squares)
    if (MODE != STAGE_PLAIN && a.Vout && valid) store_cell<NDIM, NVT>(a.Vout, N, ix, a.jx, ci, cj, v, a.bnd);
  }
  if (BF) TileBounded<NT>::post(unbounded, cells_bounded);
  __syncthreads();
  const bool bounded = BF && TileBounded<NT>::read(unbounded);

  // ---- x faces: face fi (0..TX) between tile cells fi-1 and fi
  for (int f = tid; f < NFX; f += NT) {
    int fi = f % (TX + 1), fj = f / (TX + 1);
    if (i0 + fi > a.nx || j0 + fj >= a.ny) continue;
    int hy = fj + OY;
    // one fluid at a time: the neutral face states are not live while the
    // plasma solver runs (same operations, fewer registers at its peak)
    face_flux<0, NV, 0, 1, HX * HY, NF, BF>(V + hy * HX + fi, F + f, a.ph, cmax, bounded);
    face_flux<1, NV, 0, 1, HX * HY, NF, BF>(V + NV * HX * HY + hy * HX + fi, F + NV * NF + f, a.ph, cmax, bounded);
  }
  __syncthreads();

  // ---- own cell: sources and x update
  double un[NVT];
  double Sm[5], Sh[5];
  double ion_pot = 0.0;
  double acc = a.col;
  if (valid) {
    double um[NV], uh[5];
#pragma unroll
    for (int n = 0; n < NV; n++) um[n] = KEEP ? raw[n] : a.Uin[n * N + oc];
#pragma unroll
    for (int n = 0; n < 5; n++) uh[n] = KEEP ? raw[NV + n] : a.Uin[(NV + n) * N + oc];
    if (a.ac) acc = a.ac[oc];
    if (EXT && col_type(a.ph) >= 1) {  // set_collisional (PIP_rot.f90:44-97), before set_IR
      acc = set_col_cell(um, uh, a.col, a.ph);
      if (a.ac_out) {
        a.ac_out[oc] = acc;
        for_each_image(ci, cj, ix, (NDIM == 2) ? a.jx : 1, a.bnd,
                       [&](int xi, int yj, unsigned) { a.ac_out[(long long)yj * ix + xi] = acc; });
      }
    }
    double gr = 0.0, gi = 0.0, arb = 0.0;
    if (IR) {
      set_ir_cell<NV>(um, uh, a.ph, a.irc, gr, gi);
      if (a.ph.flag_ir_type == 0) arb = a.arb_heat[oc];
    }
    // set_dt_coll (Solver_rot.f90:83-93): dt/2 per stage for t_order = 2
    const double dtc = (a.t_order == 2) ? dt * 0.5 : dt;
    double dU0[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    Phys phs = a.ph;
    if (!EXT) phs.pip_imp = 0;  // the default kernels carry no implicit branch
    source_pip(um, uh, acc, gr, gi, arb, phs, a.irc.heat_fac, Sh, Sm, ion_pot, dtc, dU0);
    if (a.ion_pot_out) a.ion_pot_out[oc] = ion_pot;
    const double ax = dt_sub / a.dx;
    const int fL = tj * (TX + 1) + ti;
#pragma unroll
    for (int n = 0; n < NVT; n++) {
      double u0 = a.U0[n * N + oc];
      if (EXT && a.ph.pip_imp == 1) {  // U_m0 += dt_c dS, U_h0 -= dt_c dS (PIP_rot.f90:1355-1356)
        if (n < 5) u0 = u0 + dU0[n];
        else if (n >= NV && n < NV + 5) u0 = u0 - dU0[n - NV];
        if (a.U0out) a.U0out[n * N + oc] = u0;
      }
      if (a.istep == 1) {
        un[n] = u0 - ax * (F[n * NF + fL + 1] - F[n * NF + fL]);
      } else {
        double ur = (n < NV) ? um[n] : uh[n - NV];
        un[n] = c0 * u0 + c1 * ur - ax * (F[n * NF + fL + 1] - F[n * NF + fL]);
      }
    }
  }

  // ---- y faces
  if (NDIM == 2) {
    __syncthreads();
    for (int f = tid; f < NFY; f += NT) {
      int fi = f % TX, fj = f / TX;
      if (i0 + fi >= a.nx || j0 + fj > a.ny) continue;
      const int o = fj * HX + fi + 2;
      face_flux<0, NV, 1, HX, HX * HY, NF>(V + o, F + f, a.ph, cmax, bounded);
      face_flux<1, NV, 1, HX, HX * HY, NF>(V + NV * HX * HY + o, F + NV * NF + f, a.ph, cmax, bounded);
    }
    __syncthreads();
    if (valid) {
      const double ay = dt_sub / a.dy;
      const int fB = tj * TX + ti;
#pragma unroll
      for (int n = 0; n < NVT; n++) un[n] = un[n] - ay * (F[n * NF + fB + TX] - F[n * NF + fB]);
    }
  }

  r = RoundOut{1.0e300, 0.0, 0.0, 0.0};
  nanflag = 0;
  if (valid) {
    // add_source (Solver_rot.f90:498-503) for the five fluid variables
#pragma unroll
    for (int n = 0; n < 5; n++) {
      un[n] = un[n] + Sm[n] * dt_sub;
      un[NV + n] = un[NV + n] + Sh[n] * dt_sub;
    }
    if (NV == 9) {  // divb_cleaning_Dedner_source (Scheme_rot.f90:546-554)
      double fac = pexp(-dt_sub / dt * a.ph.safety * a.db_clean);
      un[8] = un[8] * fac;
    }
    if (epi >= 1) {
      double* um = un;
      double* uh = un + NV;
      if (epi >= 2) cfl_rewrite<NV, IR>(um, uh, a);  // main.f90:44-47, its dt unused
      r = cfl_round<NV, IR>(um, uh, acc, ion_pot, a);
#pragma unroll
      for (int n = 0; n < NV; n++) nanflag |= !(un[n] * 0.0 == 0.0);
    }
    store_cell<NDIM, NVT>(a.Uout, N, ix, a.jx, ci, cj, un, a.bnd);
  }
  return valid;
}

// Workgroups are dealt round-robin to the 8 XCDs: tile of workgroup bid so that
// each XCD gets a contiguous range of the nb tiles, and neighbouring tiles
// (which share halo cells) meet in the same L2.
__device__ __forceinline__ int xcd_tile(int bid, int nb) {
  const int q = nb / 8, rr = nb % 8, x = bid % 8, k = bid / 8;
  return x * q + (x < rr ? x : rr) + k;
}

// ------------------------------------------------------------ stage kernel
// One workgroup per tile.  The look-ahead round of the fused step (epi=2)
// is skipped on the loop's last step (sc->last), as main.f90 ends there.
// 1-D tiles leave room for three workgroups per CU, 2-D tiles for two.
template <int NDIM, int NV, bool IR, bool EXT, int TX, int TY, int NT, int MODE>
__global__ void __launch_bounds__(NT, NDIM == 1 ? 3 : 2) k_stage(StageArgs a) {
  extern __shared__ double smem[];
  constexpr bool REPLAY = (MODE == STAGE_REPLAY);
  StepLoads<REPLAY> loads(a);
  // A run that has stopped leaves the chunk's other launches here.  The
  // arguments that the tile's loads need are asked for first, so that they
  // arrive with the flag: a return ahead of them cost a running step of 600^2
  // 1.5 % (a third wait in a row), this one 0.4 %.  us per step of a stopped
  // run, without and with it: Orszag-Tang 1024^2 52 / 9, KH + IR 2048^2 315 / 25
  // (their running steps 259 and 1293).  With fold the step's end is still to
  // be passed on; those tiles only skip their loads (300^2: 7.9 / 4.7).
  if (!REPLAY) {
    asm volatile("" ::"s"(a.Uin), "s"(a.N), "s"(a.ix), "s"(a.jx), "s"(a.nx), "s"(a.ny), "s"(a.xcd_remap),
                 "s"(gridDim.x));
    if (!a.fold && !loads.running()) return;
  }
  const int ntx = (a.nx + TX - 1) / TX;
  int bid = blockIdx.x;
  if (a.xcd_remap) bid = xcd_tile(bid, gridDim.x);
  const int i0 = (bid % ntx) * TX;
  const int j0 = (bid / ntx) * TY;
  RoundOut r;
  int nanflag;
  bool active = true;
  const bool valid = stage_tile<NDIM, NV, IR, EXT, TX, TY, NT, MODE>(
      a,
      [&] {
        const StepNow now = loads.begin_step(a);
        active = now.active;
        return now;
      },
      i0, j0, smem, r, nanflag, loads.running());
  if (!REPLAY && a.epi >= 1 && active) {
    __syncthreads();
    block_reduce_store<NT, IR>(r, nanflag, valid, a.red[blockIdx.x & (a.nred - 1)].v, smem);
  }
}

// ------------------------------------------------------ split stage tile
// The stage of stage_tile for grids that leave CUs idle, where a stage takes as
// long as one tile's chain of dependent operations: each tile spreads over eight
// waves (1-D: four), one workgroup per CU.  The waves split into jobs that run
// side by side: the plasma and the neutrals and, with DIRS, each one's x and y
// faces.  The x-face waves load, convert and update the tile's cells of their
// fluid, the y-face waves convert the ring (without DIRS one job does all of a
// fluid); the neutrals' waves, whose solver is the shorter, also form the
// sources while the plasma's faces run and hand its part over through shared
// memory.  Every value comes from the operations of stage_tile, in its order.
template <int NDIM, int NV, int TX, int TY, bool DIRS>
struct SplitGeom {
  static constexpr int NVT = NV + 5;
  static constexpr int NT = (NDIM == 2) ? 512 : 256;
  static constexpr int NB = DIRS ? NT / 4 : NT / 2;  // threads of a job
  static constexpr int HX = TX + 4;
  static constexpr int HY = (NDIM == 2) ? TY + 4 : 1;
  static constexpr int NC = TX * TY;
  static constexpr int NFX = (TX + 1) * TY;
  static constexpr int NFY = (NDIM == 2) ? TX * (TY + 1) : 0;
  static constexpr int NX = 17;  // handed from the neutrals to the plasma, per cell
  static constexpr int LDS_DOUBLES = NVT * (HX * HY + NFX + NFY) + NX * NC;
  static_assert(NFX <= NB && NFY <= NB && NC <= NB, "one pass per job");
};

// The planes of one fluid (NFL from plane OFF) of a cell and its ghost images.
template <int NDIM, int NFL, int OFF>
__device__ __forceinline__ void store_fluid(double* U, const StageArgs& a, int ci, int cj, const double* u) {
#pragma unroll
  for (int n = 0; n < NFL; n++) U[(OFF + n) * a.N + (long long)cj * a.ix + ci] = u[n];
  for_each_image(ci, cj, a.ix, (NDIM == 2) ? a.jx : 1, a.bnd, [&](int xi, int yj, unsigned m) {
    for (int n = 0; n < NFL; n++)
      U[(OFF + n) * a.N + (long long)yj * a.ix + xi] = ((m >> (OFF + n)) & 1u) ? -u[n] : u[n];
  });
}

template <int NDIM, int NV, bool IR, bool EXT, int TX, int TY, bool DIRS, int MODE>
__global__ void __launch_bounds__(NDIM == 2 ? 512 : 256, 2) k_stage_split(StageArgs a) {
  using G = SplitGeom<NDIM, NV, TX, TY, DIRS>;
  constexpr int NVT = G::NVT, NT = G::NT, NB = G::NB, HX = G::HX, HY = G::HY, NC = G::NC;
  constexpr int NFX = G::NFX, NFY = G::NFY, PV = HX * HY;
  constexpr int OY = (NDIM == 2) ? 2 : 0;
  constexpr bool REPLAY = (MODE == STAGE_REPLAY);
  extern __shared__ double smem[];
  double* V = smem;
  double* Fx = V + NVT * PV;
  double* Fy = Fx + NVT * NFX;
  double* X = Fy + NVT * NFY;  // Sm (5), um after its rewrites (5), ion_pot, alpha_c, dU0 (5)
  StepLoads<REPLAY> loads(a);
  const int ntx = (a.nx + TX - 1) / TX;
  const int bid = a.xcd_remap ? xcd_tile(blockIdx.x, gridDim.x) : (int)blockIdx.x;
  const int i0 = (bid % ntx) * TX, j0 = (bid / ntx) * TY;
  const long long N = a.N;
  const int ix = a.ix;
  const int job = __builtin_amdgcn_readfirstlane((int)threadIdx.x / NB), t = (int)threadIdx.x % NB;
  const int fluid = DIRS ? job >> 1 : job;  // 0 plasma, 1 neutrals
  const bool cells = !DIRS || (job & 1) == 0;
  const bool rest = !DIRS || (job & 1) == 1;  // the ring, the y faces
  const int ti = t % TX, tj = t / TX;
  const int ci = i0 + ti + 2, cj = (NDIM == 2) ? j0 + tj + 2 : 0;
  const long long oc = (long long)cj * ix + ci;
  const bool running = loads.running();
  const bool inside = running && cells && t < NC && ci < a.ix && cj < a.jx;
  const bool valid = running && cells && t < NC && i0 + ti < a.nx && j0 + tj < a.ny;

  // ---- load
  double own[NV], base[NV], other[NV];  // this fluid's cell, its stage base; for the neutrals the plasma's cell
  double ring[NV];
  constexpr int NRX = (NDIM == 2) ? 4 * TX : 0, NR = NRX + 4 * TY;
  static_assert(NR <= NB, "one pass over the ring");
  const int rk = (t < NRX) ? t / TX : (t - NRX) % 4;
  const int rx = (t < NRX) ? 2 + t % TX : (rk < 2 ? rk : TX + rk);
  const int ry = (t < NRX) ? (rk < 2 ? rk : TY + rk) : OY + (t - NRX) / 4;
  const int gi = i0 + rx, gj = (NDIM == 2) ? j0 + ry : 0;
  const bool on_ring = running && rest && t < NR && gi < a.ix && gj < a.jx;
  auto load = [&](auto fl) {
    constexpr int FL = decltype(fl)::value, NFL = FL ? 5 : NV, OFF = FL ? NV : 0;
    if (inside) {
#pragma unroll
      for (int n = 0; n < NFL; n++) own[n] = a.Uin[(OFF + n) * N + oc];
    }
    if (on_ring) {
#pragma unroll
      for (int n = 0; n < NFL; n++) ring[n] = a.Uin[(OFF + n) * N + (long long)gj * ix + gi];
    }
    if (valid) {
#pragma unroll
      for (int n = 0; n < NFL; n++) base[n] = a.U0[(OFF + n) * N + oc];
      if constexpr (FL == 1) {
#pragma unroll
        for (int n = 0; n < NV; n++) other[n] = a.Uin[n * N + oc];
      }
    }
  };
  if (fluid == 0) load(std::integral_constant<int, 0>{});
  else load(std::integral_constant<int, 1>{});

  const StepNow now = loads.begin_step(a);
  if (!now.active) return;
  const double dt = now.dt, cmax = now.cmax;
  const int epi = now.epi;
  double c0, c1, dt_sub;
  stage_coeffs(a.istep, a.t_order, dt, c0, c1, dt_sub);

  // ---- convert
  bool cells_bounded = true;
  auto convert = [&](auto fl) {
    constexpr int FL = decltype(fl)::value, NFL = FL ? 5 : NV, OFF = FL ? NV : 0;
    auto one = [&](const double* u0, int hx, int hy, double* v) {
      double u[NFL], pr, te;
#pragma unroll
      for (int n = 0; n < NFL; n++) u[n] = u0[n];
      for (int k = 0; k < 2; k++)  // set_collisional's, then set_IR's rewrite of E
        if ((k == 0 && EXT && col_type(a.ph) >= 1) || (k == 1 && IR)) {
          if constexpr (FL == 0) getpr_mhd(u, pr, te, a.ph);
          else getpr_hd(u, pr, te, a.ph);
        }
      if constexpr (FL == 0) u2v_mhd<NV>(u, v, a.ph);
      else u2v_hd(u, v, a.ph);
      cells_bounded = cells_bounded & bounded_cell(v, NFL);
#pragma unroll
      for (int n = 0; n < NFL; n++) V[(OFF + n) * PV + hy * HX + hx] = v[n];
    };
    double v[NFL];
    if (on_ring) one(ring, rx, ry, v);
    if (inside) {
      one(own, ti + 2, tj + OY, v);
      if (MODE != STAGE_PLAIN && a.Vout && valid) store_fluid<NDIM, NFL, OFF>(a.Vout, a, ci, cj, v);
    }
  };
  if (fluid == 0) convert(std::integral_constant<int, 0>{});
  else convert(std::integral_constant<int, 1>{});
  __shared__ int unbounded[TileBounded<NT>::NW];
  TileBounded<NT>::post(unbounded, cells_bounded);
  __syncthreads();
  const bool bounded = TileBounded<NT>::read(unbounded);

  // ---- faces
  const int xi = t % (TX + 1), xj = t / (TX + 1);
  const bool xface = t < NFX && i0 + xi <= a.nx && j0 + xj < a.ny;
  const bool yface = t < NFY && i0 + ti < a.nx && j0 + tj <= a.ny;
  const double* vx = V + (xj + OY) * HX + xi;
  const double* vy = V + tj * HX + ti + 2;
  double acc = a.col, ion_pot = 0.0, S[5], dU0[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  constexpr int PFY = (NDIM == 2) ? NFY : 1;
  if (fluid == 0) {
    if (cells && xface) face_flux<0, NV, 0, 1, PV, NFX>(vx, Fx + t, a.ph, cmax, bounded);
    if (NDIM == 2 && rest && yface) face_flux<0, NV, 1, HX, PV, PFY>(vy, Fy + t, a.ph, cmax, bounded);
  } else {
    if (cells && xface) face_flux<1, NV, 0, 1, PV, NFX>(vx + NV * PV, Fx + NV * NFX + t, a.ph, cmax, bounded);
    if (NDIM == 2 && rest && yface)
      face_flux<1, NV, 1, HX, PV, PFY>(vy + NV * PV, Fy + NV * NFY + t, a.ph, cmax, bounded);
    if (valid) {  // sources, as in stage_tile's cell phase
      if (a.ac) acc = a.ac[oc];
      if (EXT && col_type(a.ph) >= 1) {
        acc = set_col_cell(other, own, a.col, a.ph);
        if (a.ac_out) {
          a.ac_out[oc] = acc;
          for_each_image(ci, cj, ix, (NDIM == 2) ? a.jx : 1, a.bnd,
                         [&](int gx, int gy, unsigned) { a.ac_out[(long long)gy * ix + gx] = acc; });
        }
      }
      double gr = 0.0, gi = 0.0, arb = 0.0;
      if (IR) {
        set_ir_cell<NV>(other, own, a.ph, a.irc, gr, gi);
        if (a.ph.flag_ir_type == 0) arb = a.arb_heat[oc];
      }
      const double dtc = (a.t_order == 2) ? dt * 0.5 : dt;
      Phys phs = a.ph;
      if (!EXT) phs.pip_imp = 0;
      double Sm[5];
      source_pip(other, own, acc, gr, gi, arb, phs, a.irc.heat_fac, S, Sm, ion_pot, dtc, dU0);
      if (a.ion_pot_out) a.ion_pot_out[oc] = ion_pot;
#pragma unroll
      for (int n = 0; n < 5; n++) {
        X[n * NC + t] = Sm[n];
        X[(5 + n) * NC + t] = other[n];
        if (EXT) X[(12 + n) * NC + t] = dU0[n];
      }
      X[10 * NC + t] = ion_pot;
      X[11 * NC + t] = acc;
    }
  }
  __syncthreads();

  // ---- cells
  RoundOut r = {1.0e300, 0.0, 0.0, 0.0};
  int nanflag = 0;
  auto update = [&](auto fl) {
    constexpr int FL = decltype(fl)::value, NFL = FL ? 5 : NV, OFF = FL ? NV : 0;
    const bool imp = EXT && a.ph.pip_imp == 1;
    if constexpr (FL == 0) {
#pragma unroll
      for (int n = 0; n < 5; n++) {
        S[n] = X[n * NC + t];
        if (EXT) dU0[n] = X[(12 + n) * NC + t];
        own[n] = X[(5 + n) * NC + t];
      }
      ion_pot = X[10 * NC + t];
      acc = X[11 * NC + t];
    }
    const double ax = dt_sub / a.dx, ay = (NDIM == 2) ? dt_sub / a.dy : 0.0;
    const double* fx = Fx + OFF * NFX + tj * (TX + 1) + ti;
    const double* fy = Fy + OFF * NFY + t;
    double un[NFL];
#pragma unroll
    for (int n = 0; n < NFL; n++) {
      double u0 = base[n];
      if (imp) {
        if (n < 5) u0 = FL ? u0 - dU0[n] : u0 + dU0[n];
        if (a.U0out) a.U0out[(OFF + n) * N + oc] = u0;
      }
      const double dx = ax * (fx[n * NFX + 1] - fx[n * NFX]);
      un[n] = (a.istep == 1) ? u0 - dx : c0 * u0 + c1 * own[n] - dx;
      if (NDIM == 2) un[n] = un[n] - ay * (fy[n * NFY + TX] - fy[n * NFY]);
      if (n < 5) un[n] = un[n] + S[n] * dt_sub;
    }
    if constexpr (FL == 0 && NV == 9) un[8] = un[8] * pexp(-dt_sub / dt * a.ph.safety * a.db_clean);
    if (epi >= 1) {  // cfl_rewrite and cfl_round of this fluid
      double pv[8], pr, te;
      if constexpr (FL == 0) {
        if (epi >= 2) {
          if (IR) getpr_mhd(un, pr, te, a.ph);
          cq2pv_mhd(un, pv, a.ph);
          if (IR && a.ph.flag_ir_type == 0) getpr_mhd(un, pr, te, a.ph);
        }
        if (IR) {
          double gr, gi;
          getpr_mhd(un, pr, te, a.ph);
          ir_rates(un[0], te, a.ph, a.irc, gr, gi);
          r.gmax = dmax(gr, gi);
        }
        r.dtc = cfl_cell_mhd(un, a.gmin_safety, a.ph);
        r.rhoac = un[0] * acc;
        if (IR && a.ph.flag_ir_type == 0) {
          getpr_mhd(un, pr, te, a.ph);
          r.ratio = qdiv(ion_pot, quo(pr, a.ph.gm - 1.0, a.ph.rgm1));
        }
#pragma unroll
        for (int n = 0; n < NV; n++) nanflag |= !(un[n] * 0.0 == 0.0);
      } else {
        if (epi >= 2) {
          if (IR) getpr_hd(un, pr, te, a.ph);
          cq2pv_hd(un, pv, a.ph);
        }
        if (IR) getpr_hd(un, pr, te, a.ph);
        r.dtc = cfl_cell_hd(un, a.gmin_safety, a.ph);
        r.rhoac = un[0] * acc;
      }
    }
    store_fluid<NDIM, NFL, OFF>(a.Uout, a, ci, cj, un);
  };
  if (valid) {
    if (fluid == 0) update(std::integral_constant<int, 0>{});
    else update(std::integral_constant<int, 1>{});
  }
  if (!REPLAY && a.epi >= 1) {
    __syncthreads();
    block_reduce_store<NT, IR>(r, nanflag, valid, a.red[blockIdx.x & (a.nred - 1)].v, smem);
  }
}

// ------------------------------------------------ two-pass stage tile
// The stage of stage_tile for the explicit-collision configuration without
// ionisation/recombination (2-D), one fluid at a time: the plasma's
// primitives and fluxes (NV planes), then the neutrals' (5 planes), in one
// LDS tile of NV planes.  The tile (46 KB at 16x15, against 71 KB for all
// 14 planes) and the register set of one flux function at a time let three
// 256-thread workgroups share a CU.  Every value is computed by the same
// operations as in stage_tile, so the two kernels agree bit for bit.
template <int NV, int TX, int TY>
struct TileGeom2 {
  static constexpr int HX = TX + 4;
  static constexpr int HY = TY + 4;
  static constexpr int NFX = (TX + 1) * TY;
  static constexpr int NFY = TX * (TY + 1);
  static constexpr int NF = (NFX > NFY) ? NFX : NFY;
  static constexpr int LDS_DOUBLES = NV * HY * HX + NV * NF;
};

// One fluid (FL 0: plasma, NV variables from plane 0, HLLD with GLM; FL 1:
// neutrals, 5 variables from plane NV, HLLC) over the tile: halo ->
// primitives, x faces, the SSP blend with the x divergence, y faces, the y
// divergence.  un receives the fluid's part of the updated cell.  The
// plasma's partial cell value waits out the y faces in the cell's own
// output entries (read back by the same thread; in place, the stage base
// there was read first) rather than in registers next to HLLD's.
template <int FL, int NV, bool IR, int TX, int TY, int NT, int MODE>
__device__ __forceinline__ void fluid_pass(const StageArgs& a, double cmax, double c0, double c1,
                                           double dt_sub, int i0, int j0, double* smem, bool valid,
                                           long long oc, int ti, int tj, double* un) {
  constexpr int NFL = FL ? 5 : NV;  // variables of this fluid
  constexpr int OFF = FL ? NV : 0;  // its first plane
  using G = TileGeom2<NV, TX, TY>;
  constexpr int HX = G::HX, HY = G::HY, NFX = G::NFX, NFY = G::NFY, NF = G::NF;
  double* V = smem;
  double* F = smem + NV * HY * HX;
  const int tid = threadIdx.x;
  const long long N = a.N;
  const int ix = a.ix;

  // ---- halo -> primitives (u2v_mhd / u2v_hd act on one fluid each)
  for (int c = tid; c < HX * HY; c += NT) {
    int hx = c % HX, hy = c / HX;
    int gi = i0 + hx, gj = j0 + hy;
    if (gi < a.ix && gj < a.jx) {
      long long o = (long long)gj * ix + gi;
      double u[NFL], v[NFL];
#pragma unroll
      for (int n = 0; n < NFL; n++) u[n] = a.Uin[(OFF + n) * N + o];
      if (IR) {  // set_IR of set_coefficients(.,1) rewrites E (Solver_rot.f90:111-113), per fluid
        double pr, te;
        if (FL == 0) getpr_mhd(u, pr, te, a.ph);
        else getpr_hd(u, pr, te, a.ph);
      }
      if (FL == 0) u2v_mhd<NV>(u, v, a.ph);
      else u2v_hd(u, v, a.ph);
#pragma unroll
      for (int n = 0; n < NFL; n++) V[(n * HY + hy) * HX + hx] = v[n];
      if (MODE != STAGE_PLAIN && a.Vout && hx >= 2 && hx < TX + 2 && gi < a.nx + 2 && hy >= 2 && hy < TY + 2 &&
          gj < a.ny + 2) {
        // a cell of this tile: its primitives and their ghost images
#pragma unroll
        for (int n = 0; n < NFL; n++) a.Vout[(OFF + n) * N + o] = v[n];
        for_each_image(gi, gj, ix, a.jx, a.bnd, [&](int xi, int yj, unsigned m) {
          for (int n = 0; n < NFL; n++)
            a.Vout[(OFF + n) * N + (long long)yj * ix + xi] = ((m >> (OFF + n)) & 1u) ? -v[n] : v[n];
        });
      }
    }
  }
  __syncthreads();

  // ---- x faces (the general fluxes: the bounded ones spill 108 B/lane at 168
  // registers and measured 10 % slower)
  for (int f = tid; f < NFX; f += NT) {
    int fi = f % (TX + 1), fj = f / (TX + 1);
    if (i0 + fi > a.nx || j0 + fj >= a.ny) continue;
    face_flux<FL, NV, 0, 1, HX * HY, NF, false>(V + (fj + 2) * HX + fi, F + f, a.ph, cmax, false);
  }
  __syncthreads();

  // ---- the SSP blend and the x divergence; the blend takes the stage
  // input after set_IR's get_Pr rewrite (with IR) and source_PIP's cq2pv
  // rewrite of this fluid (PIP_rot.f90:1328)
  if (valid) {
    double u[NFL], pv[8];
#pragma unroll
    for (int n = 0; n < NFL; n++) u[n] = a.Uin[(OFF + n) * N + oc];
    if (IR) {
      double pr, te;
      if (FL == 0) getpr_mhd(u, pr, te, a.ph);
      else getpr_hd(u, pr, te, a.ph);
    }
    if (FL == 0) cq2pv_mhd(u, pv, a.ph);
    else cq2pv_hd(u, pv, a.ph);
    const double ax = dt_sub / a.dx;
    const int fL = tj * (TX + 1) + ti;
#pragma unroll
    for (int n = 0; n < NFL; n++) {
      const double u0 = a.U0[(OFF + n) * N + oc];
      double x;
      if (a.istep == 1) x = u0 - ax * (F[n * NF + fL + 1] - F[n * NF + fL]);
      else x = c0 * u0 + c1 * u[n] - ax * (F[n * NF + fL + 1] - F[n * NF + fL]);
      if (FL == 0) a.Uout[(OFF + n) * N + oc] = x;
      else un[n] = x;
    }
  }
  __syncthreads();

  // ---- y faces
  for (int f = tid; f < NFY; f += NT) {
    int fi = f % TX, fj = f / TX;
    if (i0 + fi >= a.nx || j0 + fj > a.ny) continue;
    face_flux<FL, NV, 1, HX, HX * HY, NF, false>(V + fj * HX + fi + 2, F + f, a.ph, cmax, false);
  }
  __syncthreads();
  if (valid) {
    const double ay = dt_sub / a.dy;
    const int fB = tj * TX + ti;
#pragma unroll
    for (int n = 0; n < NFL; n++) {
      const double x = (FL == 0) ? a.Uout[(OFF + n) * N + oc] : un[n];
      un[n] = x - ay * (F[n * NF + fB + TX] - F[n * NF + fB]);
    }
  }
}

template <int NV, bool IR, int TX, int TY, int NT, int MODE>
__global__ void __launch_bounds__(NT, 3) k_stage2p(StageArgs a) {
  extern __shared__ double smem[];
  constexpr int NVT = NV + 5;
  DevScalars* sc = a.sc;
  constexpr bool REPLAY = (MODE == STAGE_REPLAY);
  if (!REPLAY && !sc->active) return;
  const double dt = REPLAY ? a.dtc[0] : sc->dt;
  const double cmax = REPLAY ? a.dtc[1] : sc->cmax;
  const int epi = (!REPLAY && a.epi >= 2 && sc->last) ? 1 : a.epi;
  const int ntx = (a.nx + TX - 1) / TX;
  int bid = blockIdx.x;
  if (a.xcd_remap) bid = xcd_tile(bid, gridDim.x);
  const int i0 = (bid % ntx) * TX;
  const int j0 = (bid / ntx) * TY;
  double c0, c1, dt_sub;
  stage_coeffs(a.istep, a.t_order, dt, c0, c1, dt_sub);
  const int tid = threadIdx.x;
  const int ti = tid % TX, tj = tid / TX;
  const int ci = i0 + ti + 2, cj = j0 + tj + 2;
  const bool valid = (tid < TX * TY) && (i0 + ti < a.nx) && (j0 + tj < a.ny);
  const long long N = a.N;
  const long long oc = (long long)cj * a.ix + ci;
  double un[NVT];
  fluid_pass<0, NV, IR, TX, TY, NT, MODE>(a, cmax, c0, c1, dt_sub, i0, j0, smem, valid, oc, ti, tj, un);
  __syncthreads();  // the neutral pass reuses the tile
  fluid_pass<1, NV, IR, TX, TY, NT, MODE>(a, cmax, c0, c1, dt_sub, i0, j0, smem, valid, oc, ti, tj, un + NV);

  RoundOut r = {1.0e300, 0.0, 0.0, 0.0};
  int nanflag = 0;
  if (valid) {
    // source_PIP on the stage input (it rewrites its copy through cq2pv, as
    // the passes did for the blend), add_source, Dedner damping
    double um[NV], uh[5];
#pragma unroll
    for (int n = 0; n < NV; n++) um[n] = a.Uin[n * N + oc];
#pragma unroll
    for (int n = 0; n < 5; n++) uh[n] = a.Uin[(NV + n) * N + oc];
    const double acc = a.ac ? a.ac[oc] : a.col;
    double gr = 0.0, gi = 0.0, arb = 0.0;
    if (IR) {  // set_IR (rewrites and rates) before source_PIP, as in stage_tile
      set_ir_cell<NV>(um, uh, a.ph, a.irc, gr, gi);
      if (a.ph.flag_ir_type == 0) arb = a.arb_heat[oc];
    }
    double Sm[5], Sh[5], ion_pot;
    Phys phs = a.ph;
    phs.pip_imp = 0;
    source_pip(um, uh, acc, gr, gi, arb, phs, a.irc.heat_fac, Sh, Sm, ion_pot);
    if (a.ion_pot_out) a.ion_pot_out[oc] = ion_pot;
#pragma unroll
    for (int n = 0; n < 5; n++) {
      un[n] = un[n] + Sm[n] * dt_sub;
      un[NV + n] = un[NV + n] + Sh[n] * dt_sub;
    }
    if (NV == 9) {
      double fac = pexp(-dt_sub / dt * a.ph.safety * a.db_clean);
      un[8] = un[8] * fac;
    }
    if (epi >= 1) {
      if (epi >= 2) cfl_rewrite<NV, IR>(un, un + NV, a);  // main.f90:44-47, its dt unused
      r = cfl_round<NV, IR>(un, un + NV, acc, ion_pot, a);
#pragma unroll
      for (int n = 0; n < NV; n++) nanflag |= !(un[n] * 0.0 == 0.0);
    }
    store_cell<2, NVT>(a.Uout, N, a.ix, a.jx, ci, cj, un, a.bnd);
  }
  if (!REPLAY && a.epi >= 1) {
    __syncthreads();
    block_reduce_store<NT, IR>(r, nanflag, valid, a.red[blockIdx.x & (a.nred - 1)].v, smem);
  }
}

// ------------------------------------------------------- pointwise kernels
// Rewrite chain on every cell (ghosts included, as the reference's array
// statements do): flags select set_IR (+rates/arb_heat) and cfl.
struct RoundArgs {
  double* U;
  const double* ac;
  double* gm_rec;
  double* gm_ion;
  double* arb_heat;
  const double* ion_pot;
  RedSlot* red;
  int nred;
  int ix, jx, nx, ny;
  long long N;
  int do_ir, init_arb, do_cfl, read_rates, do_col;
  double* ac_out;  // do_col with col_type >= 1: alpha_c of every cell
  double col, gmin_safety;
  Phys ph;
  IRConst irc;
};

template <int NV, bool IR>
__global__ void __launch_bounds__(256) k_round(RoundArgs a) {
  constexpr int NVT = NV + 5;
  __shared__ double red_lds[4 * 5];
  long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long N = a.N;
  bool inb = k < N;
  RoundOut r = {1.0e300, 0.0, 0.0, 0.0};
  bool interior = false;
  int nanflag = 0;
  if (inb) {
    int i = (int)(k % a.ix), j = (int)(k / a.ix);
    interior = (i >= 2 && i < a.ix - 2) && (a.jx == 1 || (j >= 2 && j < a.jx - 2));
    double u[NVT];
#pragma unroll
    for (int n = 0; n < NVT; n++) u[n] = a.U[n * N + k];
    double* um = u;
    double* uh = u + NV;
    double acc = a.ac ? a.ac[k] : a.col;
    if (a.do_col && col_type(a.ph) >= 1) {  // set_collisional of set_coefficients(.,0)
      acc = set_col_cell(um, uh, a.col, a.ph);
      a.ac_out[k] = acc;
    }
    double gr = 0.0, gi = 0.0;
    if (IR && a.do_ir) {
      set_ir_cell<NV>(um, uh, a.ph, a.irc, gr, gi);
      a.gm_rec[k] = gr;
      a.gm_ion[k] = gi;
      if (a.init_arb) a.arb_heat[k] = gi * uh[0] * a.irc.heat_fac;
    } else if (IR && a.read_rates) {
      gr = a.gm_rec[k];
      gi = a.gm_ion[k];
    }
    if (a.do_cfl) {
      double dtc = cfl_cell<NV>(um, uh, a.gmin_safety, a.ph);
      r.dtc = interior ? dtc : 1.0e300;
      r.rhoac = dmax(um[0] * acc, uh[0] * acc);
      r.gmax = dmax(gr, gi);
      if (IR && a.ph.flag_ir_type == 0) {
        double pr, te;
        getpr_mhd(um, pr, te, a.ph);
        r.ratio = (a.ion_pot && interior) ? qdiv(a.ion_pot[k], quo(pr, a.ph.gm - 1.0, a.ph.rgm1)) : 0.0;
      }
      if (interior) {
#pragma unroll
        for (int n = 0; n < NV; n++) nanflag |= !(u[n] * 0.0 == 0.0);
      }
    }
#pragma unroll
    for (int n = 0; n < NVT; n++) a.U[n * N + k] = u[n];
  }
  if (a.do_cfl) block_reduce_store<256, IR>(r, nanflag, inb, a.red[blockIdx.x & (a.nred - 1)].v, red_lds);
}

// Ghost fill by the composite x-then-y map (Boundary_rot.f90:34-125).
__global__ void __launch_bounds__(256) k_bnd(double* U, int nvt, int ix, int jx, long long N, Bnd b,
                                             int ndim) {
  long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= N) return;
  int i = (int)(k % ix), j = (int)(k / ix);
  bool gx = (i < 2 || i >= ix - 2);
  bool gy = (ndim == 2) && (j < 2 || j >= jx - 2);
  if (!gx && !gy) return;
  bool fx = false, fy = false;
  int si = gx ? src_index(i, ix, b.type[0], b.type[1], fx) : i;
  int sj = gy ? src_index(j, jx, b.type[2], b.type[3], fy) : j;
  unsigned m = 0;
  if (fx) m ^= b.sym[(i < 2) ? 0 : 1];
  if (fy) m ^= b.sym[(j < 2) ? 2 : 3];
  long long s = (long long)sj * ix + si;
  for (int n = 0; n < nvt; n++) {
    double v = U[n * N + s];
    U[n * N + k] = ((m >> n) & 1u) ? -v : v;
  }
}

// mode 0: pip_cfl (optionally into the global dt); mode 2: the same at the
// top of a fused loop (also sets active/last); mode 1: end of a fused step.
// src (mode 1): the scalars and slots of the step that ends, sc / red or the
// second set of a chunk of folded steps; the result goes to sc.
__global__ void __launch_bounds__(64) k_finalize(FinArgs f) {
  DevScalars* sc = f.sc;
  if (f.mode == 1) {
    StepState s = load_state(f.src);
    if (!s.active && f.src == sc) {  // stopped before: nothing to end or to pass on, the slots are as reset
      if (f.hist && threadIdx.x == 0) record_dt(s, f.hist, f.hist_k);
      return;
    }
    if (s.active) s = step_end(s, combine_slots(load_slot(f.src_red, f.nred, f.flag_ir), f.nred, f.flag_ir), f);
    if ((int)threadIdx.x < f.nred) {
      f.red[threadIdx.x] = red_slot_init();
      if (f.src_red != f.red) f.src_red[threadIdx.x] = red_slot_init();
    }
    if (threadIdx.x != 0) return;
    store_state(sc, s);
    if (f.hist) record_dt(s, f.hist, f.hist_k);
    return;
  }
  const RedVals v = combine_slots(load_slot(f.red, f.nred, f.flag_ir), f.nred, f.flag_ir);
  if ((int)threadIdx.x < f.nred) f.red[threadIdx.x] = red_slot_init();
  if (threadIdx.x != 0) return;
  const double dttemp = cfl_dt(v, sc->ion_pot_valid, f);
  sc->dt_out = dttemp;
  if (f.into_global) sc->dt = dttemp;
  if (f.flag_divb >= 1) sc->cmax = f.safety * f.dxyz_min / sc->dt;
  sc->status = v.nan ? 2 : 0;
  if (f.mode == 2) {  // top of the time loop: decide whether this step is the last
    bool go = (sc->time < sc->tend) && (sc->nt < sc->nmax);
    sc->active = go ? 1 : 0;
    sc->last = ((sc->time + sc->dt >= sc->tend) || (sc->nt + 1 >= sc->nmax) || (sc->dt <= 1.0e-12)) ? 1 : 0;
  }
}

}  // namespace PIP_NS

namespace PIP_NS {
// Small control kernel: set loop bookkeeping fields on the device.
__global__ void k_set_loop(DevScalars* sc, double tend, long long nmax, int active, int ion_valid) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  sc->tend = tend;
  sc->nmax = nmax;
  if (active >= 0) sc->active = active;
  if (ion_valid >= 0) sc->ion_pot_valid = ion_valid;
}
}  // namespace PIP_NS

namespace PIP_NS {
// ------------------------------------------------------ batched ensemble
// One persistent launch integrates an ensemble of independent 1-D runs of
// different sizes: each workgroup pulls a member index from a device queue
// (longest expected run first) and runs that member's whole time loop
// (main.f90:31-68) in a loop over TX-cell tiles of stage_tile, with its own
// dt, time and step count.  The arithmetic per cell is that of the plain
// path, so every member equals its plain run bit for bit.
struct EnsMember {
  long long off;  // offset (doubles) of the member's block: nv + 5 planes of ix * jx
  int nx, ix;
  double dx, col, gmin_safety, tend;
  long long nmax;
  // 2-D members (ny = 0 in 1-D): rows, padded rows, dy, min(dx, dy, dz)
  int ny, jx;
  double dy, dxyz_min;
};
struct EnsOut {
  double time, dt;
  long long nt;
  int status, pad;
};
struct EnsArgs {
  double* U;
  double* U1;
  const EnsMember* mem;
  EnsOut* out;
  const int* order;
  unsigned* counter;
  int n_members;
  Phys ph;
  Bnd bnd;
  double db_clean;
};

__global__ void k_reset_counter(unsigned* c) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *c = 0u;
}

// Workgroup min/max of the dt terms; every thread gets the result.
template <int NT>
__device__ __forceinline__ RoundOut wg_reduce(RoundOut r, int& fl, double* lds) {
  for (int off = 32; off > 0; off >>= 1) {
    r.dtc = dmin(r.dtc, __shfl_xor(r.dtc, off, 64));
    r.rhoac = dmax(r.rhoac, __shfl_xor(r.rhoac, off, 64));
    fl |= __shfl_xor(fl, off, 64);
  }
  constexpr int NW = (NT + 63) / 64;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) {
    lds[wid * 3 + 0] = r.dtc;
    lds[wid * 3 + 1] = r.rhoac;
    lds[wid * 3 + 2] = (double)fl;
  }
  __syncthreads();
  RoundOut o = {lds[0], lds[1], 0.0, 0.0};
  int f = (int)lds[2];
  for (int w = 1; w < NW; w++) {
    o.dtc = dmin(o.dtc, lds[w * 3 + 0]);
    o.rhoac = dmax(o.rhoac, lds[w * 3 + 1]);
    f |= (int)lds[w * 3 + 2];
  }
  __syncthreads();
  fl = f;
  return o;
}

// cfl rewrite round over all cells of a member (ghosts included), as
// k_round does for the plain path; returns the reduced dt terms.
template <int TX>
__device__ __forceinline__ RoundOut ens_cfl_cells(double* U, const StageArgs& a, double* lds) {
  RoundOut acc = {1.0e300, 0.0, 0.0, 0.0};
  int fl = 0;
  for (int k = threadIdx.x; k < a.ix; k += TX) {
    double u[13];
#pragma unroll
    for (int n = 0; n < 13; n++) u[n] = U[n * a.N + k];
    double dtc = cfl_cell<8>(u, u + 8, a.gmin_safety, a.ph);
    bool interior = (k >= 2 && k < a.ix - 2);
    if (interior) acc.dtc = dmin(acc.dtc, dtc);
    acc.rhoac = dmax(acc.rhoac, dmax(u[0] * a.col, u[8] * a.col));
#pragma unroll
    for (int n = 0; n < 13; n++) U[n * a.N + k] = u[n];
  }
  return wg_reduce<TX>(acc, fl, lds);
}

__device__ __forceinline__ double ens_dt(const RoundOut& o, double safety) {
  // cfl without IR: Scheme_rot.f90:186-201
  double dttemp = dmin(10.0, o.dtc);
  return dmin(dttemp, dmin(safety, 0.3) / o.rhoac);
}

// StageArgs of ensemble member M (1-D, nvar_m = 8, constant alpha_c,
// explicit collisions, no IR); the state pointers are set per stage.
__device__ __forceinline__ StageArgs ens_stage_args(const EnsArgs& e, const EnsMember& M) {
  StageArgs a;
  a.ac = nullptr;
  a.ac_out = nullptr;
  a.U0out = nullptr;
  a.xcd_remap = 0;
  a.arb_heat = nullptr;
  a.ion_pot_out = nullptr;
  a.Vout = nullptr;
  a.dtc = nullptr;
  a.sc = nullptr;
  a.red = nullptr;
  a.nred = 0;
  a.fold = 0;
  a.ix = M.ix;
  a.jx = 1;
  a.nx = M.nx;
  a.ny = 1;
  a.N = M.ix;
  a.t_order = 2;
  a.col = M.col;
  a.gmin_safety = M.gmin_safety;
  a.dxyz_min = M.dx;
  a.dx = M.dx;
  a.dy = 100.0;
  a.db_clean = e.db_clean;
  a.ph = e.ph;
  a.irc = IRConst{};
  a.bnd = e.bnd;
  return a;
}

// Start of a member's run by one workgroup: the boundary map of the
// initial state (Initial_rot.f90:160), the prologue cfl and the loop-top
// cfl of the first iteration; returns the first dt.
template <int TX>
__device__ __forceinline__ double ens_start(const EnsArgs& e, const EnsMember& M, const StageArgs& a,
                                            double* U, double* lds_red) {
  if (threadIdx.x < 4) {
    int g = (threadIdx.x < 2) ? threadIdx.x : M.ix - 4 + threadIdx.x;
    bool flip;
    int sidx = src_index(g, M.ix, e.bnd.type[0], e.bnd.type[1], flip);
    unsigned msk = flip ? e.bnd.sym[(g < 2) ? 0 : 1] : 0u;
    for (int n = 0; n < 13; n++) {
      double v = U[n * a.N + sidx];
      U[n * a.N + g] = ((msk >> n) & 1u) ? -v : v;
    }
  }
  __syncthreads();
  ens_cfl_cells<TX>(U, a, lds_red);
  __syncthreads();
  RoundOut o = ens_cfl_cells<TX>(U, a, lds_red);
  return ens_dt(o, e.ph.safety);
}

template <int TX>
__global__ void __launch_bounds__(TX) k_ensemble(EnsArgs e) {
  extern __shared__ double smem[];
  __shared__ int s_member;
  constexpr int TC = TX - 1;  // cells per tile: TC+1 faces = one pass of TX threads
  using G = TileGeom<1, 8, TC, 1>;
  double* lds_red = smem + G::LDS_DOUBLES;  // 3 * (TX/64) doubles past the tile
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) s_member = (int)atomicAdd(e.counter, 1u);
    __syncthreads();
    const int q = s_member;
    if (q >= e.n_members) break;
    const int m = e.order[q];
    const EnsMember M = e.mem[m];
    double* U = e.U + M.off;
    double* U1 = e.U1 + M.off;
    StageArgs a = ens_stage_args(e, M);
    double dt = ens_start<TX>(e, M, a, U, lds_red);
    double time = 0.0;
    long long nt = 0;
    int status = 0;
    while (time < M.tend && nt < M.nmax && status == 0) {
      const bool last = (time + dt >= M.tend) || (nt + 1 >= M.nmax) || (dt <= 1.0e-12);
      // The flag is opaque and no load passes it: else parts of a tile are
      // carried over the loop of tiles (364 registers and one wave per SIMD, a
      // 432 B spill at 512 threads; 224 and none with it).
      auto now = [&](int epi) {
        int on = 1;
        asm volatile("" : "+s"(on)::"memory");
        return StepNow{dt, 0.0, epi, on != 0};
      };
      RoundOut r;
      int nanflag;
      a.istep = 1;
      a.Uin = U;
      a.U0 = U;
      a.Uout = U1;
      a.epi = 0;
      for (int i0 = 0; i0 < M.nx; i0 += TC) {
        stage_tile<1, 8, false, false, TC, 1, TX>(a, [&] { return now(0); }, i0, 0, smem, r, nanflag);
        __syncthreads();
      }
      __threadfence_block();
      __syncthreads();
      a.istep = 2;
      a.Uin = U1;
      a.U0 = U;
      a.Uout = U;
      const int epi = last ? 1 : 2;
      RoundOut acc = {1.0e300, 0.0, 0.0, 0.0};
      int fl = 0;
      for (int i0 = 0; i0 < M.nx; i0 += TC) {
        bool v = stage_tile<1, 8, false, false, TC, 1, TX>(a, [&] { return now(epi); }, i0, 0, smem, r,
                                                          nanflag);
        if (v) {
          acc.dtc = dmin(acc.dtc, r.dtc);
          acc.rhoac = dmax(acc.rhoac, r.rhoac);
          fl |= nanflag;
        }
        __syncthreads();
      }
      __threadfence_block();
      RoundOut red = wg_reduce<TX>(acc, fl, lds_red);
      double dt_new = ens_dt(red, e.ph.safety);
      time = time + dt;
      nt = nt + 1;
      if (dt <= 1.0e-12) status |= 1;
      if (fl) status |= 2;
      if (time < M.tend && nt < M.nmax && status == 0) dt = dt_new;
    }
    if (threadIdx.x == 0) {
      EnsOut out;
      out.time = time;
      out.dt = dt;
      out.nt = nt;
      out.status = status;
      out.pad = 0;
      e.out[m] = out;
    }
  }
}

// ------------------------------------------------------ lockstep ensemble
// The ensemble with every member spread over workgroups instead of one: a
// start kernel (one workgroup per member), then per step two stage launches
// over a table of (member, tile) pairs of the running members.  Per-member
// dt, time, step count, flags and reductions live in DevScalars, two
// buffers by step parity: stage 1 of step k applies the end of step k-1
// (read from buffer (k-1)&1, in every workgroup of the member alike) and the
// member's first tile writes the result to buffer k&1, which stage 2 then
// reads and reduces into; at the end of a host chunk, k_lock_end applies
// the last step's end.  Every operation is the persistent loop's
// (k_ensemble) and the plain path's, so the results agree with both bit for
// bit; the members' tiles run in parallel, as in the plain path, instead of
// one after another on one CU.
struct LockTile {
  int m, i0, j0, pad;  // member, first cell of the tile (column, row)
};

// The persistent loop's step end for one member: dt of the next step from
// the reductions, time, step count, status and the active / last flags.  A
// member that has stopped keeps its state; *stops says whether it stops at
// this step end.
struct LockState {
  StepState s;
  unsigned long long dt, rhoac, nan;  // the member's slots
};
__device__ __forceinline__ LockState load_lock(const DevScalars* p) {
  return LockState{load_state(p), p->red[RED_DT], p->red[RED_RHOAC], p->red[RED_NAN]};
}
__device__ __forceinline__ StepState lock_step_end(const LockState& l, const EnsMember& M, double safety, bool* stops) {
  StepState o = l.s;
  *stops = false;
  if (!o.active) return o;
  const RoundOut red = {as_f64(l.dt), as_f64(l.rhoac), 0.0, 0.0};
  const double dt = o.dt;
  const double dt_new = ens_dt(red, safety);
  o.time = o.time + dt;
  o.nt = o.nt + 1;
  if (dt <= 1.0e-12) o.status |= 1;
  if (l.nan != 0ull) o.status |= 2;
  if (o.time < M.tend && o.nt < M.nmax && o.status == 0) {
    o.dt = dt_new;
    if (M.ny > 0) o.cmax = safety * M.dxyz_min / dt_new;  // GLM speed of 2-D members (psi)
    o.last = ((o.time + dt_new >= M.tend) || (o.nt + 1 >= M.nmax) || (dt_new <= 1.0e-12)) ? 1 : 0;
  } else {
    o.active = 0;
    *stops = true;
  }
  return o;
}
// ... written to p with reset slots.
__device__ __forceinline__ void store_lock(DevScalars* p, const StepState& s) {
  store_state(p, s);
  const RedSlot r = red_slot_init();
#pragma unroll
  for (int n = 0; n < RED_N; n++) p->red[n] = r.v[n];
}

template <int TX>
__global__ void __launch_bounds__(TX) k_lock_start(EnsArgs e, DevScalars* scs) {
  extern __shared__ double smem[];
  constexpr int TC = TX - 1;
  using G = TileGeom<1, 8, TC, 1>;
  double* lds_red = smem + G::LDS_DOUBLES;
  const int m = blockIdx.x;
  if (m >= e.n_members) return;
  const EnsMember M = e.mem[m];
  const StageArgs a = ens_stage_args(e, M);
  const double dt = ens_start<TX>(e, M, a, e.U + M.off, lds_red);
  if (threadIdx.x == 0) {
    DevScalars sc;
    sc.dt = dt;
    sc.time = 0.0;
    sc.cmax = 0.0;
    sc.tend = M.tend;
    sc.dt_out = dt;
    sc.nt = 0;
    sc.nmax = M.nmax;
    sc.status = 0;
    sc.ion_pot_valid = 0;
    sc.red[RED_DT] = as_u64(1.0e300);
    sc.red[RED_RHOAC] = 0ull;
    sc.red[RED_GMAX] = 0ull;
    sc.red[RED_IONPOT] = 0ull;
    sc.red[RED_NAN] = 0ull;
    const bool go = (0.0 < M.tend) && (0 < M.nmax);
    sc.active = go ? 1 : 0;
    sc.last = ((0.0 + dt >= M.tend) || (1 >= M.nmax) || (dt <= 1.0e-12)) ? 1 : 0;
    scs[m] = sc;  // both parity buffers
    scs[e.n_members + m] = sc;
    if (!go) e.out[m] = EnsOut{0.0, dt, 0, 0, 0};
  }
}

// The step's scalars of a member for one of its tiles: stage 1 with apply_end
// applies the end of the step before (prev) once the tile's loads are issued,
// and the member's first tile writes it to sc.  stopped(): asked before any
// load, since the launches after a member's last step find it there.
template <int ISTEP>
struct LockStep {
  const EnsArgs& e;
  const EnsMember& M;
  DevScalars* sc;
  LockState now;
  bool end, first, active = false;
  int m;
  __device__ __forceinline__ LockStep(const EnsArgs& e_, const EnsMember& M_, DevScalars* sc_, const DevScalars* prev,
                                      int apply_end, int m_, bool first_)
      : e(e_), M(M_), sc(sc_), end(ISTEP == 1 && apply_end), first(first_), m(m_) {
    now = load_lock(end ? prev : sc);
  }
  __device__ __forceinline__ bool stopped() {
    if (now.s.active) return false;
    if (end && first && threadIdx.x == 0) store_lock(sc, now.s);
    return true;
  }
  __device__ __forceinline__ StepNow begin() {
    if (end) {
      bool stops;
      now.s = lock_step_end(now, M, e.ph.safety, &stops);
      if (first && threadIdx.x == 0) {
        store_lock(sc, now.s);
        if (stops) e.out[m] = EnsOut{now.s.time, now.s.dt, now.s.nt, now.s.status, 0};
      }
    }
    active = now.s.active != 0;
    return StepNow{now.s.dt, now.s.cmax, (ISTEP == 1) ? 0 : (now.s.last ? 1 : 2), active};
  }
};

// Stage ISTEP (1 or 2) of step k of the running members, one tile per
// workgroup; p = k & 1.  Stage 1 with apply_end first applies step k-1's
// end; stage 2 carries the cfl rounds and reduces into the member's slots.
// BF: tiles of bounded cells take the bounded fluxes.
template <int TX, int ISTEP, bool BF>
__global__ void __launch_bounds__(TX, 3) k_lock_stage(EnsArgs e, DevScalars* scs, const LockTile* tiles, int p,
                                                   int apply_end) {
  extern __shared__ double smem[];
  constexpr int TC = TX - 1;
  const LockTile t = tiles[blockIdx.x];
  const EnsMember M = e.mem[t.m];
  DevScalars* sc = scs + (long long)p * e.n_members + t.m;
  StageArgs a = ens_stage_args(e, M);
  double* U = e.U + M.off;
  double* U1 = e.U1 + M.off;
  a.istep = ISTEP;
  a.Uin = (ISTEP == 1) ? U : U1;
  a.U0 = U;
  a.Uout = (ISTEP == 1) ? U1 : U;
  a.epi = 0;
  RoundOut r;
  int nanflag;
  LockStep<ISTEP> step(e, M, sc, scs + (long long)(p ^ 1) * e.n_members + t.m, apply_end, t.m, t.i0 == 0);
  if (step.stopped()) return;
  const bool valid = stage_tile<1, 8, false, false, TC, 1, TX, STAGE_PLAIN, BF>(a, [&] { return step.begin(); }, t.i0, 0, smem, r, nanflag);
  if (ISTEP == 2 && step.active) {
    __syncthreads();
    block_reduce_store<TX, false>(r, nanflag, valid, sc->red, smem);
  }
}

// Number of members still running, from scalar buffer 0 (where a chunk's
// closing k_lock_end leaves them); one workgroup.
__global__ void k_lock_count(const DevScalars* scs, int n, int* active) {
  __shared__ int cnt;
  if (threadIdx.x == 0) cnt = 0;
  __syncthreads();
  int c = 0;
  for (int m = (int)threadIdx.x; m < n; m += (int)blockDim.x) c += scs[m].active ? 1 : 0;
  if (c) atomicAdd(&cnt, c);
  __syncthreads();
  if (threadIdx.x == 0) *active = cnt;
}

// ---------------------------------------------------- 2-D ensemble members
// Members of a 2-D ensemble: the plain path's 2-D stage (psi, no IR,
// constant alpha_c, explicit collisions) on 16x15 tiles of 256 threads,
// every member's tiles side by side in the lockstep launches.
constexpr int kEns2TX = 16, kEns2TY = 15, kEns2NT = 256;

__device__ __forceinline__ StageArgs ens_stage_args2(const EnsArgs& e, const EnsMember& M) {
  StageArgs a = ens_stage_args(e, M);
  a.jx = M.jx;
  a.ny = M.ny;
  a.N = (long long)M.ix * M.jx;
  a.dy = M.dy;
  a.dxyz_min = M.dxyz_min;
  return a;
}

// Start of the 2-D members, three launches over (256 cells, member): the
// boundary map of the initial state (ghosts from interior sources, k_bnd's
// composite map) with reset slots; the prologue cfl and the loop-top cfl of
// every cell (ghosts included, as k_round does; pointwise, so one pass makes
// both rewrites) reduced into the member's slots; the members' scalars.  One
// workgroup a member took 1.0 ms for the 68,000 cells of a 256^2 member, these
// take 0.03.  A member's workgroups go over its cells in strides, as the host
// limits their number (kStartGroups).
__global__ void __launch_bounds__(256) k_lock_bnd2(EnsArgs e, DevScalars* scs) {
  const int m = blockIdx.y;
  const EnsMember M = e.mem[m];
  const long long N = (long long)M.ix * M.jx;
  double* U = e.U + M.off;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    const RedSlot r = red_slot_init();
    for (int n = 0; n < RED_N; n++) scs[m].red[n] = r.v[n];
  }
  for (long long k = (long long)blockIdx.x * 256 + threadIdx.x; k < N; k += (long long)gridDim.x * 256) {
    const int i = (int)(k % M.ix), j = (int)(k / M.ix);
    const bool gx = (i < 2 || i >= M.ix - 2), gy = (j < 2 || j >= M.jx - 2);
    if (!gx && !gy) continue;
    bool fx = false, fy = false;
    const int si = gx ? src_index(i, M.ix, e.bnd.type[0], e.bnd.type[1], fx) : i;
    const int sj = gy ? src_index(j, M.jx, e.bnd.type[2], e.bnd.type[3], fy) : j;
    unsigned msk = 0u;
    if (fx) msk ^= e.bnd.sym[(i < 2) ? 0 : 1];
    if (fy) msk ^= e.bnd.sym[(j < 2) ? 2 : 3];
    const long long src = (long long)sj * M.ix + si;
    for (int n = 0; n < 14; n++) {
      const double v = U[n * N + src];
      U[n * N + k] = ((msk >> n) & 1u) ? -v : v;
    }
  }
}

__global__ void __launch_bounds__(256) k_lock_cfl2(EnsArgs e, DevScalars* scs) {
  __shared__ double red_lds[4 * 5];
  const int m = blockIdx.y;
  const EnsMember M = e.mem[m];
  const long long N = (long long)M.ix * M.jx;
  if ((long long)blockIdx.x * 256 >= N) return;
  double* U = e.U + M.off;
  RoundOut r = {1.0e300, 0.0, 0.0, 0.0};
  for (long long k = (long long)blockIdx.x * 256 + threadIdx.x; k < N; k += (long long)gridDim.x * 256) {
    double u[14];
#pragma unroll
    for (int n = 0; n < 14; n++) u[n] = U[n * N + k];
    cfl_cell<9>(u, u + 9, M.gmin_safety, e.ph);
    const double dtc = cfl_cell<9>(u, u + 9, M.gmin_safety, e.ph);
    const int i = (int)(k % M.ix), j = (int)(k / M.ix);
    if (i >= 2 && i < M.ix - 2 && j >= 2 && j < M.jx - 2) r.dtc = dmin(r.dtc, dtc);
    r.rhoac = dmax(r.rhoac, dmax(u[0] * M.col, u[9] * M.col));
#pragma unroll
    for (int n = 0; n < 14; n++) U[n * N + k] = u[n];
  }
  block_reduce_store<256, false>(r, 0, true, scs[m].red, red_lds);
}

__global__ void __launch_bounds__(256) k_lock_init2(EnsArgs e, DevScalars* scs) {
  const int m = (int)(blockIdx.x * 256 + threadIdx.x);
  if (m >= e.n_members) return;
  const EnsMember M = e.mem[m];
  const RoundOut o = {as_f64(scs[m].red[RED_DT]), as_f64(scs[m].red[RED_RHOAC]), 0.0, 0.0};
  const double dt = ens_dt(o, e.ph.safety);
  DevScalars sc;
  sc.dt = dt;
  sc.time = 0.0;
  sc.cmax = e.ph.safety * M.dxyz_min / dt;
  sc.tend = M.tend;
  sc.dt_out = dt;
  sc.nt = 0;
  sc.nmax = M.nmax;
  sc.status = 0;
  sc.ion_pot_valid = 0;
  const RedSlot r = red_slot_init();
  for (int n = 0; n < RED_N; n++) sc.red[n] = r.v[n];
  const bool go = (0.0 < M.tend) && (0 < M.nmax);
  sc.active = go ? 1 : 0;
  sc.last = ((0.0 + dt >= M.tend) || (1 >= M.nmax) || (dt <= 1.0e-12)) ? 1 : 0;
  scs[m] = sc;
  scs[e.n_members + m] = sc;
  if (!go) e.out[m] = EnsOut{0.0, dt, 0, 0, 0};
}

// Stage ISTEP of step k (p = k & 1) for one 16x15 tile of a 2-D member, as
// k_lock_stage does for 1-D members.  The table lists a member's tiles row by
// row, so XCD order keeps neighbours in one L2 (24 members up to 256^2, 96
// steps: 17.3 -> 16.0 ms).
template <int ISTEP>
__global__ void __launch_bounds__(kEns2NT, 2) k_lock_stage2(EnsArgs e, DevScalars* scs, const LockTile* tiles,
                                                            int p, int apply_end) {
  extern __shared__ double smem[];
  const LockTile t = tiles[xcd_tile(blockIdx.x, gridDim.x)];
  const EnsMember M = e.mem[t.m];
  DevScalars* sc = scs + (long long)p * e.n_members + t.m;
  StageArgs a = ens_stage_args2(e, M);
  double* U = e.U + M.off;
  double* U1 = e.U1 + M.off;
  a.istep = ISTEP;
  a.Uin = (ISTEP == 1) ? U : U1;
  a.U0 = U;
  a.Uout = (ISTEP == 1) ? U1 : U;
  a.epi = 0;
  RoundOut r;
  int nanflag;
  LockStep<ISTEP> step(e, M, sc, scs + (long long)(p ^ 1) * e.n_members + t.m, apply_end, t.m,
                       t.i0 == 0 && t.j0 == 0);
  if (step.stopped()) return;
  const bool valid = stage_tile<2, 9, false, false, kEns2TX, kEns2TY, kEns2NT>(a, [&] { return step.begin(); }, t.i0,
                                                                               t.j0, smem, r, nanflag);
  if (ISTEP == 2 && step.active) {
    __syncthreads();
    block_reduce_store<kEns2NT, false>(r, nanflag, valid, sc->red, smem);
  }
}

// Step end of the listed members (those of the chunk's table) after step k,
// p = k & 1: from buffer p into buffer p ^ 1; a member that stops writes its
// EnsOut.
__global__ void k_lock_end(EnsArgs e, DevScalars* scs, const int* members, int count, int p) {
  const int q = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (q >= count) return;
  const int m = members[q];
  bool stops;
  const StepState nw = lock_step_end(load_lock(scs + (long long)p * e.n_members + m), e.mem[m], e.ph.safety, &stops);
  store_lock(scs + (long long)(p ^ 1) * e.n_members + m, nw);
  if (stops) e.out[m] = EnsOut{nw.time, nw.dt, nw.nt, nw.status, 0};
}
// Step bookkeeping for recorded / replayed runs: hist[2k] = dt, hist[2k+1]
// = cmax of step k.
__global__ void k_record_dt(const DevScalars* sc, double* hist, int k) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  record_dt(load_state(sc), hist, k);
}
// End of a frozen-dt replay of n steps: the scalars a step-by-step run
// leaves (time and step count advanced, dt / cmax of the last step).
__global__ void k_replay_end(DevScalars* sc, const double* hist, int n) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  double t = sc->time;
  for (int k = 0; k < n; k++) t = t + hist[2 * k];
  sc->time = t;
  sc->nt = sc->nt + n;
  sc->dt = hist[2 * (n - 1)];
  sc->cmax = hist[2 * (n - 1) + 1];
  sc->active = 1;
  sc->last = 0;
}
__global__ void k_set_dt(DevScalars* sc, const double* hist, int k) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  sc->dt = hist[2 * k];
  sc->cmax = hist[2 * k + 1];
  sc->active = 1;
  sc->last = 0;
}


}  // namespace PIP_NS
