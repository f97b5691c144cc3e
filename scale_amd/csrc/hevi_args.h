// hevi_args.h -- arguments of a HEVI stage kernel and the RK4 combinations,
// shared by the column-march and tile kernels (hevi.hip) and the split stage
// (hevi_split.hip).
#pragma once
#include "common.h"
#include "shp_internal.h"

namespace shp {

// Arguments of a stage.  R is the type of the prognostic, tendency, flux and
// num_diff arrays: double, or float for the mixed-precision path, which keeps
// the reference state, the pressure terms (DPRES0, RT2P, REF_*) and the
// vertical solve in double; the solve's coefficients e, f and the face
// value PT pass from the upward to the downward sweep through scratch in R.
template <typename R>
struct HeviArgsT {
  const Ctx* ctx;  // host side only
  Dims d;
  Grid1D g;
  const double *GSQRT, *J13G, *J23G, *MAPF, *PHI;
  double J33G;
  // inputs (device layout)
  const R *DENS0, *MOMZ0, *MOMX0, *MOMY0, *RHOT0;
  const R *DENS, *MOMZ, *MOMX, *MOMY, *RHOT;
  const R *DENS_t, *MOMZ_t, *MOMX_t, *MOMY_t, *RHOT_t;
  // elements the tendencies are read at: index & tmask (0 where all five are
  // zero: every lane then reads element 0, one cached line instead of 5 arrays)
  size_t tmask = ~(size_t)0;
  const double *DPRES0, *RT2P, *CORIOLI;
  const R* num_diff;
  const double* wdamp_coef;
  const R* DDIV;
  const double *REF_dens, *REF_rhot;
  double divdmp_coef, dtrk;
  int has_coriolis;
  // outputs
  R *DENS_RK, *MOMZ_RK, *MOMX_RK, *MOMY_RK, *RHOT_RK, *mflx_hi, *tflx_hi;
  // scratch (n3 each): in FP32 the Thomas coefficients are rounded to float
  // between the sweeps (PT is a float value already), like the prognostics
  R *PT, *e, *f;
  // Sw between the two launches of the split terrain stage (FP64 only)
  double* Sw = nullptr;
  // optional records for the adjoint: St and the solved C
  double *trSt = nullptr, *trCp = nullptr;
  // mixed precision: DENS and RHOT (and their stage values) are stored as
  // deviations from the level profiles offD(k), offR(k), kept in double
  const double *offD = nullptr, *offR = nullptr;
  // RK4 combination fused into the last stage (hevi_tile with CMB)
  const R *c1[5], *c2[5], *c3[5];
  const R *cm[3], *ct[3];
  R* st[5];
  R *mflx_av, *tflx_av;
};
using HeviArgs = HeviArgsT<double>;

// RK4 combination (tinteg_short_rk4.F90:560-660): (2 r1 + 4 r2 + 2 r3 + r4 - 3 s0) / 6
template <typename R>
__device__ __forceinline__ R rk4c(R r1, R r2, R r3, R r4, R s0) {
  return (r1 * R(2) + r2 * R(4) + r3 * R(2) + r4 - s0 * R(3)) / R(6);
}
// (f1 + 2 f2 + 2 f3 + f4) / 6
template <typename R>
__device__ __forceinline__ R rk4f(R f1, R f2, R f3, R f4) {
  return (f1 + f2 * R(2) + f3 * R(2) + f4) / R(6);
}

// The FP64 stage as two launches, hevi_etile and hevi_columns (hevi_split.hip):
// flat or general metrics, with or without divergence damping and the fused
// RK4 combination.  Holds for grids hevi_split_fits accepts.
bool hevi_split_fits(const Dims& d);
hipError_t hevi_split(const HeviArgs& a, int scheme, bool terrain, bool divdmp, bool cmb, hipStream_t s);

}  // namespace shp
