// hevi_split.hip -- the FP64 HEVI stage as two launches (gfx950).
//
// Reference: ATMOS_DYN_Tstep_short_fvm_hevi,
//   scalelib/src/atmos-rm/dynamics/scale_atmos_dyn_tstep_short_fvm_hevi.F90:128-1089
// with the flux stencils of scale_atmos_dyn_fvm_flux_{ud3,cd4}.F90.
//   hevi_etile    the explicit part of every point (HEVI.F90:346-657, 816-1047)
//                 on LDS tiles of TI x TJ columns marching over a segment of
//                 levels: the mass and theta fluxes, MOMX_RK/MOMY_RK, Sr/St
//                 (into DENS_RK/RHOT_RK), Sw and the face value PT;
//   hevi_columns  the tridiagonal systems (HEVI.F90:688-804, 1092-1127): a
//                 block builds the rows of its columns with all its threads,
//                 keeps them in LDS, sweeps each column with one thread and
//                 updates with all of them again.
// The expressions and their order are those of the column march (hevi.hip),
// so the results are its bits.
#include <cstdlib>
#include "common.h"
#include "shp_internal.h"
#include "hevi_args.h"

namespace shp {

// the metric accessors of Met on byte offsets
template <bool TERRAIN>
struct MetO {
  const double *G, *J13, *J23, *MAPF;
  size_t n3, pl;
  int IA;
  __device__ __forceinline__ double gs(int c, unsigned o) const {
    if constexpr (TERRAIN) return ld(G + n3 * (size_t)c, o); else return 1.0;
  }
  __device__ __forceinline__ double j13(int c, unsigned o) const {
    if constexpr (TERRAIN) return ld(J13 + n3 * (size_t)c, o); else return 0.0;
  }
  __device__ __forceinline__ double j23(int c, unsigned o) const {
    if constexpr (TERRAIN) return ld(J23 + n3 * (size_t)c, o); else return 0.0;
  }
  // o: byte offset of (i,j) in a plane
  __device__ __forceinline__ double mapf(unsigned o, int n, int c) const {
    if constexpr (TERRAIN) return ld(MAPF + pl * (size_t)(n + 2 * c), o); else return 1.0;
  }
};

// ---------------------------------------------------------------------------
// Explicit part.  A block marches its tile over levels k0..k1 of one segment
// (from the level below, for the z fluxes through the segment's lower face, to
// the level above, whose Sr and St enter the segment's last row) and keeps
// DENS, MOMX, MOMY, MOMZ and POTT of levels k..k+2 in a three-level LDS ring
// with a 2-cell halo, and DPRES of the level (general metrics: of k-1..k+1).
// Every x and y face of the tile is evaluated once per level into LDS; each
// column differences its faces and carries its z fluxes from the level below.
// PART: P_T continuity, theta and MOMZ with the right-hand side of the
// column's rows, P_M the horizontal momenta.  The flat stage evaluates both in
// one launch and has the next level's loads in flight during the level's work;
// with general metrics both at once need more than 256 VGPRs, so each part is
// a launch of its own.
// Bound by memory latency at two waves per SIMD (its registers and LDS): at
// 512x512x128 flat 2.72 ms, 317 B of HBM traffic a point (208 read and 80
// written at least) at 3.9 TB/s.  The next level's num_diff of the faces is
// loaded ahead (2 % of a short step there); the ring's level too spills and is
// slower (by 17 %).  One thread per point reading its stencil
// through the caches, a launch per section, was the kernel before: 215 us
// against 105 for the flat explicit part at 128x128x64, 458 against 273 with
// general metrics, 2.88 ms against 1.59 at 301x259x80.
enum { P_T = 1, P_M = 2 };
template <int S, bool TERRAIN, bool DIVDMP, bool CMB, int PART, int TI, int TJ>
__global__ void __launch_bounds__(TI * TJ, 2) hevi_etile(HeviArgs a, unsigned ni, unsigned ntile, unsigned nblocks, int L) {
  constexpr bool PT_ = (PART & P_T) != 0, PM_ = (PART & P_M) != 0;
  constexpr bool PIPE_F = !TERRAIN;
  constexpr int CW = TI + 4, RW = TJ + 4, NT = TI * TJ;
  constexpr int ND_P = TERRAIN ? 3 : 1;
  __shared__ double sD[3][RW][CW], sMX[3][RW][CW], sMY[3][RW][CW], sW[3][RW][CW];  // slot = level % 3
  __shared__ double sPO[PT_ ? 3 : 1][PT_ ? RW : 1][PT_ ? CW : 1];
  __shared__ double sDP[PM_ ? ND_P : 1][PM_ ? TJ + 1 : 1][PM_ ? TI + 1 : 1];
  // x faces: position x = 0..TI is the face east of column i0-1+x; y faces likewise
  constexpr int XT = PT_ ? TJ : 1, XM = PM_ ? TJ : 1;
  __shared__ double xM[XT][TI + 1], xT[XT][TI + 1], xW[XT][TI + 1], xU[XM][TI + 1], xV[XM][TI + 1];
  __shared__ double yM[XT + 1][TI], yT[XT + 1][TI], yW[XT + 1][TI], yU[XM + 1][TI], yV[XM + 1][TI];

  const Dims& d = a.d;
  const unsigned lb = xcd_block(blockIdx.x, nblocks);
  const unsigned tile = lb % ntile, seg = lb / ntile;
  const int i0 = d.IS + (int)(tile % ni) * TI;
  const int j0 = d.JS + (int)(tile / ni) * TJ;
  const int tid = threadIdx.x, tx = tid % TI, ty = tid / TI;
  const int i = i0 + tx, j = j0 + ty;
  const bool own = (i <= d.IE) && (j <= d.JE);
  const int KS = d.KS, KE = d.KE;
  const int k0 = KS + (int)seg * L, k1 = min(KE, k0 + L - 1);
  const int kb = k0 > KS ? k0 - 1 : KS;                    // first level of the march
  const int ke = (PT_ && k1 < KE) ? k1 + 1 : k1;          // last one
  const size_t n3 = d.n3;
  const unsigned pl = (unsigned)d.pl * 8u, row8 = (unsigned)d.IA * 8u;  // bytes of a level, of a row
  MetO<TERRAIN> m;
  m.G = a.GSQRT; m.J13 = a.J13G; m.J23 = a.J23G; m.MAPF = a.MAPF; m.n3 = n3; m.pl = d.pl; m.IA = d.IA;
  const double* CDZ = a.g.CDZ;
  const double dtrk = a.dtrk, J33G = a.J33G;
  auto nd = [&](int v, int dir, unsigned q) { return ld(a.num_diff + n3 * (size_t)(v + 5 * dir), q); };
  auto gij = [&](int ii, int jj) { return (unsigned)(ii + d.IA * jj) * 8u; };  // byte offset in a level
  auto gix = [&](int k, int ii, int jj) { return gij(ii, jj) + pl * (unsigned)k; };
  // DPRES at any level KS-1..KE+1 (HEVI.F90:355-358)
  auto dpres = [&](int k, int ii, int jj) -> double {
    const unsigned q = gix(k, ii, jj);
    if (TERRAIN && k == KS - 1) return ld(a.DPRES0, q) - ld(a.DENS, q + pl) * (ld(a.PHI, q) - ld(a.PHI, q + 2 * pl));
    if (TERRAIN && k == KE + 1) return ld(a.DPRES0, q) - ld(a.DENS, q - pl) * (ld(a.PHI, q) - ld(a.PHI, q - 2 * pl));
    return ld(a.DPRES0, q) + ld(a.RT2P, q) * (ld(a.RHOT, q) - ld(a.REF_rhot, q));
  };

  // the first two levels of the ring; tile cell (r, c) is column i0-2+c, row j0-2+r
  for (int lv = kb; lv <= kb + 1; ++lv) {
    const int sl = lv % 3;
    for (int q = tid; q < RW * CW; q += NT) {
      const int r = q / CW, c = q - r * CW;
      const int ii = i0 - 2 + c, jj = j0 - 2 + r;
      const bool in = ii < d.IA && jj < d.JA;
      const unsigned g = in ? gix(lv, ii, jj) : 0;
      const double vD = in ? ld(a.DENS, g) : 0.0, vR = (PT_ && in) ? ld(a.RHOT, g) : 0.0;
      sD[sl][r][c] = vD;
      sMX[sl][r][c] = in ? ld(a.MOMX, g) : 0.0;
      sMY[sl][r][c] = in ? ld(a.MOMY, g) : 0.0;
      sW[sl][r][c] = in ? ld(a.MOMZ, g) : 0.0;
      if constexpr (PT_) sPO[sl][r][c] = in ? vR / vD : 0.0;
    }
  }
  if constexpr (TERRAIN && PM_) {
    for (int lv = kb - 1; lv <= kb; ++lv)
      for (int q = tid; q < (TJ + 1) * (TI + 1); q += NT) {
        const int r = q / (TI + 1), c = q - r * (TI + 1);
        const int ii = i0 + c, jj = j0 + r;
        sDP[lv % 3][r][c] = (ii < d.IA && jj < d.JA) ? dpres(lv, ii, jj) : 0.0;
      }
  }
  // the own column at level k-1 (levels k..k+2 are in the ring)
  const unsigned p0 = own ? gij(i, j) : 0;
  double pwm = 0, wwm = 0, xwm = 0, ywm = 0;
  if (own) {
    const unsigned g = p0 + pl * (unsigned)(kb - 1);
    wwm = ld(a.MOMZ, g);
    if constexpr (PT_) pwm = ld(a.RHOT, g) / ld(a.DENS, g);
    if constexpr (PM_) { xwm = ld(a.MOMX, g); ywm = ld(a.MOMY, g); }
  }
  const double rcdx = own ? a.g.RCDX[i] : 0.0, rcdy = own ? a.g.RCDY[j] : 0.0;
  const double rfdx = own ? a.g.RFDX[i] : 0.0, rfdy = own ? a.g.RFDY[j] : 0.0;
  // fluxes through the face below the level (zero at KS-1)
  double cmZ = 0, ctZ = 0, cqW = 0, cqU = 0, cqV = 0;
  double cW13 = 0, cW23 = 0, cU13 = 0, cU23 = 0, cV13 = 0, cV23 = 0;
  // general metrics of the own column carried up the march
  double gC = 1, gUW = 1, gXW = 1, gU = 1, gV = 1, gVm = 1, j13m = 0, j23m = 0;
  if constexpr (TERRAIN) {
    if (own) {
      const unsigned g = p0 + pl * (unsigned)kb;
      gC = m.gs(I_XYZ, g); gUW = m.gs(I_UYW, g); gXW = m.gs(I_XVW, g); gU = m.gs(I_UYZ, g); gV = m.gs(I_XVZ, g);
      gVm = m.gs(I_XVZ, g - pl); j13m = m.j13(I_UYW, g - pl); j23m = m.j23(I_XVW, g - pl);
    }
  }
  __syncthreads();

  // the column's row one level behind: level k-1's values
  double rt0 = 0, dp0 = 0, st0 = 0, sr0 = 0, rd0 = 0, sw0 = 0, gWm = 1, gCm = 1;

  constexpr int NX = (TJ * (TI + 1) + NT - 1) / NT, NY = ((TJ + 1) * TI + NT - 1) / NT;
  constexpr int NC = (RW * CW + NT - 1) / NT, NP = ((TJ + 1) * (TI + 1) + NT - 1) / NT;
  double fx[NX][5], fy[NY][5];
  double tD[NC], tX[NC], tY[NC], tW[NC], tR[NC], pD0[NP], pRT[NP], pRH[NP], pRR[NP];
  // the ring's new level k+2, and the inputs of DPRES at level k (general
  // metrics: k+1, whose ghost level is DPRES0 - DENS (PHI - PHI), HEVI.F90:357-358)
  auto issue_tile = [&](int k) {
#pragma unroll
    for (int h = 0; h < NC; ++h) {
      const int q = tid + h * NT, r = q / CW, c = q - r * CW;
      const int ii = i0 - 2 + c, jj = j0 - 2 + r;
      const bool ok = q < RW * CW && ii < d.IA && jj < d.JA && k + 2 < d.KA;
      const unsigned g = ok ? gix(k + 2, ii, jj) : 0;
      tD[h] = ok ? ld(a.DENS, g) : 0.0;
      tX[h] = ok ? ld(a.MOMX, g) : 0.0;
      tY[h] = ok ? ld(a.MOMY, g) : 0.0;
      tW[h] = ok ? ld(a.MOMZ, g) : 0.0;
      if constexpr (PT_) tR[h] = ok ? ld(a.RHOT, g) : 0.0;
    }
    if constexpr (PM_) {
#pragma unroll
      for (int h = 0; h < NP; ++h) {
        const int q = tid + h * NT, r = q / (TI + 1), c = q - r * (TI + 1);
        const int ii = i0 + c, jj = j0 + r;
        const bool ok = q < (TJ + 1) * (TI + 1) && ii < d.IA && jj < d.JA;
        const unsigned g = ok ? gix(TERRAIN ? k + 1 : k, ii, jj) : 0;
        pD0[h] = ok ? ld(a.DPRES0, g) : 0.0;
        if (TERRAIN && k == KE) {
          pRT[h] = ok ? -ld(a.DENS, g - pl) : 0.0;
          pRH[h] = ok ? ld(a.PHI, g) : 0.0;
          pRR[h] = ok ? ld(a.PHI, g - 2 * pl) : 0.0;
        } else {
          pRT[h] = ok ? ld(a.RT2P, g) : 0.0;
          pRH[h] = ok ? ld(a.RHOT, g) : 0.0;
          pRR[h] = ok ? ld(a.REF_rhot, g) : 0.0;
        }
      }
    }
  };
  // num_diff of the faces this thread evaluates
  auto issue_face = [&](int k) {
#pragma unroll
    for (int h = 0; h < NX; ++h) {
      const int q = tid + h * NT, row = q / (TI + 1), x = q - row * (TI + 1);
      const int ii = i0 - 1 + x, jj = j0 + row;
      const bool ok = q < TJ * (TI + 1) && ii <= d.IE && jj <= d.JE;
      const unsigned g = ok ? gix(k, ii, jj) : 0;
      if constexpr (PT_) {
        fx[h][0] = ok ? nd(I_DENS, XDIR, g) : 0.0;
        fx[h][1] = ok ? nd(I_RHOT, XDIR, g) : 0.0;
        fx[h][2] = (ok && k < KE) ? nd(I_MOMZ, XDIR, g) : 0.0;
      }
      if constexpr (PM_) {
        fx[h][3] = ok ? nd(I_MOMX, XDIR, g + 8) : 0.0;
        fx[h][4] = ok ? nd(I_MOMY, XDIR, g) : 0.0;
      }
    }
#pragma unroll
    for (int h = 0; h < NY; ++h) {
      const int q = tid + h * NT, y = q / TI, col = q - y * TI;
      const int ii = i0 + col, jj = j0 - 1 + y;
      const bool ok = q < (TJ + 1) * TI && ii <= d.IE && jj <= d.JE;
      const unsigned g = ok ? gix(k, ii, jj) : 0;
      if constexpr (PT_) {
        fy[h][0] = ok ? nd(I_DENS, YDIR, g) : 0.0;
        fy[h][1] = ok ? nd(I_RHOT, YDIR, g) : 0.0;
        fy[h][2] = (ok && k < KE) ? nd(I_MOMZ, YDIR, g) : 0.0;
      }
      if constexpr (PM_) {
        fy[h][3] = ok ? nd(I_MOMX, YDIR, g) : 0.0;
        fy[h][4] = ok ? nd(I_MOMY, YDIR, g + row8) : 0.0;
      }
    }
  };
  if constexpr (PIPE_F) { if (kb >= k0) issue_face(kb); }
  for (int k = kb; k <= ke; ++k) {
    const bool live = k >= k0;       // false: only the z fluxes through the face above level k0-1
    const bool full = live && k <= k1;  // false: Sr and St alone, for the row of level k1
    const int s0 = k % 3, s1 = (k + 1) % 3, s2 = (k + 2) % 3;
    const int sp = TERRAIN ? s1 : 0;
    issue_tile(k);
    if constexpr (!PIPE_F) { if (live) issue_face(k); }
#pragma unroll
    for (int h = 0; h < NC; ++h) {
      const int q = tid + h * NT;
      if (q >= RW * CW) continue;
      const int r = q / CW, c = q - r * CW;
      const bool in = i0 - 2 + c < d.IA && j0 - 2 + r < d.JA;
      sD[s2][r][c] = tD[h]; sMX[s2][r][c] = tX[h]; sMY[s2][r][c] = tY[h]; sW[s2][r][c] = tW[h];
      if constexpr (PT_) sPO[s2][r][c] = in ? tR[h] / tD[h] : 0.0;
    }
    if constexpr (PM_) {
#pragma unroll
      for (int h = 0; h < NP; ++h) {
        const int q = tid + h * NT;
        if (q >= (TJ + 1) * (TI + 1)) continue;
        const int r = q / (TI + 1), c = q - r * (TI + 1);
        sDP[sp][r][c] = pD0[h] + pRT[h] * (pRH[h] - pRR[h]);
      }
    }
    __syncthreads();
    // stages 1-3 of the combined fluxes of this thread's first x and y face
    double cx[CMB ? 6 : 1], cy[CMB ? 6 : 1];
    if constexpr (CMB && PT_) {
      if (full) {
        const int row = tid / (TI + 1), x = tid - row * (TI + 1), y = tid / TI, col = tid - y * TI;
        const bool okx = i0 - 1 + x <= d.IE && j0 + row <= d.JE, oky = i0 + col <= d.IE && j0 - 1 + y <= d.JE;
        const unsigned qx = okx ? gix(k, i0 - 1 + x, j0 + row) : 0, qy = oky ? gix(k, i0 + col, j0 - 1 + y) : 0;
#pragma unroll
        for (int n = 0; n < 3; ++n) {
          cx[n] = ld(a.cm[n] + n3, qx); cx[3 + n] = ld(a.ct[n] + n3, qx);
          cy[n] = ld(a.cm[n] + 2 * n3, qy); cy[3 + n] = ld(a.ct[n] + 2 * n3, qy);
        }
      }
    }
    // the column's own loads, in flight during the face evaluation
    const unsigned g = p0 + pl * (unsigned)k;
    double o_nZD = 0, o_nZT = 0, o_nZW = 0, o_nZX = 0, o_nZY = 0, o_nDw = 0;
    double o_Dt = 0, o_Rt = 0, o_Wt = 0, o_Xt = 0, o_Yt = 0, o_X0 = 0, o_Y0 = 0, o_Z0 = 0;
    double cmx[3], cmy[3];
    double o_RT = 0, o_RD = 0, o_P0 = 0, o_RR = 0, o_R = 0;
    const double wdc = a.wdamp_coef[k];
    if (own) {
      const unsigned gt = g & (unsigned)a.tmask;
      if constexpr (PT_) { o_nZD = nd(I_DENS, ZDIR, g); o_nZT = nd(I_RHOT, ZDIR, g); o_nZW = nd(I_MOMZ, ZDIR, g + pl); }
      if constexpr (PM_) { o_nZX = nd(I_MOMX, ZDIR, g); o_nZY = nd(I_MOMY, ZDIR, g); }
      if (live) {
        if constexpr (PT_) {
          o_Dt = ld(a.DENS_t, gt); o_Rt = ld(a.RHOT_t, gt); o_Wt = ld(a.MOMZ_t, gt);
          o_RT = ld(a.RT2P, g); o_RD = ld(a.REF_dens, g);
          if constexpr (!PM_) { o_P0 = ld(a.DPRES0, g); o_RR = ld(a.REF_rhot, g); o_R = ld(a.RHOT, g); }
          if (TERRAIN || wdc != 0.0) o_Z0 = ld(a.MOMZ0, g);
          if (i == d.IS && k <= KE - 1) o_nDw = nd(I_DENS, ZDIR, g - 8);
        }
        if constexpr (PM_) {
          o_Xt = ld(a.MOMX_t, gt); o_Yt = ld(a.MOMY_t, gt);
          o_X0 = ld(a.MOMX0, g); o_Y0 = ld(a.MOMY0, g);
          if constexpr (CMB) {
#pragma unroll
            for (int n = 0; n < 3; ++n) {
              const double* const* cs = n == 0 ? a.c1 : n == 1 ? a.c2 : a.c3;
              cmx[n] = ld(cs[2], g); cmy[n] = ld(cs[3], g);
            }
          }
        }
      }
    }
    // ---- faces ----
    const double cz0 = CDZ[k], cz1 = CDZ[k + 1];
    // F2H(k, 1) and F2H(k, 2) of the GSQRT values g0, g1 of levels k, k+1 (HEVI.F90:62)
    auto f2h = [&](double q0, double q1, double& f1, double& f2) {
      if constexpr (TERRAIN) {
        f1 = cz0 * q0 / (cz0 * q0 + cz1 * q1);
        f2 = cz1 * q1 / (cz0 * q0 + cz1 * q1);
      } else {
        f1 = cz0 / (cz0 + cz1);
        f2 = cz1 / (cz0 + cz1);
      }
    };
    auto D0 = [&](int r, int c) { return sD[s0][r][c]; };
    auto D1 = [&](int r, int c) { return sD[s1][r][c]; };
    if (live) {
#pragma unroll
      for (int h = 0; h < NX; ++h) {
        const int q = tid + h * NT, row = q / (TI + 1), x = q - row * (TI + 1);
        const int ii = i0 - 1 + x, jj = j0 + row;
        if (q >= TJ * (TI + 1) || ii > d.IE || jj > d.JE) continue;
        const int r = row + 2, c = x + 1;  // tile cell of column ii
        const unsigned gq = gix(k, ii, jj);
        if constexpr (PT_) {
        const double gUYZ = m.gs(I_UYZ, gq), gUYW = m.gs(I_UYW, gq);
        const double vm = gUYZ / m.mapf(gij(ii, jj), 1, I_UY) * (sMX[s0][r][c] + fx[h][0]);
        const double vt = vm * fv_int<S>(sPO[s0][r][c - 1], sPO[s0][r][c], sPO[s0][r][c + 1], sPO[s0][r][c + 2], vm)
                        + gUYZ * fx[h][1];
        xM[row][x] = vm;
        xT[row][x] = vt;
        double qw = 0.0;
        if (full && k < KE) {
          double f1, f2;
          f2h(gUYW, m.gs(I_UYW, gq + pl), f1, f2);
          const double vel = (f1 * sMX[s1][r][c] + f2 * sMX[s0][r][c])
                           / (f1 * 0.5 * (D1(r, c) + D1(r, c + 1)) + f2 * 0.5 * (D0(r, c) + D0(r, c + 1)));
          qw = gUYW / m.mapf(gij(ii, jj), 1, I_UY) * vel
             * fv_int<S>(sW[s0][r][c - 1], sW[s0][r][c], sW[s0][r][c + 1], sW[s0][r][c + 2], vel) + gUYW * fx[h][2];
        }
        xW[row][x] = qw;
        if (full) {
          if constexpr (CMB) {  // averaged over the stages at the interior faces this tile owns
            if (x > 0) {
              if (h == 0) {
                sto(a.mflx_av + n3, gq, rk4f(cx[0], cx[1], cx[2], vm));
                sto(a.tflx_av + n3, gq, rk4f(cx[3], cx[4], cx[5], vt));
              } else {
                sto(a.mflx_av + n3, gq, rk4f(ld(a.cm[0] + n3, gq), ld(a.cm[1] + n3, gq), ld(a.cm[2] + n3, gq), vm));
                sto(a.tflx_av + n3, gq, rk4f(ld(a.ct[0] + n3, gq), ld(a.ct[1] + n3, gq), ld(a.ct[2] + n3, gq), vt));
              }
            }
          } else if (x > 0 || i0 == d.IS) {  // faces IS-1 and those owned by this tile
            sto(a.mflx_hi + n3, gq, vm);
            sto(a.tflx_hi + n3, gq, vt);
          }
        }
        }
        if constexpr (PM_) {
        if (!full) continue;
        const double gUVZ = m.gs(I_UVZ, gq), gE = m.gs(I_XYZ, gq + 8);
        {  // fluxX_UYZ stored at ii (loop index ii+1)
          const double vel = (0.5 * (sMX[s0][r][c + 1] + sMX[s0][r][c])) / (D0(r, c + 1));
          xU[row][x] = gE / m.mapf(gij(ii + 1, jj), 1, I_XY) * vel
                     * fv_int<S>(sMX[s0][r][c - 1], sMX[s0][r][c], sMX[s0][r][c + 1], sMX[s0][r][c + 2], vel) + gE * fx[h][3];
        }
        {  // fluxX_XVZ at (ii, jj)
          const double vel = (0.5 * (sMX[s0][r][c] + sMX[s0][r + 1][c]))
                           / (0.25 * (D0(r, c) + D0(r, c + 1) + D0(r + 1, c) + D0(r + 1, c + 1)));
          xV[row][x] = gUVZ / m.mapf(gij(ii, jj), 1, I_UV) * vel
                     * fv_int<S>(sMY[s0][r][c - 1], sMY[s0][r][c], sMY[s0][r][c + 1], sMY[s0][r][c + 2], vel) + gUVZ * fx[h][4];
        }
        }
      }
#pragma unroll
      for (int h = 0; h < NY; ++h) {
        const int q = tid + h * NT, y = q / TI, col = q - y * TI;
        const int ii = i0 + col, jj = j0 - 1 + y;
        if (q >= (TJ + 1) * TI || ii > d.IE || jj > d.JE) continue;
        const int r = y + 1, c = col + 2;  // tile cell of row jj
        const unsigned gq = gix(k, ii, jj);
        if constexpr (PT_) {
        const double gXVZ = m.gs(I_XVZ, gq), gXVW = m.gs(I_XVW, gq);
        const double vm = gXVZ / m.mapf(gij(ii, jj), 0, I_XV) * (sMY[s0][r][c] + fy[h][0]);
        const double vt = vm * fv_int<S>(sPO[s0][r - 1][c], sPO[s0][r][c], sPO[s0][r + 1][c], sPO[s0][r + 2][c], vm)
                        + gXVZ * fy[h][1];
        yM[y][col] = vm;
        yT[y][col] = vt;
        double qw = 0.0;
        if (full && k < KE) {
          double f1, f2;
          f2h(gXVW, m.gs(I_XVW, gq + pl), f1, f2);
          const double vel = (f1 * sMY[s1][r][c] + f2 * sMY[s0][r][c])
                           / (f1 * 0.5 * (D1(r, c) + D1(r + 1, c)) + f2 * 0.5 * (D0(r, c) + D0(r + 1, c)));
          qw = gXVW / m.mapf(gij(ii, jj), 0, I_XV) * vel
             * fv_int<S>(sW[s0][r - 1][c], sW[s0][r][c], sW[s0][r + 1][c], sW[s0][r + 2][c], vel) + gXVW * fy[h][2];
        }
        yW[y][col] = qw;
        if (full) {
          if constexpr (CMB) {
            if (y > 0) {
              if (h == 0) {
                sto(a.mflx_av + 2 * n3, gq, rk4f(cy[0], cy[1], cy[2], vm));
                sto(a.tflx_av + 2 * n3, gq, rk4f(cy[3], cy[4], cy[5], vt));
              } else {
                sto(a.mflx_av + 2 * n3, gq, rk4f(ld(a.cm[0] + 2 * n3, gq), ld(a.cm[1] + 2 * n3, gq), ld(a.cm[2] + 2 * n3, gq), vm));
                sto(a.tflx_av + 2 * n3, gq, rk4f(ld(a.ct[0] + 2 * n3, gq), ld(a.ct[1] + 2 * n3, gq), ld(a.ct[2] + 2 * n3, gq), vt));
              }
            }
          } else if (y > 0 || j0 == d.JS) {
            sto(a.mflx_hi + 2 * n3, gq, vm);
            sto(a.tflx_hi + 2 * n3, gq, vt);
          }
        }
        }
        if constexpr (PM_) {
        if (!full) continue;
        const double gUVZ = m.gs(I_UVZ, gq), gN = m.gs(I_XYZ, gq + row8);
        {  // fluxY_UYZ at (ii, jj)
          const double vel = (0.5 * (sMY[s0][r][c] + sMY[s0][r][c + 1]))
                           / (0.25 * (D0(r, c) + D0(r, c + 1) + D0(r + 1, c) + D0(r + 1, c + 1)));
          yU[y][col] = gUVZ / m.mapf(gij(ii, jj), 0, I_UV) * vel
                     * fv_int<S>(sMX[s0][r - 1][c], sMX[s0][r][c], sMX[s0][r + 1][c], sMX[s0][r + 2][c], vel) + gUVZ * fy[h][3];
        }
        {  // fluxY_XVZ stored at jj (loop index jj+1)
          const double vel = (0.5 * (sMY[s0][r + 1][c] + sMY[s0][r][c])) / (D0(r + 1, c));
          yV[y][col] = gN / m.mapf(gij(ii, jj + 1), 0, I_XY) * vel
                     * fv_int<S>(sMY[s0][r - 1][c], sMY[s0][r][c], sMY[s0][r + 1][c], sMY[s0][r + 2][c], vel) + gN * fy[h][4];
        }
        }
      }
    }
    if constexpr (PIPE_F) {
      if (k < ke && k + 1 >= k0) issue_face(k + 1);
    }
    __syncthreads();

    // ---- the column ----
    if (own) {
      const int r = ty + 2, c = tx + 2;  // tile cell of the own column
      // the column's windows at k-1..k+2
      const double ww[4] = {wwm, sW[s0][r][c], sW[s1][r][c], sW[s2][r][c]};
      const double rcdz = a.g.RCDZ[k];
      const double m0 = m.mapf(p0, 0, I_XY), m1 = m.mapf(p0, 1, I_XY);
      const double gCp = m.gs(I_XYZ, g + pl);
      if constexpr (PT_) {
        const double pw[4] = {pwm, sPO[s0][r][c], sPO[s1][r][c], sPO[s2][r][c]};
        const double gW = m.gs(I_XYW, g);
        // explicit z fluxes through the face above level k
        auto explZ = [&](unsigned q, unsigned q2, int cc, double n) -> double {  // mflxZ at tile column cc
          if constexpr (TERRAIN) {
            const double t1 = m.mapf(q2, 0, I_XY), t2 = m.mapf(q2, 1, I_XY);
            return m.j13(I_XYW, q) * 0.25 / t2 * (sMX[s1][r][cc] + sMX[s1][r][cc - 1] + sMX[s0][r][cc] + sMX[s0][r][cc - 1])
                 + m.j23(I_XYW, q) * 0.25 / t1 * (sMY[s1][r][cc] + sMY[s1][r - 1][cc] + sMY[s0][r][cc] + sMY[s0][r - 1][cc])
                 + m.gs(I_XYW, q) / (t1 * t2) * n;
          } else {
            return n;
          }
        };
        const double mZ = (k <= KE - 1) ? explZ(g, p0, c, o_nZD) : 0.0;
        double tZ = 0.0;
        if (k <= KE - 1) {
          double fv;
          if (k == KS) fv = fv_lo<S>(pw[1], pw[2], pw[3], mZ);
          else if (k == KE - 1) fv = fv_hi<S>(pw[0], pw[1], pw[2], mZ);
          else fv = fv_int<S>(pw[0], pw[1], pw[2], pw[3], mZ);
          tZ = mZ * fv + gW * o_nZT;
        }
        double qw = 0.0, qW13 = 0.0, qW23 = 0.0;
        if (k < KE - 1 && k <= k1) {
          auto fvw = [&](double vel) {
            return (k == KS) ? fv_lo<S>(ww[1], ww[2], ww[3], vel) : fv_int<S>(ww[0], ww[1], ww[2], ww[3], vel);
          };
          const double vel = (0.5 * (ww[1] + ww[2])) / D1(r, c);
          qw = J33G * vel * fvw(vel) + gCp * o_nZW;
          if constexpr (TERRAIN) {
            double v13 = (0.5 * (sMX[s1][r][c] + sMX[s1][r][c - 1])) / D1(r, c);
            double v23 = (0.5 * (sMY[s1][r][c] + sMY[s1][r - 1][c])) / D1(r, c);
            if (k == KS) {
              v13 = (v13 + (0.5 * (sMX[s0][r][c] + sMX[s0][r][c - 1])) / D0(r, c)) * 0.5;
              v23 = (v23 + (0.5 * (sMY[s0][r][c] + sMY[s0][r - 1][c])) / D0(r, c)) * 0.5;
            }
            v13 = v13 * m.j13(I_XYZ, g + pl);
            v23 = v23 * m.j23(I_XYZ, g + pl);
            qW13 = v13 / m1 * fvw(v13);
            qW23 = v23 / m0 * fvw(v23);
          }
        }
        double Sr = 0.0, St = 0.0, Sw = 0.0;
        double dp1 = 0.0;
        if (live) {
          // continuity and theta (HEVI.F90:369-475, 588-657)
          double advcv = -(mZ - cmZ) * rcdz;
          double advch = -((xM[ty][tx + 1] - xM[ty][tx]) * rcdx + (yM[ty + 1][tx] - yM[ty][tx]) * rcdy);
          Sr = (advcv + advch) * m0 * m1 / gC + o_Dt;
          advcv = -(tZ - ctZ) * rcdz;
          advch = -((xT[ty][tx + 1] - xT[ty][tx]) * rcdx + (yT[ty + 1][tx] - yT[ty][tx]) * rcdy);
          St = (advcv + advch) * m0 * m1 / gC + o_Rt;
          if constexpr (PM_) dp1 = sDP[0][ty][tx];
          else dp1 = o_P0 + o_RT * (o_R - o_RR);
          if (full) {
            // momentum z, explicit part (HEVI.F90:486-577) and PT (HEVI.F90:691)
            if (k <= KE - 1) {
              double sv = qw - cqW;
              if constexpr (TERRAIN) sv = sv + qW13 - cW13 + qW23 - cW23;
              advcv = -(sv) * a.g.RFDZ[k];
              advch = -((xW[ty][tx + 1] - xW[ty][tx]) * rcdx + (yW[ty + 1][tx] - yW[ty][tx]) * rcdy) * m0 * m1;
              const double wdmp = -wdc * o_Z0;
              double sw = (advcv + advch) / gW + wdmp;
              if constexpr (DIVDMP) sw = sw + a.divdmp_coef / dtrk * (ld(a.DDIV, g + pl) - ld(a.DDIV, g)) * a.g.FDZ[k];
              Sw = sw + o_Wt;
              const double vel = ww[1];
              double PT;
              if (k == KS) PT = fv_lo<S>(pw[1], pw[2], pw[3], vel);
              else if (k == KE - 1) PT = fv_hi<S>(pw[0], pw[1], pw[2], vel);
              else PT = fv_int<S>(pw[0], pw[1], pw[2], pw[3], vel);
              sto(a.PT, g, PT);
              sto(a.tflx_hi, g, tZ);
              if constexpr (TERRAIN) sto(a.mflx_hi, g, mZ);  // flat: num_diff itself, read there again
            } else {
              sto(a.mflx_hi, g, 0.0);
              sto(a.tflx_hi, g, 0.0);
            }
            sto(a.DENS_RK, g, Sr);  // Sr/St wait in the outputs for hevi_columns
            sto(a.RHOT_RK, g, St);
            if (a.trSt) sto(a.trSt, g, St);
            if (k == KS) { sto(a.mflx_hi, g - pl, 0.0); sto(a.tflx_hi, g - pl, 0.0); }
            if (i == d.IS) {  // mflx_hi(Z) is also defined on the i = IS-1 column (HEVI.F90:370)
              sto(a.mflx_hi, g - 8, (k <= KE - 1) ? explZ(g - 8, p0 - 8, c - 1, o_nDw) : 0.0);
              if (k == KS) sto(a.mflx_hi, g - 8 - pl, 0.0);
            }
          }
          if (k > k0) {  // the right-hand side of row k-1 (HEVI.F90:716-727)
            const double rf = a.g.RFDZ[k - 1], czm = CDZ[k - 1];
            double h1, h2;  // F2H(k-1, .) of GSQRT at (x,y,z)
            if constexpr (TERRAIN) {
              h1 = czm * gCm / (czm * gCm + cz0 * gC);
              h2 = cz0 * gC / (czm * gCm + cz0 * gC);
            } else {
              h1 = czm / (czm + cz0);
              h2 = cz0 / (czm + cz0);
            }
            const double pg = -(dp1 + o_RT * dtrk * St - dp0 - rt0 * dtrk * st0) * rf * J33G / gWm
                            - GRAV * (h1 * ((D0(r, c) - o_RD) + Sr * dtrk) + h2 * (rd0 + sr0 * dtrk));
            sto(a.Sw, g - pl, ww[0] + dtrk * (pg + sw0));
          }
        }
        cmZ = mZ; ctZ = tZ; cqW = qw;
        pwm = pw[1];
        rt0 = o_RT; dp0 = dp1; st0 = St; sr0 = Sr; rd0 = D0(r, c) - o_RD; sw0 = Sw;
        if constexpr (TERRAIN) { cW13 = qW13; cW23 = qW23; gWm = gW; gCm = gC; }
      }
      if constexpr (PM_) {
        const double xw[4] = {xwm, sMX[s0][r][c], sMX[s1][r][c], sMX[s2][r][c]};
        const double yw[4] = {ywm, sMY[s0][r][c], sMY[s1][r][c], sMY[s2][r][c]};
        // z fluxes of MOMX and MOMY with their J13/J23 parts (UD3.F90:753-1039, 1173-1459)
        double qu = 0.0, qU13 = 0.0, qU23 = 0.0, qv = 0.0, qV13 = 0.0, qV23 = 0.0;
        const double gUWp = m.gs(I_UYW, g + pl), gXWp = m.gs(I_XVW, g + pl), gUp = m.gs(I_UYZ, g + pl), gVp = m.gs(I_XVZ, g + pl);
        const double j13c = m.j13(I_UYW, g), j23c = m.j23(I_XVW, g);
        double fu1 = 0.0, fu2 = 0.0, fv1 = 0.0, fv2 = 0.0;  // F2H(k, .) of GSQRT at (u,y,z) and (x,v,z)
        if constexpr (TERRAIN) { f2h(gU, gUp, fu1, fu2); f2h(gV, gVp, fv1, fv2); }
        if (k < KE && k <= k1) {
          const double dx0 = D0(r, c) + D0(r, c + 1), dx1 = D1(r, c) + D1(r, c + 1);
          const double dy0 = D0(r, c) + D0(r + 1, c), dy1 = D1(r, c) + D1(r + 1, c);
          auto fvx = [&](double vel) {
            if (k == KS) return fv_lo<S>(xw[1], xw[2], xw[3], vel);
            if (k == KE - 1) return fv_hi<S>(xw[0], xw[1], xw[2], vel);
            return fv_int<S>(xw[0], xw[1], xw[2], xw[3], vel);
          };
          auto fvy = [&](double vel) {
            if (k == KS) return fv_lo<S>(yw[1], yw[2], yw[3], vel);
            if (k == KE - 1) return fv_hi<S>(yw[0], yw[1], yw[2], vel);
            return fv_int<S>(yw[0], yw[1], yw[2], yw[3], vel);
          };
          {
            double f1, f2;
            f2h(gUW, gUWp, f1, f2);
            const double vel = (0.5 * (ww[1] + sW[s0][r][c + 1])) / (f1 * 0.5 * dx1 + f2 * 0.5 * dx0);
            qu = J33G * vel * fvx(vel) + gUW * o_nZX;
          }
          {
            double f1, f2;
            f2h(gXW, gXWp, f1, f2);
            const double vel = (0.5 * (ww[1] + sW[s0][r + 1][c])) / (f1 * 0.5 * dy1 + f2 * 0.5 * dy0);
            qv = J33G * vel * fvy(vel) + gXW * o_nZY;
          }
          if constexpr (TERRAIN) {
            {
              const double den = fu1 * 0.5 * dx1 + fu2 * 0.5 * dx0;
              double v = (fu1 * sMX[s1][r][c] + fu2 * sMX[s0][r][c]) / den;
              v = v * j13c;
              qU13 = v / m.mapf(p0, 1, I_UY) * fvx(v);
              v = (fu1 * 0.25 * (sMY[s1][r][c] + sMY[s1][r][c + 1] + sMY[s1][r - 1][c] + sMY[s1][r - 1][c + 1])
                 + fu2 * 0.25 * (sMY[s0][r][c] + sMY[s0][r][c + 1] + sMY[s0][r - 1][c] + sMY[s0][r - 1][c + 1])) / den;
              v = v * m.j23(I_UYW, g);
              qU23 = v / m.mapf(p0, 0, I_UY) * fvx(v);
            }
            {
              const double den = fv1 * 0.5 * dy1 + fv2 * 0.5 * dy0;
              double v = (fv1 * 0.25 * (sMX[s1][r][c] + sMX[s1][r][c - 1] + sMX[s1][r + 1][c] + sMX[s1][r + 1][c - 1])
                        + fv2 * 0.25 * (sMX[s0][r][c] + sMX[s0][r][c - 1] + sMX[s0][r + 1][c] + sMX[s0][r + 1][c - 1])) / den;
              v = v * m.j13(I_XVW, g);
              qV13 = v / m.mapf(p0, 1, I_XV) * fvy(v);
              v = (fv1 * sMY[s1][r][c] + fv2 * sMY[s0][r][c]) / den;
              v = v * j23c;
              qV23 = v / m.mapf(p0, 0, I_XV) * fvy(v);
            }
          }
        }
        if (full) {
          double MXn, MYn;
          {  // momentum x (HEVI.F90:816-927)
            double sv = qu - cqU;
            if constexpr (TERRAIN) sv = sv + qU13 - cU13 + qU23 - cU23;
            const double advcv = -(sv) * rcdz;
            const double m0u = m.mapf(p0, 0, I_UY), m1u = m.mapf(p0, 1, I_UY);
            const double advch = -((xU[ty][tx + 1] - xU[ty][tx]) * rfdx + (yU[ty + 1][tx] - yU[ty][tx]) * rcdy) * m0u * m1u;
            double pgh;
            if constexpr (TERRAIN) {
              // DPRES slots: k-1 at s2 (the ring's place of k+2), k at s0, k+1 at s1
              pgh = (m.gs(I_XYZ, g + 8) * sDP[s0][ty][tx + 1] - gC * sDP[s0][ty][tx]) * rfdx;
              pgh = pgh + (j13c * 0.5 * (fu1 * (sDP[s1][ty][tx + 1] + sDP[s1][ty][tx]) + fu2 * (sDP[s0][ty][tx + 1] + sDP[s0][ty][tx]))
                           - j13m * 0.5 * (fu1 * (sDP[s0][ty][tx + 1] + sDP[s0][ty][tx]) + fu2 * (sDP[s2][ty][tx + 1] + sDP[s2][ty][tx])))
                          * rcdz;
            } else {
              pgh = (sDP[0][ty][tx + 1] - sDP[0][ty][tx]) * rfdx;
            }
            const double pg = pgh * m0u;
            double t = (advcv + advch - pg) / gU;
            if (a.has_coriolis || TERRAIN) {
              double cf = 0.125 * (ld(a.CORIOLI, p0 + 8) + ld(a.CORIOLI, p0))
                        * (sMY[s0][r][c + 1] + sMY[s0][r][c] + sMY[s0][r - 1][c + 1] + sMY[s0][r - 1][c]);
              if constexpr (TERRAIN) {
                const double sy = sMY[s0][r][c] + sMY[s0][r - 1][c] + sMY[s0][r][c + 1] + sMY[s0][r - 1][c + 1];
                cf = cf + 0.25 * m0u * m1u * sy
                        * (sy * 0.25 * (1.0 / m.mapf(p0 + 8, 1, I_XY) - 1.0 / m1) * rfdx
                           - xw[1] * (1.0 / m.mapf(p0, 0, I_UV) - 1.0 / m.mapf(p0 - row8, 0, I_UV)) * rcdy)
                        * 2.0 / (D0(r, c + 1) + D0(r, c));
              }
              t = t + cf;
            }
            if constexpr (DIVDMP)
              t = t + a.divdmp_coef / dtrk * (ld(a.DDIV, g + 8) / m.mapf(p0 + 8, 1, I_XY) - ld(a.DDIV, g) / m0) * m0u * m1u * a.g.FDX[i];
            MXn = o_X0 + dtrk * (t + o_Xt);
          }
          {  // momentum y (HEVI.F90:936-1047)
            double sv = qv - cqV;
            if constexpr (TERRAIN) sv = sv + qV13 - cV13 + qV23 - cV23;
            const double advcv = -(sv) * rcdz;
            const double m0v = m.mapf(p0, 0, I_XV), m1v = m.mapf(p0, 1, I_XV);
            const double advch = -((xV[ty][tx + 1] - xV[ty][tx]) * rcdx + (yV[ty + 1][tx] - yV[ty][tx]) * rfdy) * m0v * m1v;
            double pgh;
            if constexpr (TERRAIN) {
              const double czm = CDZ[k - 1];
              const double fm1 = czm * gVm / (czm * gVm + cz0 * gV), fm2 = cz0 * gV / (czm * gVm + cz0 * gV);  // F2H(k-1, .)
              pgh = (m.gs(I_XYZ, g + row8) * sDP[s0][ty + 1][tx] - gC * sDP[s0][ty][tx]) * rfdy;
              pgh = pgh + (j23c * 0.5 * (fv1 * (sDP[s1][ty + 1][tx] + sDP[s1][ty][tx]) + fv2 * (sDP[s0][ty + 1][tx] + sDP[s0][ty][tx]))
                           - j23m * 0.5 * (fm1 * (sDP[s0][ty + 1][tx] + sDP[s0][ty][tx]) + fm2 * (sDP[s2][ty + 1][tx] + sDP[s2][ty][tx])))
                          * rcdz;
            } else {
              pgh = (sDP[0][ty + 1][tx] - sDP[0][ty][tx]) * rfdy;
            }
            const double pg = pgh * m1v;
            double t = (advcv + advch - pg) / gV;
            if (a.has_coriolis || TERRAIN) {
              double cf = -0.125 * (ld(a.CORIOLI, p0 + row8) + ld(a.CORIOLI, p0))
                        * (sMX[s0][r + 1][c] + sMX[s0][r][c] + sMX[s0][r + 1][c - 1] + sMX[s0][r][c - 1]);
              if constexpr (TERRAIN) {
                const double sx = sMX[s0][r][c] + sMX[s0][r][c - 1] + sMX[s0][r + 1][c] + sMX[s0][r + 1][c - 1];
                cf = cf - 0.25 * m0v * m1v * sx
                        * (yw[1] * (1.0 / m.mapf(p0, 1, I_UV) - 1.0 / m.mapf(p0 - 8, 1, I_UV)) * rcdx
                           - 0.25 * sx * (1.0 / m.mapf(p0 + row8, 0, I_XY) - 1.0 / m0) * rfdy)
                        * 2.0 / (D0(r + 1, c) + D0(r, c));
              }
              t = t + cf;
            }
            if constexpr (DIVDMP)
              t = t + a.divdmp_coef / dtrk * (ld(a.DDIV, g + row8) / m.mapf(p0 + row8, 0, I_XY) - ld(a.DDIV, g) / m0) * m0v * m1v * a.g.FDY[j];
            MYn = o_Y0 + dtrk * (t + o_Yt);
          }
          if constexpr (CMB) {
            const double mx = rk4c(cmx[0], cmx[1], cmx[2], MXn, o_X0);
            const double my = rk4c(cmy[0], cmy[1], cmy[2], MYn, o_Y0);
            sto(a.st[2], g, mx);
            sto(a.st[3], g, my);
            if (k == KS || k == KE) {  // ghost levels copy the combined KS / KE value
              const int lo = (k == KS) ? 0 : KE + 1, hi = (k == KS) ? KS - 1 : d.KA - 1;
              for (int kk = lo; kk <= hi; ++kk) { sto(a.st[2], p0 + pl * (unsigned)kk, mx); sto(a.st[3], p0 + pl * (unsigned)kk, my); }
            }
          } else {
            sto(a.MOMX_RK, g, MXn);
            sto(a.MOMY_RK, g, MYn);
          }
        }
        cqU = qu; cqV = qv;
        xwm = xw[1]; ywm = yw[1];
        if constexpr (TERRAIN) {
          cU13 = qU13; cU23 = qU23; cV13 = qV13; cV23 = qV23;
          gUW = gUWp; gXW = gXWp; gVm = gV; gU = gUp; gV = gVp; j13m = j13c; j23m = j23c;
        }
      }
      wwm = ww[1];
      if constexpr (TERRAIN) gC = gCp;
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// The columns' tridiagonal systems.  COLS columns of one row per block; thread
// (tx, ty) builds the rows of 4 levels of column tx into LDS (F1, F2, F3 and
// the right-hand side, COLS apart), the threads ty = 0 sweep their columns
// down and up in LDS, and every thread updates its 4 levels from C.  The sweep
// is a serial chain of a division per level; in LDS it costs about 5 us for 64
// levels, and the loads and stores around it are wide and independent.  (One
// thread per column marching both ways waited on memory level by level: 36 us
// against 159 at 128x128x64, 388 against 489 at 320x320x96.)
constexpr int SOLVE_L = 4;          // levels per thread
constexpr int SOLVE_LDS = 131072;   // bytes of LDS a block may take: 32 B per row and column
constexpr int SOLVE_KMAX = 1024 * SOLVE_L;  // levels at one column a block

template <bool TERRAIN, bool CMB, int COLS>
__global__ void __launch_bounds__(1024) hevi_columns(HeviArgs a, unsigned ni, unsigned nblocks) {
  extern __shared__ double sh[];
  const Dims& d = a.d;
  const int KS = d.KS, KE = d.KE, nr = KE - KS;  // rows 0..nr-1 are levels KS..KE-1
  double* F1 = sh;
  double* F2 = F1 + nr * COLS;
  double* F3 = F2 + nr * COLS;
  double* Cs = F3 + nr * COLS;
  const unsigned lb = xcd_block(blockIdx.x, nblocks);
  const int tx = threadIdx.x % COLS, ty = threadIdx.x / COLS;
  const int i = d.IS + (int)(lb % ni) * COLS + tx, j = d.JS + (int)(lb / ni);
  const bool own = i <= d.IE;
  const unsigned pl = (unsigned)d.pl * 8u, p0 = (unsigned)((own ? i : d.IS) + d.IA * j) * 8u;  // byte offsets
  MetO<TERRAIN> m;
  m.G = a.GSQRT; m.J13 = a.J13G; m.J23 = a.J23G; m.MAPF = a.MAPF; m.n3 = d.n3; m.pl = d.pl; m.IA = d.IA;
  const double* CDZ = a.g.CDZ; const double* RCDZ = a.g.RCDZ; const double* RFDZ = a.g.RFDZ;
  const double dtrk = a.dtrk, J33G = a.J33G;
  const int ka = KS + ty * SOLVE_L;  // the thread's first level
  // levels of the thread, kept for the update
  double pt[SOLVE_L + 1], ptm = 0.0;
  if (own) {
    double rt[SOLVE_L + 1], ck[SOLVE_L];
#pragma unroll
    for (int q = 0; q <= SOLVE_L; ++q) {
      rt[q] = ld(a.RT2P, p0 + pl * (unsigned)min(ka + q, KE));
      pt[q] = ld(a.PT, p0 + pl * (unsigned)min(ka + q, KE - 1));
    }
    if (ty > 0) ptm = ld(a.PT, p0 + pl * (unsigned)min(ka - 1, KE - 1));
#pragma unroll
    for (int q = 0; q < SOLVE_L; ++q) ck[q] = ld(a.Sw, p0 + pl * (unsigned)min(ka + q, KE - 1));
#pragma unroll
    for (int q = 0; q < SOLVE_L; ++q) {
      const int r = ka + q;
      if (r > KE - 1) break;
      const unsigned p = p0 + pl * (unsigned)r;
      const double gw = m.gs(I_XYW, p), g0 = m.gs(I_XYZ, p), g1 = m.gs(I_XYZ, p + pl);
      const double A0 = dtrk * dtrk * J33G * RCDZ[r] * rt[q] * J33G / g0;
      const double A1 = dtrk * dtrk * J33G * RCDZ[r + 1] * rt[q + 1] * J33G / g1;
      const double B = GRAV * (dtrk * dtrk) * J33G / (CDZ[r + 1] + CDZ[r]);
      const double pt1 = r < KE - 1 ? pt[q + 1] : 0.0;
      const double ptb = q > 0 ? pt[q - 1] : ptm;
      const int o = (r - KS) * COLS + tx;
      F1[o] = -(pt1 * RFDZ[r] * A1 + B) / gw;
      F2[o] = 1.0 + (pt[q] * RFDZ[r] * (A1 + A0)) / gw;
      F3[o] = -(ptb * RFDZ[r] * A0 - B) / gw;
      Cs[o] = ck[q];
    }
  }
  __syncthreads();
  if (ty == 0 && own) {  // Thomas sweeps (HEVI.F90:1092-1127); e and f take the places of F1 and C
    double e, f;
    {
      const double rdenom = 1.0 / F2[tx];
      e = -F1[tx] * rdenom;
      f = Cs[tx] * rdenom;
      F1[tx] = e; Cs[tx] = f;
    }
    int o = COLS + tx;
    double n1 = F1[o], n2 = F2[o], n3 = F3[o], nc = Cs[o];
    for (int r = 1; r < nr - 1; ++r, o += COLS) {
      const double c1 = n1, c2 = n2, c3 = n3, cc = nc;
      n1 = F1[o + COLS]; n2 = F2[o + COLS]; n3 = F3[o + COLS]; nc = Cs[o + COLS];
      const double rdenom = 1.0 / (c2 + c3 * e);
      const double en = -c1 * rdenom;
      f = (cc - c3 * f) * rdenom;
      e = en;
      F1[o] = e; Cs[o] = f;
    }
    double Cn = (nc - n3 * f) / (n2 + n3 * e);
    Cs[o] = Cn;
    for (int r = nr - 2; r >= 0; --r) {
      o -= COLS;
      Cn = F1[o] * Cn + Cs[o];
      Cs[o] = Cn;
    }
  }
  __syncthreads();
  if (!own) return;

  // ---- updates (HEVI.F90:728-790) ----
  const double M12 = m.mapf(p0, 0, I_XY) * m.mapf(p0, 1, I_XY);
  auto put_state = [&](int v, unsigned q, double val, double s0v, int k) {
    if constexpr (CMB) {
      const double c = (v == 1 && k == KE) ? 0.0 : rk4c(ld(a.c1[v], q), ld(a.c2[v], q), ld(a.c3[v], q), val, s0v);
      sto(a.st[v], q, c);
      if (k == KS || k == KE) {
        const int lo = (k == KS) ? 0 : KE + 1, hi = (k == KS) ? KS - 1 : d.KA - 1;
        for (int kk = lo; kk <= hi; ++kk) sto(a.st[v], p0 + pl * (unsigned)kk, (v == 1) ? 0.0 : c);
      }
    } else {
      double* o = v == 0 ? a.DENS_RK : (v == 1 ? a.MOMZ_RK : a.RHOT_RK);
      sto(o, q, val);
    }
  };
#pragma unroll
  for (int q = 0; q < SOLVE_L; ++q) {
    const int k = ka + q;
    if (k > KE) break;
    const unsigned p = p0 + pl * (unsigned)k;
    const int o = (k - KS) * COLS + tx;
    const double g0 = m.gs(I_XYZ, p);
    const double Cm = k > KS ? Cs[o - COLS] : 0.0, pm = q > 0 ? pt[q - 1] : ptm;
    const double d0 = ld(a.DENS0, p), r0 = ld(a.RHOT0, p);
    const double sr = ld(a.DENS_RK, p), st = ld(a.RHOT_RK, p);
    double advD, advT;
    if (k == KE) {
      advD = Cm * J33G * RCDZ[k] / g0;
      advT = Cm * pm * J33G * RCDZ[k] / g0;
      if constexpr (CMB) {
        sto(a.mflx_av, p, rk4f(ld(a.cm[0], p), ld(a.cm[1], p), ld(a.cm[2], p), 0.0));
        sto(a.tflx_av, p, rk4f(ld(a.ct[0], p), ld(a.ct[1], p), ld(a.ct[2], p), 0.0));
      }
      put_state(1, p, 0.0, 0.0, k);
    } else {
      const double Ck = Cs[o];
      if (k == KS) {
        advD = -Ck * J33G * RCDZ[k] / g0;
        advT = -Ck * pt[q] * J33G * RCDZ[k] / g0;
        if constexpr (!CMB) sto(a.MOMZ_RK, p - pl, 0.0);
      } else {
        advD = -(Ck - Cm) * J33G * RCDZ[k] / g0;
        advT = -(Ck * pt[q] - Cm * pm) * J33G * RCDZ[k] / g0;
      }
      const double me = TERRAIN ? ld(a.mflx_hi, p) : ld(a.num_diff + d.n3 * (size_t)(I_DENS + 5 * ZDIR), p);
      const double mv = me + J33G * Ck / (M12);
      const double tv = ld(a.tflx_hi, p) + J33G * Ck * pt[q] / (M12);
      if constexpr (CMB) {
        sto(a.mflx_av, p, rk4f(ld(a.cm[0], p), ld(a.cm[1], p), ld(a.cm[2], p), mv));
        sto(a.tflx_av, p, rk4f(ld(a.ct[0], p), ld(a.ct[1], p), ld(a.ct[2], p), tv));
      } else {
        sto(a.mflx_hi, p, mv);
        sto(a.tflx_hi, p, tv);
      }
      const double z0 = ld(a.MOMZ0, p);
      put_state(1, p, z0 + (Ck - ld(a.MOMZ, p)), z0, k);
      if (a.trCp) sto(a.trCp, p, Ck);
    }
    put_state(0, p, d0 + dtrk * (advD + sr), d0, k);
    put_state(4, p, r0 + dtrk * (advT + st), r0, k);
  }
}

// Columns per block of hevi_columns: the most, up to 32, that bound a block's
// threads and LDS, above 64 levels up to 16, so that two blocks fit a CU, and
// down to 8 to give every CU a block.  More than 512 levels leave room for
// fewer, whose loads fill less of a cache line: short step over terrain at
// 64x64x600 4.9 ms and 64x64x1024 8.4 (4 columns), against 110 and 188 in the
// one-launch march (hevi_march).
constexpr int columns_per_block(int imax, int jmax, int kmax, int ncu) {
  const int ny = (kmax + SOLVE_L - 1) / SOLVE_L;
  int cols = 32;
  while (cols > 1 && (cols * ny > 1024 || (kmax - 1) * cols * 32 > SOLVE_LDS || (cols > 16 && kmax > 64) ||
                      (cols > 8 && ((imax + cols - 1) / cols) * jmax < ncu)))
    cols /= 2;
  return cols;
}
// every depth that hevi_split_fits takes, on grids of many columns and of few
constexpr bool column_blocks_fit() {
  for (int kmax = 4; kmax <= SOLVE_KMAX; ++kmax)
    for (int n = 2; n <= 4096; n *= 16) {
      const int cols = columns_per_block(n, n, kmax, 256);
      if (cols * ((kmax + SOLVE_L - 1) / SOLVE_L) > 1024 || (kmax - 1) * cols * 32 > SOLVE_LDS) return false;
    }
  return true;
}
static_assert(column_blocks_fit(), "a block of hevi_columns exceeds its threads or LDS");

// one column's tridiagonal rows fit a block, a field's byte offsets 32 bits
bool hevi_split_fits(const Dims& d) { return d.KE - d.KS + 1 <= SOLVE_KMAX && d.n3 < TILE_MAX_N3; }

// Tiles of TI x 8 columns.  64 columns re-read the smaller halo (1.59 cells per
// column against 1.69) and are the faster from about half a tile per CU on; 32
// columns give small grids more blocks.
static int etiles(int imax, int jmax, int TI) { return ((imax + TI - 1) / TI) * ((jmax + 7) / 8); }

template <int S, bool TERRAIN, bool DIVDMP, bool CMB, int TI>
static void launch_etile(const HeviArgs& a, hipStream_t s) {
  constexpr int TJ = 8;
  const Dims& d = a.d;
  const int imax = d.IE - d.IS + 1, jmax = d.JE - d.JS + 1, kmax = d.KE - d.KS + 1;
  const unsigned ni = (unsigned)((imax + TI - 1) / TI), nt = (unsigned)etiles(imax, jmax, TI);
  // levels per segment (SCALE_HIP_TERRAIN_SEG sets them): a segment pays about
  // two levels' work for its ring, windows and end levels; 512 threads a CU
  const char* e = getenv("SCALE_HIP_TERRAIN_SEG");
  const int L = e && atoi(e) > 0 ? atoi(e) : seg_levels(nt, kmax, (64u / TI) * (unsigned)a.ctx->ncu, 2.0);
  const unsigned nb = nt * (unsigned)((kmax + L - 1) / L);
  const dim3 g(nb), b(TI * TJ);
  if constexpr (TERRAIN) {
    hipLaunchKernelGGL((hevi_etile<S, true, DIVDMP, CMB, P_T, TI, TJ>), g, b, 0, s, a, ni, nt, nb, L);
    hipLaunchKernelGGL((hevi_etile<S, true, DIVDMP, CMB, P_M, TI, TJ>), g, b, 0, s, a, ni, nt, nb, L);
  } else {
    hipLaunchKernelGGL((hevi_etile<S, false, DIVDMP, CMB, P_T | P_M, TI, TJ>), g, b, 0, s, a, ni, nt, nb, L);
  }
}

template <int S, bool TERRAIN, bool DIVDMP, bool CMB>
static hipError_t launch(const HeviArgs& a, hipStream_t s) {
  const Dims& d = a.d;
  const int imax = d.IE - d.IS + 1, jmax = d.JE - d.JS + 1, kmax = d.KE - d.KS + 1;
  if (2 * etiles(imax, jmax, 64) >= a.ctx->ncu) launch_etile<S, TERRAIN, DIVDMP, CMB, 64>(a, s);
  else launch_etile<S, TERRAIN, DIVDMP, CMB, 32>(a, s);
  const int ny = (kmax + SOLVE_L - 1) / SOLVE_L, cols = columns_per_block(imax, jmax, kmax, a.ctx->ncu);
  const unsigned ni = (unsigned)((imax + cols - 1) / cols), nb = ni * (unsigned)jmax;
  const unsigned lds = (unsigned)((kmax - 1) * cols * 32);
  const dim3 b((unsigned)(cols * ny));
  switch (cols) {
    case 32: hipLaunchKernelGGL((hevi_columns<TERRAIN, CMB, 32>), dim3(nb), b, lds, s, a, ni, nb); break;
    case 16: hipLaunchKernelGGL((hevi_columns<TERRAIN, CMB, 16>), dim3(nb), b, lds, s, a, ni, nb); break;
    case 8: hipLaunchKernelGGL((hevi_columns<TERRAIN, CMB, 8>), dim3(nb), b, lds, s, a, ni, nb); break;
    case 4: hipLaunchKernelGGL((hevi_columns<TERRAIN, CMB, 4>), dim3(nb), b, lds, s, a, ni, nb); break;
    case 2: hipLaunchKernelGGL((hevi_columns<TERRAIN, CMB, 2>), dim3(nb), b, lds, s, a, ni, nb); break;
    default: hipLaunchKernelGGL((hevi_columns<TERRAIN, CMB, 1>), dim3(nb), b, lds, s, a, ni, nb);
  }
  return hipGetLastError();
}

template <int S, bool TERRAIN>
static hipError_t launch_d(const HeviArgs& a, bool divdmp, bool cmb, hipStream_t s) {
  if (divdmp) return cmb ? launch<S, TERRAIN, true, true>(a, s) : launch<S, TERRAIN, true, false>(a, s);
  return cmb ? launch<S, TERRAIN, false, true>(a, s) : launch<S, TERRAIN, false, false>(a, s);
}

hipError_t hevi_split(const HeviArgs& a, int scheme, bool terrain, bool divdmp, bool cmb, hipStream_t s) {
  if (!hevi_split_fits(a.d)) return hipErrorNotSupported;
  if (scheme == UD3) return terrain ? launch_d<UD3, true>(a, divdmp, cmb, s) : launch_d<UD3, false>(a, divdmp, cmb, s);
  return terrain ? launch_d<CD4, true>(a, divdmp, cmb, s) : launch_d<CD4, false>(a, divdmp, cmb, s);
}

}  // namespace shp
