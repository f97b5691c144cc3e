// tracer_tile.hip -- the tracer stage on LDS tiles, flat or general metrics, for
// the tracer schemes whose faces read two cells on each side (UD3, CD4,
// UD3KOREN1993, UD1, CD2).  Same results as the per-point kernels of
// tracer.hip, bit for bit: every expression is the same, only the places the
// operands come from differ.
//
// Reference: ATMOS_DYN_Tstep_tracer_fvm_heve,
//   scalelib/src/atmos-rm/dynamics/scale_atmos_dyn_tstep_tracer_fvm_heve.F90:72-242,
// and ATMOS_DYN_fct, scalelib/src/atmos-rm/dynamics/scale_atmos_dyn_common.F90:1922-2734.
//
// A block owns 64 (i) x TJ (j) columns and marches a segment of levels upward
// (the segments give a grid of few tiles blocks for every CU).  Per level it
// stages the planes it reads at neighbours in LDS (with a ring of one or two
// cells); a thread finishes one cell, whose horizontal faces it evaluates
// itself and whose lower z face it carries in registers.
//   trt_ratio   FCT pass 1: the low-order field phi_lo on the tile and a
//               one-cell ring (kept in LDS, three levels), the anti-diffusive
//               fluxes, P+/P-, the along-stream or 7-point bounds and R+/R-
//   [periodic fill of R+/R-]
//   trt_update  FCT pass 2: limited anti-diffusive fluxes and the update; or
//               the whole stage without FCT
#include "common.h"
#include "fct.h"
#include "shp_internal.h"
#include "batch.h"

namespace shp {

struct TtArgs {  // nd and RHOQ_t may be null: zeros (as in TrArgs)
  Dims d;
  const double *QTRC, *QTRC0, *RHOQ_t, *DENS0, *DENS, *mflx, *nd;
  size_t nds;  // distance between the z, x and y components of nd
  const double *RCDZ, *RCDX, *RCDY;
  double dtl;
  double* QTRCo;
  double *rjpls, *rjmns;
  const double *GSQRT, *MAPF;  // general metrics: GSQRT (7 components, n3 apart), MAPF(IA,JA,2) at XY
  int dens_mode;               // stage without FCT: its density (TracerIO)
};

// Plane (k) of F on the rows j0m.. and columns i0m.. of an H x W LDS array;
// points outside the array extents (partial tiles) read as 0 and are never used.
template <int H, int W>
__device__ __forceinline__ void tt_load(double (*s)[W], const double* F, const Dims& d, int k, int i0m, int j0m, int tid,
                                        int nthr) {
  const size_t base = d.pl * (size_t)k;
  for (int t = tid; t < H * W; t += nthr) {
    const int r = t / W, c = t - r * W;
    const int i = i0m + c, j = j0m + r;
    s[r][c] = (i < d.IA && j < d.JA) ? F[base + (size_t)i + (size_t)d.IA * j] : 0.0;
  }
}

// high-order face value times velocity plus num_diff with its metric factor
// (TrOps::hX/hY/hZ of the per-point kernels); q holds the four cells around the face
template <int S>
__device__ __forceinline__ double tt_hflux(double vel, double qm1, double q0, double q1, double q2, double nd) {
  if constexpr (S == UD1) return vel * fv_int<UD1>(0.0, q0, q1, 0.0, vel);
  return vel * fv_int<S>(qm1, q0, q1, q2, vel) + nd;
}
__device__ __forceinline__ double tt_lflux(double vel, double q0, double q1) {
  return vel * fv_int<UD1>(0.0, q0, q1, 0.0, vel);
}

// vertical high-order flux through face kk of a column; w holds val(kk-1..kk+2)
template <int S>
__device__ __forceinline__ double tt_hz(const Dims& d, int kk, double vel, const double* w, double nd) {
  if (kk == d.KS - 1 || kk == d.KE) return 0.0;
  double fv;
  if (kk == d.KS) fv = fv_lo<S>(w[1], w[2], w[3], vel);
  else if (kk == d.KE - 1) fv = fv_hi<S>(w[0], w[1], w[2], vel);
  else fv = fv_int<S>(w[0], w[1], w[2], w[3], vel);
  if constexpr (S == UD1) return vel * fv;
  return vel * fv + nd;
}

// ---- FCT pass 1: phi_lo (ring of one), anti-diffusive fluxes, R+/R- ------------
// each pass is a body over tile lb of a grid ni_tiles tiles across, run by
// its kernel once per block or, for an ensemble, by trt_batch over a table
// of members
//
// Bound by FP64 instruction issue (the along-stream bounds are six divisions
// and 112 multiply-adds of LDS operands): at three wavefronts per SIMD each
// issues for 30 % of its time.  A thread owns a cell: phi_lo, the faces and P+/P- of level u,
// then, a barrier later, R+/R- of level u - 1, for which it keeps six values
// in registers; the ring's cells are one item each of the first threads, and
// every load of a level is issued before its first barrier.  Sharing the
// faces through LDS instead needs a second slot of them and items for the
// tile's west and south faces: 0.36 ms a pass at 320x320x96 against 0.34, and
// 0.50 with one list of faces and ring cells that the threads took in turn.
// A tile of 8 rows (fewer ring cells, but one block of 8 wavefronts a CU):
// 0.38 ms, and 0.039 against 0.045 at 128x128x64.  Held to four wavefronts
// per SIMD it spills 23 registers: 0.47 ms.
template <bool TER>
struct TtCell {  // what phi_lo of a cell reads
  double mx, mxm, my, mym, mz, D0, D, g;
};
template <int S, int TJ, bool VECT, bool TER>
__device__ __forceinline__ void trt_ratio_body(const TtArgs& a, unsigned lb, unsigned ni_tiles, int k0, int k1) {
  constexpr int W2 = 68, H2 = TJ + 4, W1 = 66, H1 = TJ + 2, NT = 64 * TJ, NQ = (H2 * W2 + NT - 1) / NT;
  constexpr int NRING = 2 * W1 + 2 * TJ;  // ring cells
  static_assert(NRING <= NT, "one rim item a thread");
  __shared__ double sQ0[5][H2][W2];  // QTRC0, two-cell ring, levels u-2..u+1 (slot = level % 5)
  __shared__ double sQ[H2][W2];      // QTRC at level u, two-cell ring
  __shared__ double sPL[3][H1][W1];  // phi_lo, one-cell ring, levels u-2..u (slot = level % 3)
  const Dims& d = a.d;
  const int KS = d.KS, KE = d.KE;
  const int i0 = d.IS + 64 * (int)(lb % ni_tiles), j0 = d.JS + TJ * (int)(lb / ni_tiles);
  const int tx = threadIdx.x, ty = threadIdx.y, tid = tx + 64 * ty;
  const int i = i0 + tx, j = j0 + ty;
  const bool act = i <= d.IE && j <= d.JE;            // R+/R- and the faces
  const bool pact = i <= d.IE + 1 && j <= d.JE + 1;   // phi_lo
  const double dt = a.dtl;
  const unsigned plb = 8u * (unsigned)d.pl;  // bytes of a level; points are 32-bit byte offsets
  const unsigned IA = (unsigned)d.IA;
  const unsigned qc = 8u * (pact ? (unsigned)i + IA * (unsigned)j : (unsigned)d.IS + IA * (unsigned)d.JS);
  const double rdx = a.RCDX[pact ? i : d.IS], rdy = a.RCDY[pact ? j : d.JS];
  double m1 = 1.0, m2 = 1.0, em1 = 1.0, em2 = 1.0;
  // the rim item: ring cell (er, ec) of the first threads
  bool rim = tid < NRING;
  int er = 0, ec = 0;
  if (rim) {
    if (tid < 2 * W1) { er = tid < W1 ? 0 : H1 - 1; ec = tid < W1 ? tid : tid - W1; }
    else { er = 1 + (tid - 2 * W1) / 2; ec = (tid & 1) * (W1 - 1); }
    rim = i0 - 1 + ec <= d.IE + 1 && j0 - 1 + er <= d.JE + 1;
  }
  const unsigned qe = rim ? 8u * ((unsigned)(i0 - 1 + ec) + IA * (unsigned)(j0 - 1 + er)) : qc;
  const double erdx = rim ? a.RCDX[i0 - 1 + ec] : 0.0, erdy = rim ? a.RCDY[j0 - 1 + er] : 0.0;
  if constexpr (TER) { m1 = ld(a.MAPF, qc); m2 = ld(a.MAPF + d.pl, qc); em1 = ld(a.MAPF, qe); em2 = ld(a.MAPF + d.pl, qe); }
  const double *mZ = a.mflx, *mX = mZ + d.n3, *mY = mX + d.n3;
  auto cell = [&](unsigned o) {
    TtCell<TER> v;
    v.mx = ld(mX, o); v.mxm = ld(mX, o - 8u);
    v.my = ld(mY, o); v.mym = ld(mY, o - 8u * IA);
    v.mz = ld(mZ, o);
    v.D0 = ld(a.DENS0, o); v.D = ld(a.DENS, o);
    v.g = TER ? ld(a.GSQRT, o) : 1.0;
    return v;
  };
  auto nd = [&](unsigned o, int dir, int c) {
    double v = ld(a.nd + a.nds * (size_t)dir, o);
    if constexpr (TER) v = ld(a.GSQRT + d.n3 * (size_t)c, o) * v;
    return v;
  };
  // phi_lo of ring cell (r, c) at level u (COMMON.F90:2033-2045); lf: the
  // low-order fluxes west, east, south and north; lz: the flux through its
  // bottom face, replaced by that through its top face
  auto phi = [&](int u, int r, int c, const TtCell<TER>& v, double rx, double ry, double f1, double f2, double* lf,
                 double& lz) {
    const double(*Q1)[W2] = sQ0[u % 5];
    const int c2 = c + 1, r2 = r + 1;
    const double q = Q1[r2][c2];
    const double lzu = (u == KE) ? 0.0 : tt_lflux(v.mz, q, sQ0[(u + 1) % 5][r2][c2]);
    lf[0] = tt_lflux(v.mxm, Q1[r2][c2 - 1], q);
    lf[1] = tt_lflux(v.mx, q, Q1[r2][c2 + 1]);
    lf[2] = tt_lflux(v.mym, Q1[r2 - 1][c2], q);
    lf[3] = tt_lflux(v.my, q, Q1[r2 + 1][c2]);
    double t = -((lzu - lz) * a.RCDZ[u] + (lf[1] - lf[0]) * rx + (lf[3] - lf[2]) * ry);
    if constexpr (TER) t = t * f1 * f2 / v.g;
    sPL[u % 3][r][c] = (q * v.D0 + dt * t) / v.D;
    lz = lzu;
  };

  // levels u of faces and phi_lo from one below the segment to one above it;
  // level k = u - 1 of R+/R- follows
  const int kq = k0 > KS ? k0 - 1 : KS;
  tt_load<H2, W2>(sQ0[kq % 5], a.QTRC0, d, kq, i0 - 2, j0 - 2, tid, NT);
  double w[4];  // QTRC of the own column, levels u-1..u+2
  for (int m = 0; m < 4; ++m) w[m] = ld(a.QTRC, qc + plb * (unsigned)(kq - 1 + m));
  double lz = 0.0, elz = 0.0;  // low-order fluxes through the bottom face of level u
  if (kq > KS) {
    const unsigned b = plb * (unsigned)(kq - 1), o = qc + b, oe = qe + b;
    lz = tt_lflux(ld(mZ, o), ld(a.QTRC0, o), ld(a.QTRC0, o + plb));
    if (rim) elz = tt_lflux(ld(mZ, oe), ld(a.QTRC0, oe), ld(a.QTRC0, oe + plb));
  }
  // anti-diffusive and mass flux through that face (first used at k0, after level kq)
  double azm = 0.0, mzm = 0.0;
  // of the own cell, level k: P+, P-, velocities of the along-stream bounds, density
  double pp = 0.0, pm = 0.0, rw = 0.0, ru = 0.0, rv = 0.0, D = 1.0;
  for (int u = kq; u <= k1 + 1; ++u) {
    double ppu = 0.0, pmu = 0.0, rwu = 0.0, ruu = 0.0, rvu = 0.0, Du = 1.0;
    if (u <= KE) {
      // every load of the level before its first barrier
      double tQ[NQ], tP[NQ];
      const unsigned b = plb * (unsigned)u, b1 = u < KE ? b + plb : b, oc = qc + b, oe = qe + b;
#pragma unroll
      for (int h = 0; h < NQ; ++h) {
        const int q = tid + h * NT, r = q / W2, c = q - r * W2;
        const int ii = i0 - 2 + c, jj = j0 - 2 + r;
        const bool ok = q < H2 * W2 && ii < d.IA && jj < d.JA;  // (partial tiles: the rest is never used)
        const unsigned o = ok ? 8u * ((unsigned)ii + IA * (unsigned)jj) : 0u;
        tQ[h] = ld(a.QTRC, o + b);
        tP[h] = ld(a.QTRC0, o + b1);
      }
      const TtCell<TER> v = cell(oc);
      TtCell<TER> e;
      if (rim) e = cell(oe);
      double nz = 0.0, nx = 0.0, nxm = 0.0, ny = 0.0, nym = 0.0;
      if (a.nd) {
        nz = nd(oc, 0, I_XYW);
        nx = nd(oc, 1, I_UYZ); nxm = nd(oc - 8u, 1, I_UYZ);
        ny = nd(oc, 2, I_XVZ); nym = nd(oc - 8u * IA, 2, I_XVZ);
      }
      const double wn = ld(a.QTRC, qc + plb * (unsigned)min(u + 3, d.KA - 1));
#pragma unroll
      for (int h = 0; h < NQ; ++h) {
        const int q = tid + h * NT, r = q / W2, c = q - r * W2;
        if (q < H2 * W2) {
          sQ[r][c] = tQ[h];
          if (u + 1 <= KE) sQ0[(u + 1) % 5][r][c] = tP[h];
        }
      }
      __syncthreads();
      double lf[4];
      if (pact) {
        const int c = tx + 2, r = ty + 2;
        phi(u, ty + 1, tx + 1, v, rdx, rdy, m1, m2, lf, lz);
        // anti-diffusive fluxes through the cell's faces, P+ and P-
        const double q = sQ[r][c], qw = sQ[r][c - 1], qe1 = sQ[r][c + 1], qs = sQ[r - 1][c], qn = sQ[r + 1][c];
        const double ax = tt_hflux<S>(v.mx, qw, q, qe1, sQ[r][c + 2], nx) - lf[1];
        const double axm = tt_hflux<S>(v.mxm, sQ[r][c - 2], qw, q, qe1, nxm) - lf[0];
        const double ay = tt_hflux<S>(v.my, qs, q, qn, sQ[r + 2][c], ny) - lf[3];
        const double aym = tt_hflux<S>(v.mym, sQ[r - 2][c], qs, q, qn, nym) - lf[2];
        const double az = u != KE ? tt_hz<S>(d, u, v.mz, w, nz) - lz : 0.0;
        ppu = dt * ((fmax2(0.0, azm) - fmin2(0.0, az)) * a.RCDZ[u]
                  + (fmax2(0.0, axm) - fmin2(0.0, ax)) * rdx
                  + (fmax2(0.0, aym) - fmin2(0.0, ay)) * rdy);
        pmu = dt * ((fmax2(0.0, az) - fmin2(0.0, azm)) * a.RCDZ[u]
                  + (fmax2(0.0, ax) - fmin2(0.0, axm)) * rdx
                  + (fmax2(0.0, ay) - fmin2(0.0, aym)) * rdy);
        if constexpr (TER) { ppu = ppu * m1 * m2 / v.g; pmu = pmu * m1 * m2 / v.g; }
        azm = az;
      }
      if (rim) phi(u, er, ec, e, erdx, erdy, em1, em2, lf, elz);
      rwu = (u == KS ? v.mz : u == KE ? mzm : v.mz + mzm) * a.RCDZ[u];
      ruu = (v.mx + v.mxm) * rdx;
      rvu = (v.my + v.mym) * rdy;
      Du = v.D;
      mzm = v.mz;
      w[0] = w[1]; w[1] = w[2]; w[2] = w[3]; w[3] = wn;
    }
    __syncthreads();
    const int k = u - 1;
    if (act && k >= k0) {
      const int c2 = tx + 2, r2 = ty + 2;  // the cell in the two-cell-ring arrays
      const int c1 = tx + 1, r1 = ty + 1;  // ... and in the one-cell-ring arrays
      const double(*Q0k)[W2] = sQ0[k % 5];
      const double pin = Q0k[r2][c2], plo = sPL[k % 3][r1][c1];
      double qmax, qmin;
      if constexpr (VECT) {
        const int ka = k == KE ? k : k + 1, kb = k == KS ? k : k - 1;
        double f[18];
        get_fact(f, rw, ru, rv);
        // upstream (qa) / downstream (qb) 14-point combinations (COMMON.F90:2096-2155),
        // in the order of fct_qa / fct_qb; P(l, dj, di) is level l at (j+dj, i+di)
        auto qa = [&](auto P, int k1, int k0) {
          return f[17] * P(k1, 1, 1) + f[16] * P(k0, 1, 1) + f[15] * P(k1, 1, 0) + f[14] * P(k0, 1, 0)
               + f[13] * P(k1, 1, -1) + f[11] * P(k1, 0, 1) + f[10] * P(k0, 0, 1) + f[9] * P(k1, 0, 0)
               + f[7] * P(k1, 0, -1) + f[5] * P(k1, -1, 1) + f[4] * P(k0, -1, 1) + f[3] * P(k1, -1, 0)
               + f[1] * P(k1, -1, -1) + f[8] * P(k0, 0, 0);
        };
        auto qb = [&](auto P, int k1, int k0) {
          return f[17] * P(k1, -1, -1) + f[16] * P(k0, -1, -1) + f[15] * P(k1, -1, 0) + f[14] * P(k0, -1, 0)
               + f[13] * P(k1, -1, 1) + f[11] * P(k1, 0, -1) + f[10] * P(k0, 0, -1) + f[9] * P(k1, 0, 0)
               + f[7] * P(k1, 0, 1) + f[5] * P(k1, 1, -1) + f[4] * P(k0, -1, -1) + f[3] * P(k1, -1, 0)
               + f[1] * P(k1, 1, 1) + f[8] * P(k0, 0, 0);
        };
        auto PI = [&](int l, int dj, int di) { return sQ0[l % 5][r2 + dj][c2 + di]; };
        auto PL = [&](int l, int dj, int di) { return sPL[l % 3][r1 + dj][c1 + di]; };
        const double qa_in = qa(PI, ka, k);
        const double qb_in = qb(PI, kb, k);
        const double qa_lo = qa(PL, ka, k);
        const double qb_lo = qb(PL, kb, k);
        qmax = fmax2(fmax2(fmax2(fmax2(fmax2(pin, qa_in), qb_in), plo), qa_lo), qb_lo);
        qmin = fmin2(fmin2(fmin2(fmin2(fmin2(pin, qa_in), qb_in), plo), qa_lo), qb_lo);
      } else {  // 7-point bounds (COMMON.F90:2312-2515)
        const int kp = k == KE ? k : k + 1, km = k == KS ? k : k - 1;
        qmax = pin; qmin = pin;
        {
          const double v[7] = {Q0k[r2][c2], sQ0[kp % 5][r2][c2], sQ0[km % 5][r2][c2], Q0k[r2][c2 + 1], Q0k[r2][c2 - 1],
                               Q0k[r2 + 1][c2], Q0k[r2 - 1][c2]};
#pragma unroll
          for (int q = 0; q < 7; ++q) { qmax = fmax2(qmax, v[q]); qmin = fmin2(qmin, v[q]); }
        }
        {
          const double(*L)[W1] = sPL[k % 3];
          const double v[7] = {L[r1][c1], sPL[kp % 3][r1][c1], sPL[km % 3][r1][c1], L[r1][c1 + 1], L[r1][c1 - 1],
                               L[r1 + 1][c1], L[r1 - 1][c1]};
#pragma unroll
          for (int q = 0; q < 7; ++q) { qmax = fmax2(qmax, v[q]); qmin = fmin2(qmin, v[q]); }
        }
      }
      const double qjpls = (qmax - plo) * D;
      const double qjmns = (plo - qmin) * D;
      double zerosw = 0.5 - fsign(0.5, pp - EPS_RP);
      const unsigned o = qc + plb * (unsigned)k;
      sto(a.rjpls, o, fmin2(1.0, qjpls * (1.0 - zerosw) / (pp - zerosw)));
      zerosw = 0.5 - fsign(0.5, pm - EPS_RP);
      sto(a.rjmns, o, fmin2(1.0, qjmns * (1.0 - zerosw) / (pm - zerosw)));
    }
    pp = ppu; pm = pmu; rw = rwu; ru = ruu; rv = rvu; D = Du;
  }
}

// (tile lb of ntile tiles, the segments of L levels one after the other)
template <int S, int TJ, bool VECT, bool TER>
__global__ void __launch_bounds__(64 * TJ, 3) trt_ratio(TtArgs a, unsigned ni_tiles, unsigned ntile, unsigned nblocks, int L) {
  const unsigned lb = xcd_block(blockIdx.x, nblocks);
  const int k0 = a.d.KS + (int)(lb / ntile) * L;
  trt_ratio_body<S, TJ, VECT, TER>(a, lb % ntile, ni_tiles, k0, min(a.d.KE, k0 + L - 1));
}

// ---- FCT pass 2: limited anti-diffusive fluxes and the update ------------------
// With LIM false the same march is the stage without FCT (tracer_fvm_heve.F90:
// 226-231): the high-order fluxes alone, no limiter arrays staged or read.
// Bound by the latency of a level's loads: a thread evaluates the four
// horizontal faces of its cell itself, twice the face work of a tile that
// shares them through LDS, but with one barrier a level (the tiles alternate
// between two slots), no items beside the cells, and few enough registers
// that three blocks of 4 wavefronts (LIM; two of 8 without) cover each
// other's loads.  At 320x320x96: 0.217 ms (4.5 TB/s) against 0.331 with shared
// faces and the next level's loads in flight at one block per CU; 8 rows
// 0.25-0.27; without FCT 0.154 (4.5 TB/s) against 0.172.
template <int S, int TJ, bool LIM, bool TER>
__device__ __forceinline__ void trt_update_body(const TtArgs& a, unsigned lb, unsigned ni_tiles, int k0, int k1) {
  constexpr int W2 = 68, H2 = TJ + 4, W1 = 66, H1 = TJ + 2, NT = 64 * TJ;
  constexpr int NQ = (H2 * W2 + NT - 1) / NT, NR = LIM ? (H1 * W1 + NT - 1) / NT : 0;
  constexpr int R0 = LIM ? H1 : 1;
  __shared__ double sQ[2][H2][W2];  // QTRC, two-cell ring (slot = level & 1)
  __shared__ double sQ0[2][R0][W1], sRP[2][R0][W1], sRM[2][R0][W1];  // QTRC0, R+ and R-, one-cell ring
  const Dims& d = a.d;
  const int KS = d.KS, KE = d.KE;
  const int i0 = d.IS + 64 * (int)(lb % ni_tiles), j0 = d.JS + TJ * (int)(lb / ni_tiles);
  const int tx = threadIdx.x, ty = threadIdx.y, tid = tx + 64 * ty;
  const int i = i0 + tx, j = j0 + ty;
  const bool act = i <= d.IE && j <= d.JE;
  const unsigned IA = (unsigned)d.IA, plb = 8u * (unsigned)d.pl;
  const unsigned qc = 8u * (act ? (unsigned)i + IA * (unsigned)j : (unsigned)d.IS + IA * (unsigned)d.JS);
  const double *mZ = a.mflx, *mX = mZ + d.n3, *mY = mX + d.n3;
  const double rdx = a.RCDX[act ? i : d.IS], rdy = a.RCDY[act ? j : d.JS];
  double m1 = 1.0, m2 = 1.0;
  if constexpr (TER) { m1 = ld(a.MAPF, qc); m2 = ld(a.MAPF + d.pl, qc); }
  auto nd = [&](unsigned o, int dir, int c) {
    double v = ld(a.nd + a.nds * (size_t)dir, o);
    if constexpr (TER) v = ld(a.GSQRT + d.n3 * (size_t)c, o) * v;
    return v;
  };
  auto lim = [](double an, double rpb, double rma, double rpa, double rmb) {
    const double dirsw = 0.5 + fsign(0.5, an);
    return an * (1.0 - fmin2(rpb, rma) * (dirsw) - fmin2(rpa, rmb) * (1.0 - dirsw));
  };
  double w[4];  // QTRC of the own column, levels k-1..k+2
  for (int m = 0; m < 4; ++m) w[m] = ld(a.QTRC, qc + plb * (unsigned)(k0 - 1 + m));
  const unsigned o0 = qc + plb * (unsigned)k0;
  // own QTRC0 and R+/R- at level k
  double q0 = ld(a.QTRC0, o0), rp = 0.0, rm = 0.0;
  if constexpr (LIM) { rp = ld(a.rjpls, o0); rm = ld(a.rjmns, o0); }
  double hzm = 0.0, lzm = 0.0;  // fluxes through the face below
  if (k0 > KS) {
    const unsigned o = o0 - plb;
    const double vel = ld(mZ, o), wl[4] = {ld(a.QTRC, o - plb), w[0], w[1], w[2]};
    hzm = tt_hz<S>(d, k0 - 1, vel, wl, a.nd ? nd(o, 0, I_XYW) : 0.0);
    if constexpr (LIM) lzm = lim(hzm - tt_lflux(vel, ld(a.QTRC0, o), q0), rp, ld(a.rjmns, o), ld(a.rjpls, o), rm);
  }
  for (int k = k0; k <= k1; ++k) {
    const unsigned b = plb * (unsigned)k, oc = qc + b, ou = k < KE ? oc + plb : oc;
    // every load of the level before its barrier
    double tQ[NQ], t0[NR + 1], tp[NR + 1], tm[NR + 1];
#pragma unroll
    for (int h = 0; h < NQ; ++h) {
      const int q = tid + h * NT, r = q / W2, c = q - r * W2;
      const int ii = i0 - 2 + c, jj = j0 - 2 + r;
      const bool ok = q < H2 * W2 && ii < d.IA && jj < d.JA;  // (partial tiles: the rest is never used)
      tQ[h] = ld(a.QTRC, b + (ok ? 8u * ((unsigned)ii + IA * (unsigned)jj) : 0u));
    }
#pragma unroll
    for (int h = 0; h < NR; ++h) {
      const int q = tid + h * NT, r = q / W1, c = q - r * W1;
      const int ii = i0 - 1 + c, jj = j0 - 1 + r;
      const bool ok = q < H1 * W1 && ii < d.IA && jj < d.JA;
      const unsigned o = b + (ok ? 8u * ((unsigned)ii + IA * (unsigned)jj) : 0u);
      t0[h] = ld(a.QTRC0, o);
      tp[h] = ld(a.rjpls, o);
      tm[h] = ld(a.rjmns, o);
    }
    const double mx = ld(mX, oc), mxm = ld(mX, oc - 8u), my = ld(mY, oc), mym = ld(mY, oc - 8u * IA), mz = ld(mZ, oc);
    const double D0 = ld(a.DENS0, oc), rq = a.RHOQ_t ? ld(a.RHOQ_t, oc) : 0.0;
    double D = ld(a.DENS, oc), G = 1.0;
    if constexpr (TER) G = ld(a.GSQRT, oc);
    const double q0u = ld(a.QTRC0, ou), wn = ld(a.QTRC, qc + plb * (unsigned)min(k + 3, d.KA - 1));
    double rpu = 0.0, rmu = 0.0;
    if constexpr (LIM) { rpu = ld(a.rjpls, ou); rmu = ld(a.rjmns, ou); }
    double nz = 0.0, nx = 0.0, nxm = 0.0, ny = 0.0, nym = 0.0;
    if (a.nd) {
      nz = nd(oc, 0, I_XYW);
      nx = nd(oc, 1, I_UYZ); nxm = nd(oc - 8u, 1, I_UYZ);
      ny = nd(oc, 2, I_XVZ); nym = nd(oc - 8u * IA, 2, I_XVZ);
    }
    if constexpr (!LIM) {
      if (a.dens_mode == 1) D = D0 + (D - D0) / 3.0;
      else if (a.dens_mode == 2) D = D0 + (D - D0) * 0.5;
    }
#pragma unroll
    for (int h = 0; h < NQ; ++h) {
      const int q = tid + h * NT;
      if (q < H2 * W2) sQ[k & 1][q / W2][q % W2] = tQ[h];
    }
#pragma unroll
    for (int h = 0; h < NR; ++h) {
      const int q = tid + h * NT;
      if (q < H1 * W1) {
        sQ0[k & 1][q / W1][q % W1] = t0[h];
        sRP[k & 1][q / W1][q % W1] = tp[h];
        sRM[k & 1][q / W1][q % W1] = tm[h];
      }
    }
    __syncthreads();
    if (act) {
      const double(*Q)[W2] = sQ[k & 1];
      const double(*Q0)[W1] = sQ0[k & 1];
      const double(*RP)[W1] = sRP[k & 1];
      const double(*RM)[W1] = sRM[k & 1];
      // high-order flux and limited anti-diffusive flux through the face between cells (r, c) and (r + dj, c + di)
      auto face = [&](int r, int c, int dj, int di, double vel, double n, double& h, double& l) {
        h = tt_hflux<S>(vel, Q[r + 2 - dj][c + 2 - di], Q[r + 2][c + 2], Q[r + 2 + dj][c + 2 + di],
                        Q[r + 2 + 2 * dj][c + 2 + 2 * di], n);
        if constexpr (LIM) {
          const int r1 = r + 1, c1 = c + 1, r2 = r1 + dj, c2 = c1 + di;
          l = lim(h - tt_lflux(vel, Q0[r1][c1], Q0[r2][c2]), RP[r2][c2], RM[r1][c1], RP[r1][c1], RM[r2][c2]);
        }
      };
      double hx, hxm, hy, hym, lx = 0.0, lxm = 0.0, ly = 0.0, lym = 0.0;
      face(ty, tx, 0, 1, mx, nx, hx, lx);
      face(ty, tx - 1, 0, 1, mxm, nxm, hxm, lxm);
      face(ty, tx, 1, 0, my, ny, hy, ly);
      face(ty - 1, tx, 1, 0, mym, nym, hym, lym);
      double hz = 0.0, lz = 0.0;
      if (k != KE) {
        hz = tt_hz<S>(d, k, mz, w, nz);
        if constexpr (LIM) lz = lim(hz - tt_lflux(mz, q0, q0u), rpu, rm, rp, rmu);
      }
      double v;
      if constexpr (LIM)
        v = -((hz - lz - hzm + lzm) * a.RCDZ[k] + (hx - lx - hxm + lxm) * rdx + (hy - ly - hym + lym) * rdy);
      else
        v = -((hz - hzm) * a.RCDZ[k] + (hx - hxm) * rdx + (hy - hym) * rdy);
      if constexpr (TER) v = v * m1 * m2 / G;
      sto(a.QTRCo, oc, (q0 * D0 + a.dtl * (v + rq)) / D);
      hzm = hz;
      lzm = lz;
    }
    w[0] = w[1]; w[1] = w[2]; w[2] = w[3]; w[3] = wn;
    q0 = q0u; rp = rpu; rm = rmu;
  }
}

template <int S, int TJ, bool LIM, bool TER>
__global__ void __launch_bounds__(64 * TJ) trt_update(TtArgs a, unsigned ni_tiles, unsigned ntile, unsigned nblocks, int L) {
  const unsigned lb = xcd_block(blockIdx.x, nblocks);
  const int k0 = a.d.KS + (int)(lb / ntile) * L;
  trt_update_body<S, TJ, LIM, TER>(a, lb % ntile, ni_tiles, k0, min(a.d.KE, k0 + L - 1));
}

// the passes over the tiles of many members (batch.h tables; ni[m] the
// member's tiles across): kinds 0 R+/R-, 1 the update, 2 the stage without FCT
template <int KIND, int S, int TJ, bool VECT>
__global__ void __launch_bounds__(64 * TJ) trt_batch(const TtArgs* __restrict__ tab, const unsigned* __restrict__ first,
                                                     const unsigned* __restrict__ ni, int nmem, unsigned total) {
  for (unsigned t = blockIdx.x; t < total; t += gridDim.x) {
    const unsigned lt = xcd_block(t, total);
    const int m = batch_member(first, nmem, lt);
    const Dims& d = tab[m].d;
    if constexpr (KIND == 0) trt_ratio_body<S, TJ, VECT, false>(tab[m], lt - first[m], ni[m], d.KS, d.KE);
    else trt_update_body<S, TJ, KIND == 1, false>(tab[m], lt - first[m], ni[m], d.KS, d.KE);
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// rows of the tiles: the FCT passes and the stage without FCT
constexpr int TT_TJ = 4, TT_TJN = 8;

// blocks of a pass: tiles by segments of levels; slots blocks resident at
// once, pro levels' work before a segment's first level
struct TtGrid {
  unsigned ni, nt, nb;
  int L;
};
static TtGrid tt_grid(const Ctx& c, int tj, unsigned per_cu, double pro) {
  const Dims& d = c.d;
  TtGrid g;
  g.ni = (unsigned)((d.IE - d.IS + 1 + 63) / 64);
  g.nt = g.ni * (unsigned)((d.JE - d.JS + 1 + tj - 1) / tj);
  const int kmax = d.KE - d.KS + 1;
  g.L = seg_levels(g.nt, kmax, per_cu * (unsigned)c.ncu, pro);
  g.nb = g.nt * (unsigned)((kmax + g.L - 1) / g.L);
  return g;
}

template <int S, bool TER>
static hipError_t trt_launch(const Ctx& c, const TtArgs& a, bool fct, bool along, hipStream_t s) {
  constexpr int TJ = TT_TJ, TJN = TT_TJN;
  if (!fct) {
    const TtGrid g = tt_grid(c, TJN, 2, 1.0);
    prof_start(c, "tracer_nofct", s);
    hipLaunchKernelGGL((trt_update<S, TJN, false, TER>), dim3(g.nb), dim3(64, TJN), 0, s, a, g.ni, g.nt, g.nb, g.L);
    prof_stop(c, s);
    return hipGetLastError();
  }
  const TtGrid gr = tt_grid(c, TJ, 3, 2.0), gu = tt_grid(c, TJ, 3, 1.0);
  prof_start(c, "fct_ratio", s);
  if (along) hipLaunchKernelGGL((trt_ratio<S, TJ, true, TER>), dim3(gr.nb), dim3(64, TJ), 0, s, a, gr.ni, gr.nt, gr.nb, gr.L);
  else hipLaunchKernelGGL((trt_ratio<S, TJ, false, TER>), dim3(gr.nb), dim3(64, TJ), 0, s, a, gr.ni, gr.nt, gr.nb, gr.L);
  prof_stop(c, s);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  double* r[2] = {a.rjpls, a.rjmns};
  e = halo_fill(c, r, 2, s);
  if (e != hipSuccess) return e;
  prof_start(c, "fct_update", s);
  hipLaunchKernelGGL((trt_update<S, TJ, true, TER>), dim3(gu.nb), dim3(64, TJ), 0, s, a, gu.ni, gu.nt, gu.nb, gu.L);
  prof_stop(c, s);
  return hipGetLastError();
}

// Where a CU gets at least eight levels of an FCT tile.  Below, the segments
// are short and their prologues cost more than the per-point kernels' repeated
// loads; a large step with three tracers, tiles against per-point kernels:
// 64x64x48 (3 levels a CU) 516 us against 484, 97x61x45 (5.6) 594 / 588,
// 96x96x64 (12) 848 / 903, 128x128x64 (16) 1180 / 1267, 320x320x96 (150) 10.0
// / 11.5 ms; over terrain 40x40x80 752 / 735, 96x96x64 1283 / 1369.
bool tracer_tile_supported(const Ctx& c) {
  const int st = c.scheme_tracer;
  if (!(st == UD3 || st == CD4 || st == UD3KOREN || st == UD1 || st == CD2)) return false;
  const Dims& d = c.d;
  if (d.n3 >= TILE_MAX_N3) return false;
  const long nb = (long)((d.IE - d.IS + 1 + 63) / 64) * ((d.JE - d.JS + 1 + TT_TJ - 1) / TT_TJ);
  return c.tracer_tile == 2 || nb * (d.KE - d.KS + 1) >= 8L * c.ncu;
}

hipError_t tracer_stage_tile(const Ctx& c, const TracerIO& io, double* rjpls, double* rjmns, hipStream_t s) {
  TtArgs a;
  a.d = c.d;
  a.QTRC = io.QTRC; a.QTRC0 = io.QTRC0; a.RHOQ_t = io.RHOQ_t; a.DENS0 = io.DENS0; a.DENS = io.DENS;
  a.mflx = io.mflx_hi; a.nd = io.num_diff; a.nds = c.d.n3;
  a.RCDZ = c.g1.RCDZ; a.RCDX = c.g1.RCDX; a.RCDY = c.g1.RCDY;
  a.dtl = io.dtl; a.QTRCo = io.QTRCo;
  a.rjpls = rjpls; a.rjmns = rjmns;
  a.GSQRT = c.GSQRT; a.MAPF = c.MAPF; a.dens_mode = io.dens_mode;
  const bool along = io.flag_along != 0, fct = io.flag_fct != 0;
  if (fct && io.dens_mode) return hipErrorNotSupported;
  switch (c.scheme_tracer) {
    case UD3: return c.terrain ? trt_launch<UD3, true>(c, a, fct, along, s) : trt_launch<UD3, false>(c, a, fct, along, s);
    case CD4: return c.terrain ? trt_launch<CD4, true>(c, a, fct, along, s) : trt_launch<CD4, false>(c, a, fct, along, s);
    case UD3KOREN: return c.terrain ? trt_launch<UD3KOREN, true>(c, a, fct, along, s) : trt_launch<UD3KOREN, false>(c, a, fct, along, s);
    case UD1: return c.terrain ? trt_launch<UD1, true>(c, a, fct, along, s) : trt_launch<UD1, false>(c, a, fct, along, s);
    case CD2: return c.terrain ? trt_launch<CD2, true>(c, a, fct, along, s) : trt_launch<CD2, false>(c, a, fct, along, s);
    default: return hipErrorNotSupported;
  }
}

static unsigned batch_tiles(const Dims& d) {
  return (unsigned)((d.IE - d.IS + 1 + 63) / 64) * (unsigned)((d.JE - d.JS + 1 + TT_TJ - 1) / TT_TJ);
}
unsigned trt_batch_tiles(const Ctx* const* cs, int n) {
  unsigned t = 0;
  for (int m = 0; m < n; ++m) t += batch_tiles(cs[m]->d);
  return t;
}

// the stages of every member on tiles (the members' stage arguments;
// flat terrain, one two-cell scheme, one bound kind)
hipError_t trt_batch_build(const Ctx* const* cs, const TracerIO* ios, int n, BatchBuf& b) {
  if (n <= 0) return hipErrorInvalidValue;
  std::vector<TtArgs> args((size_t)n);
  std::vector<unsigned> first((size_t)n + 1, 0), ni((size_t)n, 0);
  const int scheme = cs[0]->scheme_tracer, along = ios[0].flag_along;
  for (int m = 0; m < n; ++m) {
    const Ctx& c = *cs[m];
    const TracerIO& io = ios[m];
    const int st = c.scheme_tracer;
    if (c.terrain || st != scheme || io.flag_along != along || !(st == UD3 || st == CD4 || st == UD3KOREN || st == UD1 || st == CD2))
      return hipErrorNotSupported;
    TtArgs& a = args[(size_t)m];
    a.d = c.d;
    a.QTRC = io.QTRC; a.QTRC0 = io.QTRC0; a.RHOQ_t = io.RHOQ_t; a.DENS0 = io.DENS0; a.DENS = io.DENS;
    a.mflx = io.mflx_hi; a.nd = io.num_diff; a.nds = c.d.n3;
    a.RCDZ = c.g1.RCDZ; a.RCDX = c.g1.RCDX; a.RCDY = c.g1.RCDY;
    a.dtl = io.dtl; a.QTRCo = io.QTRCo;
    a.rjpls = c.scr[1]; a.rjmns = c.scr[2];
    a.GSQRT = nullptr; a.MAPF = nullptr; a.dens_mode = io.dens_mode;
    const Dims& d = c.d;
    ni[(size_t)m] = (unsigned)((d.IE - d.IS + 1 + 63) / 64);
    first[(size_t)m + 1] = first[(size_t)m] + batch_tiles(d);
  }
  const hipError_t e = batch_upload(args, first, ni, b);
  b.scheme = scheme; b.tj = along;
  return e;
}

template <int KIND, int S>
static hipError_t trt_batch_t(const BatchBuf& b, hipStream_t s) {
  const TtArgs* tab;
  const unsigned *first, *ni;
  batch_tables(b, tab, first, ni);
  if (KIND == 0 && b.tj)
    hipLaunchKernelGGL((trt_batch<0, S, TT_TJ, true>), dim3(b.total), dim3(64, TT_TJ), 0, s, tab, first, ni, b.nmem, b.total);
  else if (KIND == 0)
    hipLaunchKernelGGL((trt_batch<0, S, TT_TJ, false>), dim3(b.total), dim3(64, TT_TJ), 0, s, tab, first, ni, b.nmem, b.total);
  else
    hipLaunchKernelGGL((trt_batch<KIND == 0 ? 1 : KIND, S, TT_TJ, false>), dim3(b.total), dim3(64, TT_TJ), 0, s, tab, first, ni, b.nmem, b.total);
  return hipGetLastError();
}
template <int KIND>
static hipError_t trt_batch_k(const BatchBuf& b, hipStream_t s) {
  switch (b.scheme) {
    case UD3: return trt_batch_t<KIND, UD3>(b, s);
    case UD3KOREN: return trt_batch_t<KIND, UD3KOREN>(b, s);
    case CD2: return trt_batch_t<KIND, CD2>(b, s);
    case UD1: return trt_batch_t<KIND, UD1>(b, s);
    default: return trt_batch_t<KIND, CD4>(b, s);
  }
}
hipError_t trt_batch_launch(const BatchBuf& b, int kind, hipStream_t s) {
  if (!b.dev) return hipErrorInvalidValue;
  return kind == 0 ? trt_batch_k<0>(b, s) : kind == 1 ? trt_batch_k<1>(b, s) : trt_batch_k<2>(b, s);
}

}  // namespace shp
