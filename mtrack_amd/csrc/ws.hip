// The weak-strong multi-bunch turn with fast beam-ion interaction (FBII) on one
// MI355X: the reference's BunchModel = STRONG path, manager_weakstrong +
// worker_weakstrong (src/manager_weakstrong.c:7-263, src/worker_weakstrong.c:14-247).
//
// Each filled bunch is 2 Nslc + 1 slice centroids (tau, delta, x, x', z, z')
// resident in HBM.  The launches of a turn, on one stream:
//
//   k_ws_step    (without FBII) one block per bunch: phase 2 of the turn before
//                and phase 1 of this one; with FBII it only ends a call;
//   k_ws_phase1  (with FBII) blocks 0 .. G-1: the ion kicks of the turn before and
//                phase 1; the others, one thread per point, the Bassetti-Erskine
//                field of every slice on the 5 x 5 absolute grid (two Faddeeva
//                evaluations per point);
//   k_ws_create  the ions each bunch creates, one thread each, kicked by the
//                bunch's later slices (fbi_weakstrong_bunch,
//                src/fbi_weakstrong.c:49-298);
//   k_ws_ions    the reference's manager relay (fbi_weakstrong_train
//                :301-451): the accumulated ion cloud drifts to each bunch in
//                train order, passes its slices (bilinear field interpolation,
//                src/fbi_weakstrong.c:454-580), kicks the slice centroids with
//                the summed ion field, and the bunch's own ions join the cloud.
//                An ion's path depends only on the field tables phase 1 made
//                and on the drift times, never on the kicks the train gives the
//                electrons, so the whole relay is one launch with one lane per
//                ion over every later bunch (per-slice wave sums, block partials
//                per bunch);
//   k_ws_ksum    a per-bunch, per-quantity sum of the partials, and phase 2 of the
//                turn in blocks beside.
//
// Phase 1 is the synchrotron step of the centroids (transformSbunch_shortrange,
// src/rw_weakstrong.c:10-67), the bunch centroid, the CM history append
// (src/bunch.c:94-115) and the monitor-turn statistics (src/bunch.c:516-550);
// phase 2 the betatron rotation (transformSbunch_optic, :194-253) and the
// resistive-wall kick of every other bucket's centroid history
// (transformSbunch_longrange, :69-192).  k_ws_cloud_reset + k_ws_train keep the
// bunch-by-bunch relay (one launch per bunch) for MBT_WS_SERIAL_TRAIN and for
// trains whose partials would not fit.
//
// Everything but the ion-field sums, sin and the Faddeeva function keeps the
// reference's operation order; constants derived with libm are computed on the
// host with glibc.  Results are bitwise reproducible run to run.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include "mbt_host.h"
#include "wofz_dev.h"
#include "wave_dev.h"

#pragma clang fp contract(off)

#define WS_S 50       // slice capacity of the reference's bunch_strong_t
#define WS_PTS 1250   // 50 slices x 25 grid points
#define WS_TQ (2 * WS_S + 3 + 12) // per bunch in WSD::tot: 2 S + 3 train sums, 4 x 3 own-ion sums
#define WS_HIST 30    // CM history depth (src/bunch.h:155)
#define WS_RING 31    // rows of the dipole history: the depth and the row being written
#define WS_MSG 5000   // doubles of the history message (src/manager_weakstrong.c:170-173)
#define WS_T 256      // turns of outputs per device buffer block
#define WS_WG 256
// device memory the ion-parallel train may use for its per-bunch partials
#define WS_TRAIN_PARTIAL_MAX (8LL << 30)

#define K_C 2.997925e+08
#define K_EPS0 8.854187817620e-12
#define K_E 1.602e-19

#define CK(x)                                                                                    \
  do {                                                                                           \
    hipError_t e_ = (x);                                                                         \
    if (e_ != hipSuccess) {                                                                      \
      mbt_set_error("%s failed: %s (%s:%d)", #x, hipGetErrorString(e_), __FILE__, __LINE__);     \
      return MBT_EDEVICE;                                                                        \
    }                                                                                            \
  } while (0)

extern "C" int mbt_ws_generate(const mbt_config *c, double *slices, int *npop, int *nofe, double *dist);
extern "C" void mbt_ws_grid(const mbt_config *c, double *agLOCx, double *agLOCz);

struct WSP {
  int S, G, h, Nmlt, NmultiT, fbii, rw, track_h, track_v, track[3], Nions;
  int mixed; // Faddeeva function of the field tables in FP32 (MBT_WS_MIXED)
  double eps, wrf, phai0, Urad, T0, ac;                 // synchrotron step
  double gamma1[3], alpha1[3], beta1[3];                // statistics
  double v11, v12, v21, v22, h11, h12, h21, h22;        // one-turn rotation (glibc cos/sin)
  double rwa11[2], rwa12[2];                            // RW: [HOR, VER]
  int triggerRW;
  double fNp;
  double ntot; // macro-electrons in the slices
  double factBE, sxx, szz, deltT, aAx, aAz, aLx, aLz, den_dQ; // FBII fields
  double iaAx, iaAz;                                          // 1 / aAx, 1 / aAz
  double factF, factjp0, CdeltT;
  double dtF; // deltT * factF: the ion train's velocity kick per unit field
};

struct WSD {
  double *sl;       // [G][6][S] xtau xeps xx xp zz zp
  const int *npop;  // [S]
  const int *nofe;  // [S*25]
  const int *bucket; // [G]
  const double *wallcur, *nelec, *convion; // [G] RW constant times bunch current, electrons, ions per macro-ion
  double *dip;      // [2][WS_RING][G] wall dipoles of the bunches' centroids (HOR, VER), a row per turn
  const double *wall; // [trigger][2][Nmlt + 1][h] wake per tap and distance in buckets (entry d - 1)
  double2 *Exy;     // [G][S*25] (Ex, Ey) of every grid point
  double2 *tab;     // [G][S][WS_QT] the ion train's tables of it
  double *li;       // [5][G][S*25] local ions: Nri x x' y y'
  double *cl;       // [5][cap] ion cloud
  long long cap;
  double *part;     // [blocks][S][2]
  double *psum;     // [blocks][3]
  unsigned *done;
  const double *dtime;    // [G] drift time from the previous bunch
  double *tpart;          // ion-parallel train: per bunch ib, [2 S + 3][blocks with an ion ahead of ib]
  const long long *toff;  // [G] offset of bunch ib's partials in tpart
  int nblk_ions;          // blocks of k_ws_ions
  double *tot;            // ion-parallel train: [G][WS_TQ] per-bunch sums of the partials and own-ion sums
  double *cm, *mon, *ion, *zcm; // output blocks [WS_T][G][4|18|3], [WS_T][h]
};

// ------------------------------------------------------------ device helpers

// get_linearly_interpolated_Efields, src/fbi_weakstrong.c:454-580, on one
// slice's 25 field values, stored as (Ex, Ey) pairs so that one 16-byte LDS
// read fetches both fields of a grid point.  The grid quotients multiply by the
// reciprocal spacings (iax = 1 / aAx, iaz = 1 / aAz) in place of the
// reference's four FP64 divisions per interaction; such a quotient can differ
// from the divided one in its last bit, which moves a cell choice only where
// the bilinear field is continuous.
__device__ __forceinline__ void ws_interp(const double2 *t, double aAx, double aAz, double iax, double iaz, double xx,
                                          double yy, double &Ex, double &Ey)
{
  // the bilinear steps as fused multiply-adds (one rounding less each)
#pragma clang fp contract(fast)
  // Grid point (kx, kz), kx, kz in [-2, 2], is entry 5 kx + kz + 12.  The cell
  // is k1 = trunc(x / d) clamped to the grid, its partner one step further from
  // the centre in the direction of the coordinate's sign (the same point at the
  // clamped edge), as in the reference's two sign cases.  The fraction is
  // |x - k1 d| / d: the reference's fraction, negated where it interpolates
  // towards the negative side (the sign flips are exact).
  const int k1x = min(max((int)(xx * iax), -2), 2);
  const int k1z = min(max((int)(yy * iaz), -2), 2);
  const int k2x = min(max(k1x + (xx >= 0 ? 1 : -1), -2), 2);
  const int k2z = min(max(k1z + (yy >= 0 ? 1 : -1), -2), 2);
  const double2 *tc = t + 12;
  const double2 e1 = tc[5 * k1x + k1z], e2 = tc[5 * k2x + k1z], e3 = tc[5 * k1x + k2z], e4 = tc[5 * k2x + k2z];
  const double sx = fabs((xx - k1x * aAx) * iax), sz = fabs((yy - k1z * aAz) * iaz);
  const double y5 = e1.y + sx * (e2.y - e1.y);
  const double y6 = e3.y + sx * (e4.y - e3.y);
  const double x5 = e1.x + sx * (e2.x - e1.x);
  const double x6 = e3.x + sx * (e4.x - e3.x);
  Ey = y5 + sz * (y6 - y5);
  Ex = x5 + sz * (x6 - x5);
}

// ------------------------------------------------------------- the electron side

// The electron side of a turn for one bunch per block, on the bunch's slices
// staged in LDS.  Three parts, any of which a launch may ask for:
//   kicks of the ion train of the turn before (the sums of k_ws_ksum);
//   phase 2 of turn rev2: the betatron rotation, the resistive-wall kick of every
//     bunch's centroid history and the slice-averaged vertical centroid of the
//     bunch's bucket (writeoutVCMmotionsPM2, src/fbi_weakstrong.c:688-737; the
//     train's kicks, on the slopes, leave it alone);
//   phase 1 of turn rev1: the synchrotron step of every slice, the centroids the
//     bunch reports, the dipole history and the monitor statistics.
// Phase 1 of a turn needs nothing but the bunch's own slices after phase 2 of the
// turn before, so without FBII a turn is one launch (phase 2 of the turn before,
// then phase 1) and one more ends the call.  The resistive wall reads only
// dipoles of earlier launches: the history is a ring of WS_RING rows, and the row
// phase 1 writes is older than any the same launch reads.
// Bound: latency (sums of 41 slices and of up to h kicks kept in the
// reference's order, one lane each).  416 bunches, 10 wall turns, per turn: 107 us
// as three launches (one lane for all of a bunch's sums; a test of the filling, a
// square root and two divisions per tap) -> 13.1 us as one, kernel time; a turn takes
// 19.5, the rest lies between the launches.
struct WSStep {
  int kick;            // slot of the turn whose ion sums to apply, -1: none
  long long rev2;      // phase 2 of this turn, -1: none
  int slot2;
  long long rev1;      // phase 1 of this turn, -1: none
  int slot1, monitor;
};

#ifndef WS_STEP_WG
#define WS_STEP_WG 512
#endif

// Row of turn rev - age in the dipole history ring.
__device__ __forceinline__ int ws_row(long long rev, int age)
{
  const int r = (int)((rev - age) % WS_RING);
  return r < 0 ? r + WS_RING : r;
}

// The resistive-wall kick bunch b (bucket kb) gets from bunch s, plane pl: the
// taps j = 0 .. Nmlt of the source's dipole history over the tabulated wake
// (transformSbunch_longrange, src/rw_weakstrong.c:69-192).  The worker's copy of
// the history holds zeros where jb + j h falls outside the 5000-double message.
__device__ __forceinline__ double ws_wall_kick(const WSP &P, const WSD &D, int kb, int s, int pl, long long rev)
{
  if (rev < P.Nmlt) return 0.0;
  const int jb = D.bucket[s], h = P.h;
  const double cur = D.wallcur[s];
  // distance in buckets, h for the bunch's own (a full turn)
  const int d = jb > kb ? jb - kb : h + jb - kb;
  const int trig = P.triggerRW && rev < 50 ? 1 : 0;
  const double *W = D.wall + (size_t)(trig * 2 + pl) * (P.Nmlt + 1) * h + d - 1;
  const double *dip = D.dip + (size_t)pl * WS_RING * P.G + s;
  const int a0 = jb > kb ? 0 : 1;
  // oldest age the history and the message hold
  const int amax = min(P.NmultiT - 1, (WS_MSG - 1 - jb) / h);
  int row = ws_row(rev, a0);
  double Dup = 0.0;
  const int nj = min(P.Nmlt + 1, amax - a0 + 1);
#pragma unroll 8
  for (int j = 0; j < nj; j++) {
    Dup = Dup + dip[row * P.G] * W[j * h];
    row = row == 0 ? WS_RING - 1 : row - 1;
  }
  return cur * Dup;
}

// a + k[0] + k[1] + ... + k[n - 1] in that order, k in LDS, 16-byte aligned and
// zero from n to the next multiple of 16.  The chain of additions is the
// reference's; the reads of a group of eight are under way while the group before
// is added (read one by one, the 416 kicks of a full ring took 5 us more).
__device__ __forceinline__ double ws_add_in_order(double a, const double *k, int n)
{
  const double2 *q = (const double2 *)k;
  double2 u[4], v[4];
#pragma unroll
  for (int i = 0; i < 4; i++) u[i] = q[i];
  for (int s = 0; s < n; s += 16, q += 8) {
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = q[4 + i];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      a += u[i].x;
      a += u[i].y;
    }
#pragma unroll
    for (int i = 0; i < 4; i++) u[i] = q[8 + i]; // past the end at the last group: unused
#pragma unroll
    for (int i = 0; i < 4; i++) {
      a += v[i].x;
      a += v[i].y;
    }
  }
  return a;
}

// LDS of ws_electrons, in doubles: the six slice arrays, populations and six rows
// of products, each row and the two rows of kicks padded for ws_add_in_order.
#define WS_PAD16(n) (((n) + 15) / 16 * 16)
__host__ __device__ __forceinline__ int ws_electrons_lds(int S, int G)
{
  return 13 * WS_PAD16(S) + 2 * WS_PAD16(G) + 8;
}

// One block's bunch b; lds: ws_electrons_lds(S, G) doubles, as the double2 that
// ws_add_in_order reads, so that they are aligned to it.
__device__ void ws_electrons(const WSP &P, const WSD &D, int b, const WSStep &T, double2 *lds)
{
  double *sm = (double *)lds;
  const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63, wv = tid >> 6, S = P.S, G = P.G;
  const int kb = D.bucket[b];
  const int SP = WS_PAD16(S), GP = WS_PAD16(G);
  double *xtau = sm, *xeps = xtau + SP, *xx = xeps + SP, *xp = xx + SP, *zz = xp + SP, *zp = zz + SP;
  double *np = zp + SP, *wt = np + SP, *dup = wt + 6 * SP;
  __shared__ double cms[6];
  double *sl = D.sl + (size_t)b * 6 * S;
  for (int i = tid; i < 6 * SP; i += nt) {
    const int c = i / SP, ic = i - c * SP;
    sm[i] = ic < S ? sl[c * S + ic] : 0.0;
  }
  for (int i = tid; i < SP; i += nt) np[i] = i < S ? (double)D.npop[i] : 0.0;
  const bool p2 = T.rev2 >= 0, p1 = T.rev1 >= 0, wall = p2 && P.rw;
  if (wall)
    for (int e = tid; e < 2 * GP; e += nt) {
      const int pl = e >= GP, s = e - pl * GP;
      dup[e] = s < G && (pl ? P.track_v : P.track_h) ? ws_wall_kick(P, D, kb, s, pl, T.rev2) : 0.0;
    }
  __syncthreads();
  if (T.kick >= 0) {
    const int NQ = 2 * S + 3;
    const double *tot = D.tot + (size_t)b * WS_TQ;
    if (b > 0) {
      const double nel = D.nelec[b];
      for (int c = tid; c < S; c += nt) {
        const double dQ = nel * D.npop[c] * K_E;
        const double fjp = dQ > 0.0 ? P.factjp0 / dQ : 0.0;
        const double sx = fjp * tot[2 * c], sy = fjp * tot[2 * c + 1];
        xp[c] = xp[c] + P.CdeltT * sx;
        zp[c] = zp[c] + P.CdeltT * sy;
      }
    }
    if (tid >= 64 && tid < 67) {
      const int m = tid - 64;
      double v = b > 0 ? tot[2 * S + m] : 0.0;
      for (int w = 0; w < WS_WG / 64; w++) v += tot[NQ + 3 * w + m];
      D.ion[((size_t)T.kick * G + b) * 3 + m] = v;
    }
    __syncthreads();
  }
  if (p2) {
    // wave 0 the horizontal plane, wave 1 the vertical one, a lane per slice
    if (wv < 2 && lane < S) {
      double *u = wv ? zz : xx, *q = wv ? zp : xp;
      const double m11 = wv ? P.v11 : P.h11, m12 = wv ? P.v12 : P.h12, m21 = wv ? P.v21 : P.h21,
                   m22 = wv ? P.v22 : P.h22;
      const double un = m11 * u[lane] + m12 * q[lane];
      double a = m21 * u[lane] + m22 * q[lane];
      if (wall && (wv ? P.track_v : P.track_h)) a = ws_add_in_order(a, dup + wv * GP, G); // in bucket order
      u[lane] = un;
      q[lane] = a;
    }
    __syncthreads();
    if (tid == 128) D.zcm[(size_t)T.slot2 * P.h + kb] = ws_add_in_order(0.0, zz, S) / ((double)S);
  }
  if (p1) {
    for (int ic = tid; ic < S; ic += nt) {
      const double e0 = xeps[ic];
      const double gain = P.eps * sin(P.wrf * xtau[ic] + P.phai0);
      xeps[ic] = e0 + gain - P.Urad;
      xtau[ic] = xtau[ic] - e0 * P.T0 * P.ac;
    }
    __syncthreads();
    // bunch_strong_updateCM (src/bunch_strong.c:221-266), one lane per coordinate
    for (int i = tid; i < 6 * SP; i += nt) wt[i] = sm[i] * np[i % SP];
    __syncthreads();
    if (tid < 6) cms[tid] = ws_add_in_order(0.0, wt + tid * SP, S) / P.ntot;
    __syncthreads();
    if (tid < 4) D.cm[((size_t)T.slot1 * G + b) * 4 + tid] = cms[2 + tid];
    if (P.rw && tid < 2)
      D.dip[((size_t)tid * WS_RING + ws_row(T.rev1, 0)) * G + b] =
          P.fNp * (P.rwa11[tid] * cms[2 + 2 * tid] + P.rwa12[tid] * cms[3 + 2 * tid]);
    if (T.monitor && tid < 18) {
      // quantity k (position, its rms, slope, its rms, ampinv, its centroid's) of plane pl
      const int k = tid / 3, pl = tid % 3;
      const double *u = sm + 2 * pl * SP, *p = u + SP, avr = cms[2 * pl], avs = cms[2 * pl + 1];
      double v = 0.0;
      if (k == 1 || k == 3) {
        const double *w = k == 1 ? u : p, av = k == 1 ? avr : avs;
        for (int ic = 0; ic < S; ic++) v += (w[ic] - av) * (w[ic] - av) * np[ic];
        v = sqrt(v / P.ntot);
      } else if (k == 4) {
        for (int ic = 0; ic < S; ic++)
          v += np[ic] * (P.gamma1[pl] * (u[ic] * u[ic]) + 2.0 * P.alpha1[pl] * u[ic] * p[ic] +
                         P.beta1[pl] * (p[ic] * p[ic]));
        v = v / P.ntot;
      } else if (k == 5) {
        v = P.gamma1[pl] * (avr * avr) + 2.0 * P.alpha1[pl] * avr * avs + P.beta1[pl] * (avs * avs);
      } else {
        v = k == 0 ? avr : avs;
      }
      D.mon[((size_t)T.slot1 * G + b) * 18 + 3 * k + pl] = P.track[pl] ? v : 0.0;
    }
  }
  // back to memory: tau and delta move in phase 1 only, the positions in phase 2
  // only (other blocks of a launch without it read them)
  __syncthreads();
  for (int i = tid; i < 6 * S; i += nt) {
    const int c = i / S;
    if (c < 2 ? p1 : (c == 2 || c == 4 ? p2 : p2 || T.kick >= 0)) sl[i] = sm[c * SP + i - c * S];
  }
}

// Blocks 0 .. G-1: the electron side of a bunch each.
__global__ __launch_bounds__(WS_STEP_WG) void k_ws_step(WSP P, WSD D, WSStep T)
{
  extern __shared__ double2 sm[];
  ws_electrons(P, D, blockIdx.x, T, sm);
}

// With FBII, phase 1: blocks 0 .. G-1 the electron side (the train's kicks of the
// turn before and phase 1), the others the Bassetti-Erskine field at one absolute
// grid point of one slice of one bunch per thread; the field needs the slices'
// transverse positions only, which kicks and phase 1 leave alone.
__global__ __launch_bounds__(WS_WG) void k_ws_phase1(WSP P, WSD D, WSStep T)
{
  extern __shared__ double2 sm[];
  const int tid = threadIdx.x, S = P.S;
  if ((int)blockIdx.x < P.G) {
    ws_electrons(P, D, blockIdx.x, T, sm);
    return;
  }
  const int npts = S * 25;
  const long long gq = (long long)(blockIdx.x - P.G) * WS_WG + tid;
  if (gq >= (long long)P.G * npts) return;
  const int b = (int)(gq / npts), q = (int)(gq - (long long)b * npts);
  const double *xx = D.sl + (size_t)b * 6 * S + 2 * S, *zz = xx + 2 * S;
  const int cell = q / 25, r = q % 25, msx = r / 5 - 2, msz = r % 5 - 2;
  const double dQ = D.nelec[b] * D.npop[cell] * K_E;
  const double fdQ = dQ / P.den_dQ;
  const double Dx = msx * P.aAx - xx[cell];
  const double xi1 = Dx / P.factBE, xi2 = xi1 * P.szz / P.sxx;
  const double Dy = msz * P.aAz - zz[cell];
  const double yi1 = Dy / P.factBE, yi2 = yi1 * P.sxx / P.szz;
  double u1, v1, u2, v2;
  if (P.mixed) {
    float a1, b1, a2, b2;
    mbt_wofz_dev<float>((float)xi1, (float)yi1, a1, b1);
    mbt_wofz_dev<float>((float)xi2, (float)yi2, a2, b2);
    u1 = a1;
    v1 = b1;
    u2 = a2;
    v2 = b2;
  } else {
    mbt_wofz_dev<double>(xi1, yi1, u1, v1);
    mbt_wofz_dev<double>(xi2, yi2, u2, v2);
  }
  const double g = exp(-(Dx * Dx * 1.0e+06 / (2 * P.sxx * P.sxx) + Dy * Dy * 1.0e+06 / (2 * P.szz * P.szz)));
  const double Ex = -fdQ * (v1 - g * v2), Ey = -fdQ * (u1 - g * u2);
  D.Exy[gq] = make_double2(Ex, Ey);
}

// The ion train's field table of a slice: the 5 x 5 grid fields with the edge rows in
// x repeated once more, rows kx = 0 .. 5 for the cells [kx - 3, kx - 2]: WS_ROWS
// double2 (Ex, Ey) of the row's lower point, as many of its step to the upper one,
// E(kx + 1, z) - E(kx, z), zero past the edge.  The steps are the subtractions of
// the bilinear formula, made once per table instead of once per ion.  Two arrays of
// 16-byte entries rather than 32-byte pairs: the lanes of one read then spread over
// all sixteen 16-byte bank groups of the LDS, not eight (measured: a sixth of the
// bank-conflict cycles, SQ_LDS_BANK_CONFLICT).
#define WS_ROWS 30
#define WS_QT (2 * WS_ROWS) // double2 per slice

// Entry k of the table of a slice with grid fields t.
__device__ __forceinline__ void ws_table_entry(const double2 *t, int k, double2 *T)
{
  const int kx = k / 5, z = k - 5 * kx;
  const double2 e1 = t[5 * (min(max(kx - 3, -2), 2) + 2) + z], e2 = t[5 * (min(max(kx - 2, -2), 2) + 2) + z];
  T[k] = e1;
  T[WS_ROWS + k] = make_double2(e2.x - e1.x, e2.y - e1.y);
}

// The ions every bunch creates, one per thread: one per local grid point of
// each slice, kicked by the bunch's later slices (their field tables read from
// the one k_ws_phase1 wrote); the blocks after those (ion-parallel train) write the
// train's tables, an entry and its step per thread.
__global__ __launch_bounds__(WS_WG) void k_ws_create(WSP P, WSD D)
{
  const int S = P.S, npts = S * 25;
  const int made = (int)(((long long)P.G * npts + WS_WG - 1) / WS_WG);
  if ((int)blockIdx.x >= made) {
    const long long k = (long long)(blockIdx.x - made) * WS_WG + threadIdx.x, sl = k / WS_ROWS;
    if (sl < (long long)P.G * S) ws_table_entry(D.Exy + sl * 25, (int)(k - sl * WS_ROWS), D.tab + sl * WS_QT);
    return;
  }
  const long long gq = (long long)blockIdx.x * WS_WG + threadIdx.x;
  if (gq >= (long long)P.G * npts) return;
  const int b = (int)(gq / npts), q = (int)(gq - (long long)b * npts);
  const double *xx = D.sl + (size_t)b * 6 * S + 2 * S, *zz = xx + 2 * S;
  const double2 *exy = D.Exy + (size_t)b * npts;
  const int cell = q / 25, r = q % 25, msx = r / 5 - 2, msz = r % 5 - 2;
  const double Nri = D.convion[b] * ((double)D.nofe[q]);
  double x = xx[cell] + msx * P.aLx, xd = 0.0, y = zz[cell] + msz * P.aLz, yd = 0.0;
  for (int c = cell + 1; c < S; c++) {
    double Ex, Ey;
    ws_interp(exy + c * 25, P.aAx, P.aAz, P.iaAx, P.iaAz, x, y, Ex, Ey);
    const double ax = P.factF * Ex;
    xd = xd + P.deltT * ax;
    x = x + P.deltT * xd;
    const double ay = P.factF * Ey;
    yd = yd + P.deltT * ay;
    y = y + P.deltT * yd;
  }
  const size_t GP = (size_t)P.G * npts;
  D.li[gq] = Nri;
  D.li[GP + gq] = x;
  D.li[2 * GP + gq] = xd;
  D.li[3 * GP + gq] = y;
  D.li[4 * GP + gq] = yd;
}

// ------------------------------------------------------------------ the train

// head bunch: the cloud becomes its ions (src/fbi_weakstrong.c:335-353)
__global__ __launch_bounds__(WS_WG) void k_ws_cloud_reset(WSP P, WSD D, int slot)
{
  __shared__ double red[WS_WG / 64][3];
  const int tid = threadIdx.x, npts = P.S * 25;
  const size_t GP = (size_t)P.G * npts;
  double s0 = 0.0, s1 = 0.0, s2 = 0.0;
  for (int q = tid; q < npts; q += WS_WG) {
    for (int a = 0; a < 5; a++) D.cl[a * D.cap + q] = D.li[a * GP + q];
    s0 += D.li[q] * D.li[GP + q];
    s1 += D.li[q] * D.li[3 * GP + q];
    s2 += D.li[q];
  }
  s0 = wsum64(s0);
  s1 = wsum64(s1);
  s2 = wsum64(s2);
  if ((tid & 63) == 0) {
    red[tid >> 6][0] = s0;
    red[tid >> 6][1] = s1;
    red[tid >> 6][2] = s2;
  }
  __syncthreads();
  if (tid < 3) {
    double s = 0.0;
    for (int w = 0; w < WS_WG / 64; w++) s += red[w][tid];
    D.ion[((size_t)slot * P.G) * 3 + tid] = s;
  }
}

// bunch ib (bucket kb) meets the cloud of nF ions that drifted Dtime since the
// previous bunch; the last block applies the slice kicks and appends the
// bunch's ions
__global__ __launch_bounds__(WS_WG) void k_ws_train(WSP P, WSD D, int ib, long long nF, double Dtime, int slot)
{
  __shared__ double2 exy_s[WS_PTS];
  __shared__ double red[WS_WG / 64][2];
  __shared__ int last;
  const int tid = threadIdx.x, S = P.S, npts = S * 25;
  const size_t GP = (size_t)P.G * npts;
  for (int q = tid; q < npts; q += WS_WG) exy_s[q] = D.Exy[(size_t)ib * npts + q];
  __syncthreads();
  const long long q = (long long)blockIdx.x * WS_WG + tid;
  const bool act = q < nF;
  double Nri = 0.0, x = 0.0, xd = 0.0, y = 0.0, yd = 0.0;
  if (act) {
    Nri = D.cl[q];
    x = D.cl[D.cap + q];
    xd = D.cl[2 * D.cap + q];
    y = D.cl[3 * D.cap + q];
    yd = D.cl[4 * D.cap + q];
    x = x + Dtime * xd;
    y = y + Dtime * yd;
  }
  double *part = D.part + (size_t)blockIdx.x * S * 2;
  for (int c = 0; c < S; c++) {
    double sx = 0.0, sy = 0.0;
    if (act) {
      double Ex, Ey;
      ws_interp(exy_s + c * 25, P.aAx, P.aAz, P.iaAx, P.iaAz, x, y, Ex, Ey);
      const double ax = P.factF * Ex;
      xd = xd + P.deltT * ax;
      x = x + P.deltT * xd;
      const double ay = P.factF * Ey;
      yd = yd + P.deltT * ay;
      y = y + P.deltT * yd;
      sx = Nri * Ex;
      sy = Nri * Ey;
    }
    sx = wsum64(sx);
    sy = wsum64(sy);
    if ((tid & 63) == 0) {
      red[tid >> 6][0] = sx;
      red[tid >> 6][1] = sy;
    }
    __syncthreads();
    if (tid < 2) {
      double s = 0.0;
      for (int w = 0; w < WS_WG / 64; w++) s += red[w][tid];
      part[2 * c + tid] = s;
    }
    __syncthreads();
  }
  double s0 = act ? Nri * x : 0.0, s1 = act ? Nri * y : 0.0, s2 = act ? Nri : 0.0;
  if (act) {
    D.cl[D.cap + q] = x;
    D.cl[2 * D.cap + q] = xd;
    D.cl[3 * D.cap + q] = y;
    D.cl[4 * D.cap + q] = yd;
  }
  s0 = wsum64(s0);
  s1 = wsum64(s1);
  s2 = wsum64(s2);
  __shared__ double red3[WS_WG / 64][3];
  if ((tid & 63) == 0) {
    red3[tid >> 6][0] = s0;
    red3[tid >> 6][1] = s1;
    red3[tid >> 6][2] = s2;
  }
  __syncthreads();
  if (tid < 3) {
    double s = 0.0;
    for (int w = 0; w < WS_WG / 64; w++) s += red3[w][tid];
    D.psum[(size_t)blockIdx.x * 3 + tid] = s;
  }
  // ---- the last block to finish: fixed-order sums, slice kicks, append
  __threadfence();
  __syncthreads();
  if (tid == 0) last = atomicAdd(D.done, 1u) == gridDim.x - 1;
  __syncthreads();
  if (!last) return;
  __threadfence();
  const double nel = D.nelec[ib];
  double *xp = D.sl + (size_t)ib * 6 * S + 3 * S, *zp = xp + 2 * S;
  for (int c = tid; c < S; c += WS_WG) {
    double sx = 0.0, sy = 0.0;
    for (unsigned k = 0; k < gridDim.x; k++) {
      sx += D.part[((size_t)k * S + c) * 2];
      sy += D.part[((size_t)k * S + c) * 2 + 1];
    }
    const double dQ = nel * D.npop[c] * K_E;
    const double fjp = dQ > 0.0 ? P.factjp0 / dQ : 0.0;
    sx = fjp * sx;
    sy = fjp * sy;
    xp[c] = xp[c] + P.CdeltT * sx;
    zp[c] = zp[c] + P.CdeltT * sy;
  }
  // append the bunch's ions and finish the cloud sums
  double t0 = 0.0, t1 = 0.0, t2 = 0.0;
  for (int p = tid; p < npts; p += WS_WG) {
    const size_t o = (size_t)ib * npts + p;
    for (int a = 0; a < 5; a++) D.cl[a * D.cap + nF + p] = D.li[a * GP + o];
    t0 += D.li[o] * D.li[GP + o];
    t1 += D.li[o] * D.li[3 * GP + o];
    t2 += D.li[o];
  }
  t0 = wsum64(t0);
  t1 = wsum64(t1);
  t2 = wsum64(t2);
  if ((tid & 63) == 0) {
    red3[tid >> 6][0] = t0;
    red3[tid >> 6][1] = t1;
    red3[tid >> 6][2] = t2;
  }
  __syncthreads();
  if (tid < 3) {
    double s = 0.0;
    for (unsigned k = 0; k < gridDim.x; k++) s += D.psum[(size_t)k * 3 + tid];
    for (int w = 0; w < WS_WG / 64; w++) s += red3[w][tid];
    D.ion[((size_t)slot * P.G + ib) * 3 + tid] = s;
  }
  if (tid == 0) {
    *D.done = 0;
  }
}

#define WS_CH 8 // slices per chunk of a bunch's tables (a multiple of 4)
// double2 a block reads per chunk: two per lane
#define WS_BUF (2 * WS_WG)
static_assert(WS_CH * WS_QT <= WS_BUF, "a chunk fits its buffer");

// An ion's cell [kx - 3, kx - 2] x [kz - 3, kz - 2] of the grid, kx, kz in 0 .. 5 the
// floor of its grid quotient plus 3: ion_weight(x, ix, gx) is its weight in the cell
// (the quotient's fraction), in [0, 1) as long as it stays there; e1, e3 the table's
// entries of the cell's lower and upper row ends.  The outer cells have no step (in z
// because both ends are the same entry), so their weight says only whether the ion is
// still there: the quotient is scaled so that [0, 1) takes in 2^20 spacings beyond the
// grid, as far as lost ions get, and ends 2^-30 of one outside it, clear of its rounding.
// The reference anchors at the grid point nearer zero (trunc of the quotient) and weighs
// toward the next one out; above zero that is the same cell and steps, below it the same
// bilinear interpolant taken from its other end.
struct IonCell {
  double ix, iz, gx, gz;
  const double2 *e1, *e3;
};

// The weights' (ix, gx) per kx, then (iz, gz) per kz, for the kernel's LDS.
__device__ __forceinline__ double2 ion_cell_weight(const WSP &P, int i)
{
  const double far = 0x1p-20, ia = i < 6 ? P.iaAx : P.iaAz;
  const int k = i % 6;
  return make_double2(k == 0 || k == 5 ? ia * far : ia,
                      k == 0 ? 2.0 - 2.0 * far - 0x1p-50 : k == 5 ? 3.0 + 2.0 * far + 0x1p-50 : (double)k);
}

__device__ __forceinline__ double ion_weight(double x, double ix, double gx) { return fma(x, ix, 3.0) - gx; }

__device__ __forceinline__ IonCell ion_cell(const WSP &P, const double2 *qt, const double2 *wt, double x, double y)
{
  const int kx = min(max((int)floor(fma(x, P.iaAx, 3.0)), 0), 5);
  const int kz = min(max((int)floor(fma(y, P.iaAz, 3.0)), 0), 5);
  const double2 a = wt[kx], b = wt[6 + kz];
  return {a.x, b.x, a.y, b.y, qt + 5 * kx + max(kz - 1, 0), qt + 5 * kx + min(kz, 4)};
}

// The entries the cell has in a slice's table, o entries on.
struct IonField {
  double2 e1, e3, d1, d3;
};

__device__ __forceinline__ IonField ion_load(const IonCell &c, int o)
{
  return {c.e1[o], c.e3[o], c.e1[o + WS_ROWS], c.e3[o + WS_ROWS]};
}

// High words of a weight at or above this one, unsigned: outside [0, 1), or NaN.
#define ION_ONE 0x3ff00000u

// The lane's ion.
struct Ion {
  double Nri, x, xd, y, yd;
};

// One slice for the lane's ion: the field at the ion, its kick, and its share Nri E of
// the slice's kick.  f holds the entries of the ion's cell; the velocity kick
// deltT (factF E) of the reference is taken as (deltT factF) E, one fused
// multiply-add with the product precomputed (a rounding-level change).
__device__ __forceinline__ void ion_kick(const WSP &P, const IonField &f, double wx, double wz, Ion &I, double &sx,
                                         double &sy)
{
  // the bilinear steps and the kicks as fused multiply-adds (one rounding less each)
#pragma clang fp contract(fast)
  const double y5 = f.e1.y + wx * f.d1.y;
  const double y6 = f.e3.y + wx * f.d3.y;
  const double x5 = f.e1.x + wx * f.d1.x;
  const double x6 = f.e3.x + wx * f.d3.x;
  const double Ey = y5 + wz * (y6 - y5);
  const double Ex = x5 + wz * (x6 - x5);
  I.xd = I.xd + P.dtF * Ex;
  I.x = I.x + P.deltT * I.xd;
  I.yd = I.yd + P.dtF * Ey;
  I.y = I.y + P.deltT * I.yd;
  sx = I.Nri * Ex;
  sy = I.Nri * Ey;
}

// The wave's sums of v into wred: the 2 N field sums of slices c0 .. in v[0 ..], into
// rows 2 c0 .., and (CLOUD) the cloud sums Nri x, Nri y, Nri in v[4 .. 6].
template <int N, bool CLOUD>
__device__ __forceinline__ void ions_sum(const Ion &I, bool act, double v[8], int c0, int S,
                                         double (*wred)[WS_WG / 64], int lane, int wv)
{
  if (CLOUD && act) {
    v[4] = I.Nri * I.x;
    v[5] = I.Nri * I.y;
    v[6] = I.Nri;
  }
  const double t = wsum64x8(v);
  const int m = lane >> 3;
  if ((lane & 7) == 0) {
    if (m < 2 * N)
      wred[2 * c0 + m][wv] = t;
    else if (CLOUD && m >= 4 && m < 7)
      wred[2 * S + m - 4][wv] = t;
  }
}

// N <= 4 slices of a bunch from entry o of the tables on: the kicks, then the 2 N field
// sums and (CLOUD, N <= 1: the bunch's last slice) the cloud sums after them, over the
// wave in one reduction into wred from row 2 c0 on.
// Each slice's entries are read before the ion's place in the slice is known, from the
// cell it had: an ion changes cells in one of five thousand slices, and the weights
// show it (they leave [0, 1)).  Then the wave finds its cells and reads again (in one of
// sixty slices).  One test for four slices, done again from their start where it fails,
// with or without entries read a slice ahead, was no faster.
template <int N, bool CLOUD>
__device__ __forceinline__ void ions_group(const WSP &P, const double2 *qt, const double2 *wt, int o, int c0,
                                           IonCell &cl, Ion &I, double (*wred)[WS_WG / 64], int lane, int wv)
{
  double v[8] = {};
#pragma unroll
  for (int k = 0; k < N; k++) {
    const int ok = o + k * WS_QT;
    IonField f = ion_load(cl, ok);
    asm volatile("" ::: "memory"); // keeps these reads here, ahead of the branch
    double wx = ion_weight(I.x, cl.ix, cl.gx), wz = ion_weight(I.y, cl.iz, cl.gz);
    const unsigned out = max((unsigned)__double2hiint(wx), (unsigned)__double2hiint(wz));
    if (__builtin_expect(__any(out >= ION_ONE), 0)) {
      cl = ion_cell(P, qt, wt, I.x, I.y);
      f = ion_load(cl, ok);
      wx = ion_weight(I.x, cl.ix, cl.gx);
      wz = ion_weight(I.y, cl.iz, cl.gz);
    }
    ion_kick(P, f, wx, wz, I, v[2 * k], v[2 * k + 1]);
  }
  ions_sum<N, CLOUD>(I, true, v, c0, P.S, wred, lane, wv);
}

// The slices cb .. ce - 1 of a bunch (their tables at entry o; cb a multiple of 4) and,
// when they end the bunch (ce = S), the cloud sums after it.
__device__ __forceinline__ void ions_chunk(const WSP &P, const double2 *qt, const double2 *wt, int o, int cb, int ce,
                                           IonCell &cl, Ion &I, double (*wred)[WS_WG / 64], int lane, int wv)
{
  if (cb == 0) cl = ion_cell(P, qt, wt, I.x, I.y);
  int c0 = cb;
  for (; c0 + 4 <= ce; c0 += 4, o += 4 * WS_QT) ions_group<4, false>(P, qt, wt, o, c0, cl, I, wred, lane, wv);
  if (ce < P.S) return;
  // one slice left or three: their number is odd
  if (P.S - c0 == 3) {
    ions_group<3, false>(P, qt, wt, o, c0, cl, I, wred, lane, wv);
    ions_group<0, true>(P, qt, wt, o, P.S, cl, I, wred, lane, wv);
  } else
    ions_group<1, true>(P, qt, wt, o, c0, cl, I, wred, lane, wv);
}

// The slices of a chunk in a bunch that some of the lanes' ions are not yet made in:
// only those in the cloud (act) move and count.
__device__ __forceinline__ void ions_chunk_some(const WSP &P, const double2 *qt, const double2 *wt, int o, int cb,
                                                int ce, bool act, Ion &I, double (*wred)[WS_WG / 64], int lane,
                                                int wv)
{
  for (int c = cb; c < ce; c++, o += WS_QT) {
    double v[8] = {};
    if (act) {
      const IonCell cl = ion_cell(P, qt, wt, I.x, I.y);
      ion_kick(P, ion_load(cl, o), ion_weight(I.x, cl.ix, cl.gx), ion_weight(I.y, cl.iz, cl.gz), I, v[0], v[1]);
    }
    ions_sum<1, false>(I, act, v, c, P.S, wred, lane, wv);
  }
  if (ce < P.S) return;
  double v[8] = {};
  ions_sum<0, true>(I, act, v, 0, P.S, wred, lane, wv);
}

// A barrier for what the block shares in LDS alone: loads and stores of global
// memory stay under way across it (__syncthreads waits for them).
__device__ __forceinline__ void lds_barrier()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Ion-parallel train: lane q carries ion q = j * Nions + p (ion p made by bunch
// j, its state after the creator's later slices) through bunches j+1 .. G-1,
// each reached after its drift time.  Per bunch ib the block writes the 2 S
// slice sums of Nri * E and the cloud sums Nri x, Nri y, Nri after the bunch,
// each the fixed-order sum of its four waves' sums.  The bunches up to the
// block's last creator (some ions not yet made) run with per-lane
// predicates, the rest without.
// Bound: vector issue for a long train, of 356 bunches 92 % of the kernel's cycles with
// 34.7 instructions a lane, ion and slice, 61 % of them FP64; a slice's latency for a
// short one, of 61 bunches 364 cycles per slice in the chain of the longest block's
// (G - 1) S slices, with one wave per SIMD and vector issue 19 % of the cycles.  (The
// long train's chain is 80 % of its time at that rate.)  So the chain has no wait for
// memory in it: the tables of a bunch come ready-made in chunks of WS_CH slices through two buffers
// in LDS, one barrier a chunk (for LDS alone), the next chunk's entries on their way in
// registers while a chunk is used, and a slice's reads don't wait for its cell.  A
// chunk is read in full: past the bunch's last slice it holds the next bunch's tables,
// past the last bunch's the room left for it.  356 bunches x 41 slices 3.03 -> 2.82 ms,
// 61 x 39 421 -> 350 us, results the same to the bit (tables built from the grid fields
// by every block, waited for; the cell found in every slice).  In trials of this form
// 16 slices a chunk were better for the short train by 8 % and worse for the long by
// 6 %, 4 or 6 waves per SIMD worse, two ions per lane 1.2 and 1.6 times slower.
__global__ __launch_bounds__(WS_WG, 5) void k_ws_ions(WSP P, WSD D)
{
  constexpr int NW = WS_WG / 64;
  __shared__ double2 qt[2 * WS_BUF];
  __shared__ double2 wt[12];
  __shared__ double wredb[2][2 * WS_S + 3][NW];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, S = P.S, npts = S * 25, NQ = 2 * S + 3;
  const size_t GP = (size_t)P.G * npts;
  const long long nI = (long long)(P.G - 1) * npts;
  // Dispatch order: a block's work is the number of bunches after its ions'
  // creator, longest first.  Blocks are dealt to the CUs round-robin, so
  // blocks c, c + 256, c + 512, ... share a CU: in each run of 512 blocks
  // (or the last, shorter run, if it holds more than 256) block c takes the
  // logical block 255 - c and block c + 256 the logical block 256 + c, so
  // that every CU holds pairs of the same total work instead of the longest
  // trains on the first CUs (measured 4 % on the 356-bunch train).  Every
  // logical block computes and writes what it would at its own index.
  int L = blockIdx.x;
  {
    const int c = L & 255, k = L >> 8, base = (k >> 1) * 512;
    if ((int)gridDim.x - base > 256) L = (k & 1) ? base + 256 + c : base + 255 - c;
  }
  const long long q0 = (long long)L * WS_WG, q = q0 + tid;
  const int jmin = (int)(q0 / npts);
  const int jmax = (int)(min(q0 + WS_WG - 1, nI - 1) / npts);
  double2 g0, g1;
  const auto fetch = [&](int ib, int cb) {
    const double2 *t = D.tab + ((size_t)ib * S + cb) * WS_QT + tid;
    g0 = t[0];
    g1 = t[WS_WG];
  };
  const auto stage = [&](int o) {
    qt[o + tid] = g0;
    qt[o + WS_WG + tid] = g1;
  };
  fetch(jmin + 1, 0);
  const bool valid = q < nI;
  const int j = valid ? (int)(q / npts) : P.G;
  Ion I = {0.0, 0.0, 0.0, 0.0, 0.0};
  if (valid) I = {D.li[q], D.li[GP + q], D.li[2 * GP + q], D.li[3 * GP + q], D.li[4 * GP + q]};
  if (tid < 12) wt[tid] = ion_cell_weight(P, tid);
  stage(0);
  lds_barrier();
  IonCell cl;
  int o = 0;
  for (int ib = jmin + 1; ib < P.G; ib++) {
    double(*wred)[NW] = wredb[ib & 1];
    const double dt = D.dtime[ib];
    const long long to = D.toff[ib];
    const bool act = ib > jmax || j < ib;
    if (act) {
      I.x = I.x + dt * I.xd;
      I.y = I.y + dt * I.yd;
    }
    for (int cb = 0; cb < S; cb += WS_CH) {
      const int ce = min(S, cb + WS_CH);
      if (ce < S)
        fetch(ib, ce);
      else
        fetch(min(ib + 1, P.G - 1), 0);
      if (ib <= jmax)
        ions_chunk_some(P, qt, wt, o, cb, ce, act, I, wred, lane, wv);
      else
        ions_chunk(P, qt, wt, o, cb, ce, cl, I, wred, lane, wv);
      // the other buffer's last readers are a barrier behind
      o = WS_BUF - o;
      stage(o);
      lds_barrier();
    }
    // quantity-major, so that k_ws_ksum reads each quantity's partials contiguously;
    // the bunch after next is the first to write its sums over these, a barrier on
    const long long nbi = min(((long long)ib * npts + WS_WG - 1) / WS_WG, (long long)D.nblk_ions);
    for (int i = tid; i < NQ; i += WS_WG) {
      double v = 0.0;
      for (int w = 0; w < NW; w++) v += wred[i][w];
      D.tpart[to + i * nbi + L] = v;
    }
  }
}

// Per bunch ib (blockIdx.x) and group of KSUM_Q quantities (blockIdx.y): the
// blocks' partials summed in a fixed order, one quantity per wave (lane l adds
// blocks l, l + 64, ... in turn, then the wave sum), into D.tot[ib][i].  The
// last group but one of each bunch sums instead the bunch's own ions (Nri x, Nri
// y, Nri over its S * 25 ions, four waves' sums in order) into D.tot[ib][NQ + 3 w
// + m], which the kicks add to the cloud sums after the bunch.  The last group is
// phase 2 of the turn (nothing of the train reads the slices once the ions are
// made), a launch fewer per turn.
#define KSUM_Q 8
__global__ __launch_bounds__(64 * KSUM_Q) void k_ws_ksum(WSP P, WSD D, WSStep T)
{
  extern __shared__ double2 sm[];
  if (blockIdx.y == gridDim.y - 1) {
    ws_electrons(P, D, blockIdx.x, T, sm);
    return;
  }
  const int ib = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, S = P.S, npts = S * 25;
  const int NQ = 2 * S + 3;
  double *tot = D.tot + (size_t)ib * WS_TQ;
  if (blockIdx.y == gridDim.y - 2) {
    if (tid >= WS_WG) return;
    const size_t GP = (size_t)P.G * npts;
    double t0 = 0.0, t1 = 0.0, t2 = 0.0;
    for (int p = tid; p < npts; p += WS_WG) {
      const size_t o = (size_t)ib * npts + p;
      t0 += D.li[o] * D.li[GP + o];
      t1 += D.li[o] * D.li[3 * GP + o];
      t2 += D.li[o];
    }
    t0 = wsum64(t0);
    t1 = wsum64(t1);
    t2 = wsum64(t2);
    if (lane == 0) {
      tot[NQ + 3 * wv] = t0;
      tot[NQ + 3 * wv + 1] = t1;
      tot[NQ + 3 * wv + 2] = t2;
    }
    return;
  }
  const int i = blockIdx.y * KSUM_Q + wv;
  if (ib == 0 || i >= NQ) return;
  long long nb = ((long long)ib * npts + WS_WG - 1) / WS_WG; // blocks of k_ws_ions ahead of ib
  if (nb > D.nblk_ions) nb = D.nblk_ions;
  const double *tp = D.tpart + D.toff[ib] + i * nb;
  double v = 0.0;
#pragma unroll 4
  for (long long k = lane; k < nb; k += 64) v += tp[k];
  v = wsum64(v);
  if (lane == 0) tot[i] = v;
}

// ================================================================ host side

struct mbt_ws {
  mbt_config cfg;
  int device;
  hipStream_t stream;
  WSP P;
  WSD D;
  int *d_bucket, *d_npop, *d_nofe;
  double *d_wallcur, *d_nelec, *d_convion;
  int *bucket_h;
  int npop_h[WS_S];
  double *dist; // generated macro-electrons [6][Np]
  double *nelec_h;
  long long rev;
  int maxblk;
  int serial;          // bunch-by-bunch relay instead of the ion-parallel train
  double *d_dtime, *d_wall;
  long long *d_toff;
  int timing;         // HIP events around the ion train of every turn
  hipEvent_t *ev;     // [2 WS_T] train start / end per turn of a block
  double train_ms;    // summed train time of the last mbt_ws_track call
  long train_launches;
  long async_n;       // turns enqueued by mbt_ws_track_async, not yet collected (0: none)
};

// Tracking calls that would overwrite the output block of turns enqueued by
// mbt_ws_track_async fail while those turns are pending.
static int ws_no_pending(const mbt_ws *w)
{
  if (w->async_n) {
    mbt_set_error("%ld turns enqueued by mbt_ws_track_async are pending: collect them with mbt_ws_track_wait",
                  w->async_n);
    return MBT_EINVAL;
  }
  return MBT_OK;
}

extern "C" void mbt_ws_destroy(mbt_ws *w)
{
  if (!w) return;
  (void)hipSetDevice(w->device);
  if (w->stream) (void)hipStreamSynchronize(w->stream); // turns of mbt_ws_track_async may still run
  void *p[] = {w->D.sl,  w->D.dip, w->d_wall, w->D.Exy, w->D.li,     w->D.cl,     w->D.part,    w->D.psum,
               w->D.done, w->D.cm,  w->D.mon,  w->D.ion, w->D.zcm,    w->d_bucket, w->d_npop,
               w->d_nofe, w->d_wallcur, w->d_nelec, w->d_convion, w->D.tpart, w->d_dtime, w->d_toff,
               w->D.tot,  w->D.tab};
  for (size_t i = 0; i < sizeof p / sizeof p[0]; i++)
    if (p[i]) (void)hipFree(p[i]);
  if (w->ev)
    for (int i = 0; i < 2 * WS_T; i++) (void)hipEventDestroy(w->ev[i]);
  free(w->ev);
  if (w->stream) (void)hipStreamDestroy(w->stream);
  free(w->bucket_h);
  free(w->dist);
  free(w->nelec_h);
  free(w);
}

template <typename T> static int walloc(T **p, size_t n)
{
  if (n == 0) n = 1;
  if (hipMalloc((void **)p, n * sizeof(T)) != hipSuccess) {
    mbt_set_error("hipMalloc of %zu bytes failed", n * sizeof(T));
    return MBT_ENOMEM;
  }
  return hipMemset(*p, 0, n * sizeof(T)) == hipSuccess ? MBT_OK : MBT_EDEVICE;
}

#define WA(p, n)                                                                                 \
  do {                                                                                           \
    int rc_ = walloc(&(p), (size_t)(n));                                                         \
    if (rc_) {                                                                                   \
      mbt_ws_destroy(w);                                                                         \
      return rc_;                                                                                \
    }                                                                                            \
  } while (0)
#define WUP(dst, src, n) CK(hipMemcpyAsync((dst), (src), (size_t)(n) * sizeof(*(src)), hipMemcpyHostToDevice, w->stream))

extern "C" int mbt_ws_create(const mbt_config *c, int device, int flags, mbt_ws **out)
{
  *out = NULL;
  if (c->bunch_model != 1) {
    mbt_set_error("mbt_ws_create needs BunchModel = STRONG");
    return MBT_EINVAL;
  }
  const int S = 2 * c->Nslc + 1, H = (int)c->Nharm, G = c->Nbunch;
  if (c->Nslc < 0 || S > WS_S || H > 500 || G <= 0 || c->NmultiT > WS_HIST || c->Nmlt + 2 > WS_HIST ||
      c->NrevMon <= 0) {
    mbt_set_error("weak-strong limits: 2 Nslc + 1 <= 50, h <= 500, Nmlt + 2 <= 30, NrevMon > 0");
    return MBT_EINVAL;
  }
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= device) {
    mbt_set_error("no HIP device %d", device);
    return MBT_EDEVICE;
  }
  mbt_ws *w = (mbt_ws *)calloc(1, sizeof *w);
  w->cfg = *c;
  w->cfg.nfFill = NULL;
  w->cfg.Ibunch = NULL;
  w->cfg.bucket = NULL;
  w->cfg.bunch_Ib = NULL;
  w->cfg.Ib_frac = NULL;
  w->cfg.bunch_out = NULL;
  w->device = device;
  CK(hipSetDevice(device));
  CK(hipStreamCreate(&w->stream));
  // ---- slices, populations, grid counts (host, the reference's generator)
  double *slices = (double *)malloc(sizeof(double) * 6 * (size_t)S * H);
  int nofe[WS_PTS];
  w->dist = (double *)malloc(sizeof(double) * 6 * (size_t)(c->Np > 0 ? c->Np : 1));
  int rc = mbt_ws_generate(c, slices, w->npop_h, nofe, w->dist);
  if (rc) {
    free(slices);
    mbt_ws_destroy(w);
    return rc;
  }
  w->bucket_h = (int *)malloc(sizeof(int) * G);
  memcpy(w->bucket_h, c->bucket, sizeof(int) * G);
  double *Ib = (double *)calloc(H, sizeof(double));
  if (flags & MBT_WS_BUNCH_CURRENTS) memcpy(Ib, c->Ibunch, sizeof(double) * H);
  // ---- constants (glibc on the host, the reference's expressions)
  WSP &P = w->P;
  P.S = S;
  P.G = G;
  P.h = H;
  P.Nmlt = c->Nmlt;
  P.NmultiT = c->NmultiT;
  P.fbii = c->EnableFBII != 0;
  P.rw = c->EnableRW_long != 0;
  P.track_h = c->TrackPlane[1] != 0;
  P.track_v = c->TrackPlane[2] != 0;
  for (int p = 0; p < 3; p++) P.track[p] = c->TrackPlane[p] != 0;
  P.Nions = S * 25;
  P.mixed = (flags & MBT_WS_MIXED) ? 1 : 0;
  P.eps = c->Vrf0 / (c->E0 * MBT_FKILO);
  P.wrf = c->wrf;
  P.phai0 = c->phai0;
  P.Urad = c->Urad;
  P.T0 = c->T0;
  P.ac = c->ac;
  double prfrw[2], prfrw_trig[2]; // wake strengths of the resistive wall, the second with the trigger
  for (int p = 0; p < 3; p++) {
    P.gamma1[p] = c->gamma1[p];
    P.alpha1[p] = c->alpha1[p];
    P.beta1[p] = c->beta1[p];
  }
  {
    double PsiV0 = 2.0 * M_PI * c->QV0 / 1.0, PsiH0 = 2.0 * M_PI * c->QH0 / 1.0;
    double cv = cos(PsiV0), sv = sin(PsiV0), ch = cos(PsiH0), sh = sin(PsiH0);
    P.v11 = cv + c->alpha1[2] * sv;
    P.v12 = c->beta1[2] * sv;
    P.v21 = -c->gamma1[2] * sv;
    P.v22 = cv - c->alpha1[2] * sv;
    P.h11 = ch + c->alpha1[1] * sh;
    P.h12 = c->beta1[1] * sh;
    P.h21 = -c->gamma1[1] * sh;
    P.h22 = ch - c->alpha1[1] * sh;
    for (int pl = 0; pl < 2; pl++) {
      const int plane = pl + 1;
      double Psi0 = 2.0 * M_PI * (plane == 1 ? c->QH0 : c->QV0) / 1.0;
      double Psi = 0.0 + Psi0;
      double cp = cos(Psi), sp = sin(Psi);
      P.rwa11[pl] = cp + c->alpha1[plane] * sp;
      P.rwa12[pl] = +c->beta1[plane] * sp;
      const double kappa = 1.0 / 2.8e-08;
      double beff3 = pow(plane == 1 ? c->beffH[0] : c->beffV[0], 3);
      prfrw[pl] = 2.0 * c->R / (beff3) / sqrt(M_PI * kappa * K_EPS0) / 1.0;
      beff3 = pow(2.0e-3, 3);
      prfrw_trig[pl] = 2.0 * c->R / (beff3) / sqrt(M_PI * kappa * K_EPS0) / 1.0;
    }
  }
  P.triggerRW = c->triggerRW;
  P.fNp = c->fNp;
  for (int i = 0; i < S; i++) P.ntot += w->npop_h[i];
  P.factBE = sqrt(2 * (c->sgm_xx * c->sgm_xx - c->sgm_zz * c->sgm_zz)) / MBT_FKILO;
  P.sxx = c->sgm_xx;
  P.szz = c->sgm_zz;
  P.deltT = 0.3 * c->sgmatau;
  mbt_ws_grid(c, &P.aLx, &P.aLz);
  P.aAx = 2.0 * P.aLx;
  P.aAz = 2.0 * P.aLz;
  P.iaAx = 1.0 / P.aAx;
  P.iaAz = 1.0 / P.aAz;
  P.den_dQ = 2 * K_EPS0 * sqrt(M_PI) * P.factBE * K_C * P.deltT;
  {
    double Pave = 2.7e-9, Pu20 = 5 * Pave, Pm = 0.15 * Pu20 / 1.3332, dm = 3.22e22 * Pm, sigmam = 1.78;
    double Lu20 = 354.0, Ldmsgm = Lu20 * dm * sigmam * 1e-22;
    P.factF = K_E / (28.0 * 1.836e3 * 9.1e-31);
    P.factjp0 = 1e+2 * 4.0 * M_PI * K_EPS0 * 2.819e-15 / c->Gamma;
    P.CdeltT = K_C * P.deltT;
    P.dtF = P.deltT * P.factF;
    w->nelec_h = (double *)malloc(sizeof(double) * G);
    const double Pref0 = c->T0 / c->E0 / c->fNp / MBT_FTERA;
    double *conv = (double *)malloc(sizeof(double) * G), *wcur = (double *)malloc(sizeof(double) * G);
    for (int b = 0; b < G; b++) {
      w->nelec_h[b] = (Ib[c->bucket[b]] * c->T0 / (c->Np * K_E * MBT_FKILO));
      conv[b] = w->nelec_h[b] * Ldmsgm;
      wcur[b] = c->nfFill[c->bucket[b]] ? Pref0 * Ib[c->bucket[b]] : 0.0; // only filled buckets act
    }
    // ---- device memory
    const size_t npts = (size_t)S * 25;
    WA(w->D.sl, (size_t)G * 6 * S);
    WA(w->d_npop, S);
    WA(w->d_nofe, npts);
    WA(w->d_bucket, G);
    WA(w->d_wallcur, G);
    WA(w->d_nelec, G);
    WA(w->d_convion, G);
    if (P.rw) {
      // the wake W = prf / sqrt(D / c) of every distance a dipole can act over, D =
      // d buckets (d = h: the bunch's own, one turn) and j turns; none without a tap
      const size_t nw = c->Nmlt < 0 ? 0 : (size_t)4 * (c->Nmlt + 1) * H;
      double *wl = (double *)malloc(sizeof(double) * nw);
      const double Dub0 = c->Lc / ((double)c->Nharm);
      for (int t = 0, i = 0; t < 2; t++)
        for (int pl = 0; pl < 2; pl++)
          for (int j = 0; j <= c->Nmlt; j++)
            for (int d = 1; d <= H; d++, i++) {
              const double D0 = d == H ? c->Lc : ((double)d) * Dub0, Du = D0 + ((double)j) * c->Lc;
              const double Dt = Du / K_C;
              wl[i] = (t ? prfrw_trig[pl] : prfrw[pl]) / sqrt(Dt);
            }
      const int rca = walloc(&w->d_wall, nw);
      if (!rca && hipMemcpy(w->d_wall, wl, sizeof(double) * nw, hipMemcpyHostToDevice) != hipSuccess) rc = MBT_EDEVICE;
      free(wl);
      if (rca || rc) {
        mbt_ws_destroy(w);
        return rca ? rca : rc;
      }
      WA(w->D.dip, (size_t)2 * WS_RING * G);
    }
    WA(w->D.Exy, (size_t)G * npts);
    WA(w->D.li, (size_t)5 * G * npts);
    // train: drift times, then the ion-parallel form's partials (one block
    // row per bunch for every block holding an ion made ahead of it), or the
    // relay's cloud when those would not fit
    double *dt = (double *)calloc(G, sizeof(double));
    for (int ib = 1; ib < G; ib++) dt[ib] = fabs((double)(w->bucket_h[ib] - w->bucket_h[ib - 1])) * (c->T0 / c->h);
    WA(w->d_dtime, G);
    WUP(w->d_dtime, dt, G);
    CK(hipStreamSynchronize(w->stream));
    free(dt);
    const int NQ = 2 * S + 3;
    const long long nI = (long long)(G - 1) * (long long)npts;
    w->D.nblk_ions = (int)((nI + WS_WG - 1) / WS_WG);
    long long *toff = (long long *)malloc(sizeof(long long) * G), ntp = 0;
    for (int ib = 0; ib < G; ib++) {
      toff[ib] = ntp;
      long long nb = ((long long)ib * (long long)npts + WS_WG - 1) / WS_WG;
      if (nb > w->D.nblk_ions) nb = w->D.nblk_ions;
      ntp += nb * NQ;
    }
    w->serial = (flags & MBT_WS_SERIAL_TRAIN) || G < 2 || ntp * (long long)sizeof(double) > WS_TRAIN_PARTIAL_MAX;
    if (!w->serial && P.fbii) {
      WA(w->D.tpart, ntp);
      WA(w->D.tab, (size_t)G * S * WS_QT + WS_BUF);
      WA(w->D.tot, (size_t)G * WS_TQ);
      WA(w->d_toff, G);
      WUP(w->d_toff, toff, G);
      CK(hipStreamSynchronize(w->stream));
    } else if (P.fbii) {
      w->D.cap = (long long)G * npts;
      WA(w->D.cl, (size_t)5 * w->D.cap);
      w->maxblk = (int)((w->D.cap + WS_WG - 1) / WS_WG);
      WA(w->D.part, (size_t)w->maxblk * S * 2);
      WA(w->D.psum, (size_t)w->maxblk * 3);
    }
    free(toff);
    WA(w->D.done, 1);
    WA(w->D.cm, (size_t)WS_T * G * 4);
    WA(w->D.mon, (size_t)WS_T * G * 18);
    WA(w->D.ion, (size_t)WS_T * G * 3);
    WA(w->D.zcm, (size_t)WS_T * H);
    double *sl = (double *)malloc(sizeof(double) * 6 * (size_t)S * G);
    for (int b = 0; b < G; b++)
      memcpy(sl + (size_t)b * 6 * S, slices + (size_t)c->bucket[b] * 6 * S, sizeof(double) * 6 * S);
    WUP(w->D.sl, sl, (size_t)G * 6 * S);
    WUP(w->d_npop, w->npop_h, S);
    WUP(w->d_nofe, nofe, npts);
    WUP(w->d_bucket, w->bucket_h, G);
    WUP(w->d_wallcur, wcur, G);
    WUP(w->d_nelec, w->nelec_h, G);
    WUP(w->d_convion, conv, G);
    CK(hipStreamSynchronize(w->stream));
    free(sl);
    free(conv);
    free(wcur);
  }
  free(slices);
  free(Ib);
  w->D.npop = w->d_npop;
  w->D.nofe = w->d_nofe;
  w->D.bucket = w->d_bucket;
  w->D.wallcur = w->d_wallcur;
  w->D.nelec = w->d_nelec;
  w->D.convion = w->d_convion;
  w->D.dtime = w->d_dtime;
  w->D.toff = w->d_toff;
  w->D.wall = w->d_wall;
  *out = w;
  return MBT_OK;
}

static int ws_download(mbt_ws *w, long n, double *cm, double *mon, double *ion, double *zcm)
{
  CK(hipStreamSynchronize(w->stream));
  const int G = w->P.G, H = w->P.h;
  if (cm) CK(hipMemcpy(cm, w->D.cm, sizeof(double) * 4 * G * n, hipMemcpyDeviceToHost));
  if (mon) CK(hipMemcpy(mon, w->D.mon, sizeof(double) * 18 * G * n, hipMemcpyDeviceToHost));
  if (ion) CK(hipMemcpy(ion, w->D.ion, sizeof(double) * 3 * G * n, hipMemcpyDeviceToHost));
  if (zcm) CK(hipMemcpy(zcm, w->D.zcm, sizeof(double) * H * n, hipMemcpyDeviceToHost));
  return MBT_OK;
}

// Enqueues n <= WS_T turns on the object's stream, their outputs in slots
// 0 .. n-1 of the device's output block (with HIP events around each ion train
// when timing is on).
static int ws_enqueue(mbt_ws *w, long n)
{
  const int G = w->P.G, S = w->P.S;
  const size_t lds = sizeof(double) * ws_electrons_lds(S, G);
  const bool fbii = w->P.fbii != 0, relay = fbii && w->serial;
  // phase 1 with FBII: a block per bunch, then one thread per grid point of every
  // slice of every bunch (for the fields, then the ions)
  const long long np = (long long)G * S * 25;
  const int nbp = (int)((np + WS_WG - 1) / WS_WG);
  CK(hipMemsetAsync(w->D.mon, 0, sizeof(double) * 18 * G * n, w->stream));
  CK(hipMemsetAsync(w->D.ion, 0, sizeof(double) * 3 * G * n, w->stream));
  int kick = -1; // slot of the turn whose ion kicks are still to apply
  for (long t = 0; t < n; t++) {
    const long long rev = w->rev;
    WSStep T = {kick, -1, 0, rev, (int)t, rev % w->cfg.NrevMon == 0};
    kick = -1;
    if (!fbii) {
      if (t > 0) {
        T.rev2 = rev - 1;
        T.slot2 = (int)t - 1;
      }
      hipLaunchKernelGGL(k_ws_step, dim3(G), dim3(WS_STEP_WG), lds, w->stream, w->P, w->D, T);
      CK(hipGetLastError());
      w->rev++;
      continue;
    }
    hipLaunchKernelGGL(k_ws_phase1, dim3(G + nbp), dim3(WS_WG), lds, w->stream, w->P, w->D, T);
    CK(hipGetLastError());
    // the ions start from the slices' positions before the betatron rotation
    const int nbt = relay ? 0 : (int)(((long long)G * S * WS_ROWS + WS_WG - 1) / WS_WG);
    hipLaunchKernelGGL(k_ws_create, dim3(nbp + nbt), dim3(WS_WG), 0, w->stream, w->P, w->D);
    CK(hipGetLastError());
    const WSStep T2 = {-1, rev, (int)t, -1, 0, 0};
    if (!relay) {
      if (w->timing) CK(hipEventRecord(w->ev[2 * t], w->stream));
      hipLaunchKernelGGL(k_ws_ions, dim3(w->D.nblk_ions), dim3(WS_WG), 0, w->stream, w->P, w->D);
      CK(hipGetLastError());
      if (w->timing) CK(hipEventRecord(w->ev[2 * t + 1], w->stream));
      hipLaunchKernelGGL(k_ws_ksum, dim3(G, (2 * S + 3 + KSUM_Q - 1) / KSUM_Q + 2), dim3(64 * KSUM_Q), lds, w->stream,
                         w->P, w->D, T2);
      CK(hipGetLastError());
      kick = (int)t;
    } else {
      hipLaunchKernelGGL(k_ws_step, dim3(G), dim3(WS_STEP_WG), lds, w->stream, w->P, w->D, T2);
      CK(hipGetLastError());
      if (w->timing) CK(hipEventRecord(w->ev[2 * t], w->stream));
      hipLaunchKernelGGL(k_ws_cloud_reset, dim3(1), dim3(WS_WG), 0, w->stream, w->P, w->D, (int)t);
      CK(hipGetLastError());
      for (int ib = 1; ib < G; ib++) {
        const long long nF = (long long)ib * w->P.Nions;
        const double Dtime =
            fabs((double)(w->bucket_h[ib] - w->bucket_h[ib - 1])) * (w->cfg.T0 / w->cfg.h);
        const int nblk = (int)((nF + WS_WG - 1) / WS_WG);
        hipLaunchKernelGGL(k_ws_train, dim3(nblk), dim3(WS_WG), 0, w->stream, w->P, w->D, ib, nF, Dtime, (int)t);
        CK(hipGetLastError());
      }
      if (w->timing) CK(hipEventRecord(w->ev[2 * t + 1], w->stream));
    }
    w->rev++;
  }
  // what the last turn leaves: its phase 2 (without FBII) or its train's kicks
  const WSStep T = {kick, fbii ? -1 : w->rev - 1, (int)n - 1, -1, 0, 0};
  if (n > 0 && (!fbii || kick >= 0)) {
    hipLaunchKernelGGL(k_ws_step, dim3(G), dim3(WS_STEP_WG), lds, w->stream, w->P, w->D, T);
    CK(hipGetLastError());
  }
  return MBT_OK;
}

extern "C" int mbt_ws_track(mbt_ws *w, long nturns, double *cm, double *mon, double *ion, double *zcm)
{
  int rc;
  if ((rc = ws_no_pending(w))) return rc;
  CK(hipSetDevice(w->device));
  (void)hipGetLastError();
  const int G = w->P.G, H = w->P.h;
  long done = 0;
  w->train_ms = 0.0;
  w->train_launches = 0;
  while (done < nturns) {
    long n = nturns - done;
    if (n > WS_T) n = WS_T;
    if ((rc = ws_enqueue(w, n))) return rc;
    if (w->timing && w->P.fbii) {
      CK(hipStreamSynchronize(w->stream));
      for (long t = 0; t < n; t++) {
        float ms = 0.0f;
        CK(hipEventElapsedTime(&ms, w->ev[2 * t], w->ev[2 * t + 1]));
        w->train_ms += ms;
        w->train_launches++;
      }
    }
    rc = ws_download(w, n, cm ? cm + (size_t)done * G * 4 : NULL, mon ? mon + (size_t)done * G * 18 : NULL,
                     ion ? ion + (size_t)done * G * 3 : NULL, zcm ? zcm + (size_t)done * H : NULL);
    if (rc) return rc;
    done += n;
  }
  return MBT_OK;
}

extern "C" long mbt_ws_async_max(const mbt_ws *w)
{
  (void)w;
  return WS_T;
}

extern "C" int mbt_ws_track_async(mbt_ws *w, long nturns)
{
  int rc;
  if ((rc = ws_no_pending(w))) return rc;
  if (nturns < 1 || nturns > WS_T) {
    mbt_set_error("mbt_ws_track_async: 1 .. %d turns per call", WS_T);
    return MBT_EINVAL;
  }
  if (w->timing) {
    mbt_set_error("mbt_ws_track_async: not with train timing on");
    return MBT_EINVAL;
  }
  CK(hipSetDevice(w->device));
  (void)hipGetLastError(); // launch checks below must not report an earlier call's error
  if ((rc = ws_enqueue(w, nturns))) return rc;
  w->async_n = nturns;
  return MBT_OK;
}

extern "C" int mbt_ws_track_wait(mbt_ws *w, double *cm, double *mon, double *ion, double *zcm)
{
  if (!w->async_n) {
    mbt_set_error("mbt_ws_track_wait: no turns pending");
    return MBT_EINVAL;
  }
  CK(hipSetDevice(w->device));
  const long n = w->async_n;
  w->async_n = 0;
  return ws_download(w, n, cm, mon, ion, zcm);
}

extern "C" int mbt_ws_get_slices(const mbt_ws *w, int ib, double *out)
{
  if (ib < 0 || ib >= w->P.G) return MBT_EINVAL;
  CK(hipSetDevice(w->device));
  CK(hipStreamSynchronize(w->stream));
  CK(hipMemcpy(out, w->D.sl + (size_t)ib * 6 * w->P.S, sizeof(double) * 6 * w->P.S, hipMemcpyDeviceToHost));
  return MBT_OK;
}

extern "C" int mbt_ws_population(const mbt_ws *w, int *npop, int *nslices)
{
  for (int i = 0; i < w->P.S; i++) npop[i] = w->npop_h[i];
  if (nslices) *nslices = w->P.S;
  return MBT_OK;
}

extern "C" int mbt_ws_distribution(const mbt_ws *w, double *dist)
{
  memcpy(dist, w->dist, sizeof(double) * 6 * (size_t)w->cfg.Np);
  return MBT_OK;
}

extern "C" long mbt_ws_turn(const mbt_ws *w) { return (long)w->rev; }

extern "C" int mbt_ws_set_timing(mbt_ws *w, int on)
{
  CK(hipSetDevice(w->device));
  if (on && !w->ev) {
    w->ev = (hipEvent_t *)calloc(2 * WS_T, sizeof(hipEvent_t));
    if (!w->ev) return MBT_ENOMEM;
    for (int i = 0; i < 2 * WS_T; i++) CK(hipEventCreate(&w->ev[i]));
  }
  w->timing = on ? 1 : 0;
  return MBT_OK;
}

extern "C" int mbt_ws_train_time(const mbt_ws *w, double *ms, long *launches)
{
  if (!w || !ms || !launches) {
    mbt_set_error("mbt_ws_train_time: null argument");
    return MBT_EINVAL;
  }
  *ms = w->train_ms;
  *launches = w->train_launches;
  return MBT_OK;
}
