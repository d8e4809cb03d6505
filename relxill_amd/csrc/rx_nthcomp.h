// rx_nthcomp.h -- device building blocks of the nthcomp primary continuum
// (c_donthcomp, src/donthcomp.c:683-793; spec_nthcomp, src/Xillspec.cpp:243-253),
// shared by the rx_nthcomp kernels and the relxill primary of the nthcomp
// models.
#pragma once

#include <hip/hip_runtime.h>

#include "rx_engine.h"

namespace rx {

constexpr int NTH_N = NTH_MAX_POINTS;  // photon energies (the reference's arrays of 900)

namespace {

// diskbb interpolation formula (f_mcdint__, src/donthcomp.c:50-115): the
// model's published coefficients
__constant__ double c_mcd_gc[3] = {.078196667, -1.066202, 1.192418};
__constant__ double c_mcd_gw[3] = {.5207874, .513457, .4077983};
__constant__ double c_mcd_gn[3] = {.3728691, .039775528, .037766505};
__constant__ double c_mcd_res[98] = {
    9.6198382e-4,   .0010901181,    .0012310012,    .0013841352,    .0015481583,    .0017210036,
    .0018988943,    .002076939,     .0022484281,    .0024049483,    .0025366202,    .0026316255,
    .0026774985,    .0026613059,    .0025708784,    .0023962965,    .002130655,     .0017725174,
    .0013268656,    8.0657672e-4,   2.3337584e-4,   -3.6291778e-4,  -9.4443569e-4,  -.0014678875,
    -.0018873741,   -.0021588493,   -.0022448371,   -.0021198179,   -.0017754602,   -.0012246034,
    -5.0414167e-4,  3.2507078e-4,   .0011811065,    .0019673402,    .0025827094,    .0029342526,
    .0029517083,    .0026012166,    .0018959062,    9.0128649e-4,   -2.6757144e-4,  -.0014567885,
    -.002492855,    -.0032079776,   -.0034678637,   -.0031988217,   -.0024080969,   -.001193624,
    2.6134145e-4,   .0017117758,    .0028906898,    .0035614435,    .0035711778,    .0028921374,
    .0016385898,    4.9857464e-5,   -.0015572671,   -.0028578151,   -.0035924212,   -.0036253044,
    -.002975086,    -.0018044436,   -3.7796664e-4,  .0010076215,    .0020937327,    .0027090854,
    .0028031667,    .0024276576,    .0017175597,    8.1030795e-4,   -1.2592304e-4,  -9.4888491e-4,
    -.0015544816,   -.0018831972,   -.0019203142,   -.0016905849,   -.0012487737,   -6.6789911e-4,
    -2.7079461e-5,  5.9931935e-4,   .0011499748,    .0015816521,    .0018709224,    .0020129966,
    .0020184702,    .0019089181,    .0017122289,    .001458377,     .0011760717,    8.9046768e-4,
    6.2190822e-4,   3.8553762e-4,   1.9155022e-4,   4.5837109e-5,   -4.9177834e-5,  -9.3670762e-5,
    -8.9622968e-5,  -4.01538532e-5};
// five-point Gauss-Legendre weights and nodes of f_xsdskb__ (:149-151)
__constant__ double c_gl_w[5] = {.236926885, .47862867, .568888888, .47862867, .236926885};
__constant__ double c_gl_x[5] = {-.906179846, -.53846931, 0., .53846931, .906179846};

__device__ inline double nth_lg10(double x) {
#pragma clang fp contract(off)
  return 0.43429448190325182765 * log(x);  // d_lg10, src/donthcomp.c:41-45
}

__device__ inline double nth_mcd_shape(double et) {
#pragma clang fp contract(off)
  const double loget = nth_lg10(et);
  double pos = (loget - nth_lg10(0.001)) / .06 + 1;
  const int j = (int)pos;
  double resfact;
  if (j < 1) {
    resfact = c_mcd_res[0];
  } else if (j >= 98) {
    resfact = c_mcd_res[97];
  } else {
    pos -= j;
    resfact = c_mcd_res[j - 1] * (1. - pos) + c_mcd_res[j] * pos;
  }
  double gaufact = 1.;
  for (int k = 0; k < 3; k++) {
    const double z = (loget - c_mcd_gc[k]) / c_mcd_gw[k];
    gaufact += c_mcd_gn[k] * exp(-z * z / 2.);
  }
  return pow(et / .001, -.66666666666666663) * 193.21556 * (pow(et, 1.663753) * .52876731 + 1.) * exp(-et) *
         gaufact * (resfact + 1.);
}

// the scalars every thread of a solve derives the same way
struct NthGrid {
  double tautom, deltal, xmin;
  int jmax, jmaxth, ne, jnr, jrel;
};

__device__ inline NthGrid nth_grid(double tempbb, double theta, double gamma) {
#pragma clang fp contract(off)
  NthGrid q;
  const double delta = .02;
  const double gh = gamma + .5;
  q.tautom = sqrt(3. / (theta * (gh * gh - 2.25)) + 2.25) - 1.5;
  q.deltal = delta * log(10.);
  q.xmin = tempbb * 1e-4;
  const double xmax = theta * 40.;
  q.jmax = min(899, (int)(nth_lg10(xmax / q.xmin) / delta) + 1);
  q.jmaxth = min(900, (int)(nth_lg10(tempbb * 50. / q.xmin) / delta));
  if (q.jmaxth > q.jmax) q.jmaxth = q.jmax;
  q.ne = q.jmaxth - 2;
  q.jnr = min((int)(nth_lg10(.1 / q.xmin) / delta + 1), q.jmax - 1);
  q.jrel = min((int)(nth_lg10(1. / q.xmin) / delta + 1), q.jmax);
  return q;
}

}  // namespace

// What every solve shares: the seed temperature is the same for all of them
// (NTH_KTBB), so the photon grid and the factors that depend on it alone are
// laid out once per device (k_nth_grid), NTH_N doubles each behind the
// NTH_N + 1 energies.
constexpr double NTH_KTBB = 0.05;  // keV (src/relutility.c:625-632)
struct NthGridTab {
  const double *x;    // photon energies x_j = 1e-4 T_bb 10^(0.02 j), m_e c^2
  const double *w1;   // sqrt(x_j x_{j+1})
  const double *c2;   // Cooper's coefficient there (:544-566)
  const double *x3;   // x_j^3
  const double *rel;  // Klein-Nishina ratio of the escape probability (:598-626)
  const double *dph;  // the disc seed (:570-592)
};
__host__ __device__ inline NthGridTab nth_grid_tab(const double *t) {
  const double *f = t + NTH_N + 1;
  return NthGridTab{t, f, f + NTH_N, f + 2 * NTH_N, f + 3 * NTH_N, f + 4 * NTH_N};
}
constexpr size_t NTH_GRID_DOUBLES = (NTH_N + 1) + 5 * (size_t)NTH_N;

// The LDS of one Kompaneets solve (43 KB).
struct NthLds {
  double x[NTH_N + 1];
  double t1[NTH_N], t2[NTH_N], t3[NTH_N], d[NTH_N], bet[NTH_N];
};

__device__ __forceinline__ double nth_shfl_up(double v, int d) { return __shfl_up(v, d, 64); }
__device__ __forceinline__ double nth_shfl_down(double v, int d) { return __shfl_down(v, d, 64); }

// One Kompaneets solve by the nt threads of a workgroup (f_thdscompton__ with
// f_thermlc__, src/donthcomp.c:200-301, :468-648; 0-based arrays, the
// reference's 1-based bounds jnr / jrel kept as they are).  Leaves x[0..jmax] in
// L.x and E F_E in L.t1[0..NTH_N) (0 from jmax - 1 on); returns jmax.  Begins
// and ends with a barrier, so L may hold other data before the call.
//
// The interior rows j = 1 .. jmax-2 of the system read
//   -t2_{j+1} u_{j+1} + (t1_j + t2_j + t3_j) u_j - t1_{j-1} u_{j-1} = d_j
// with t1, t2, t3 > 0 (diffusion up and down the grid, escape; the first row's
// t2 goes with the boundary u_0 = (t2_1 / t1_0) u_1, the last u is 0): an
// M-matrix whose columns sum to t3.  Eliminating downwards, the pivot is
// b_j = t1_j + t3_j + t2_j s_{j-1} with s_j = (t3_j + t2_j s_{j-1}) / b_j, a
// quotient of linear forms with positive coefficients, and the two sweeps are
// linear recurrences with positive coefficients: all three are taken as scans
// by the first wavefront, a run of consecutive rows per lane and six shuffle
// steps between the lanes.  Nothing is subtracted, so the result is closer to
// the system's solution than elimination row by row: against extended
// precision over kTe 0.5-400 keV and Gamma 1.1-3.6 the largest error of a point
// is 3.2e-14 (4.1e-14 row by row).
// Bound: latency.  One thread's 3 x 400 dependent steps, two of them divisions,
// and the grid's powers made a solve 135 us; the scans and the shared grid make
// it 22 us (704 solves: 274 and 28 us).
__device__ inline int nth_solve(NthLds &L, const NthGridTab &G, double kte, double gam, int tid, int nt) {
#pragma clang fp contract(off)
  const double tempbb = NTH_KTBB / 511., theta = kte / 511.;
  const NthGrid q = nth_grid(tempbb, theta, gam);
  const int jmax = q.jmax;
  const double tautom = q.tautom, deltal = q.deltal, c20 = tautom / deltal;
  __syncthreads();
  const int n = max(0, jmax - 2);  // interior rows
  if (n > 0) {
    const double xnr = G.x[q.jnr - 1], xr = G.x[q.jrel - 1];
    for (int j = tid; j <= jmax; j += nt) L.x[j] = G.x[j];
    for (int j = tid; j < jmax; j += nt) {
      const int j1 = j + 1;  // the reference's 1-based index
      const double w = G.x[j];
      const double taukn = tautom * G.rel[j];
      double bet;  // the escape probability (:598-626)
      if (j1 <= q.jnr - 1) {
        bet = 1 / tautom / (taukn / 3 + 1);
      } else if (j1 <= q.jrel) {
        const double flz = 1 - (w - xnr) / (xr - xnr);
        bet = 1 / tautom / (taukn / 3 * flz + 1);
      } else {
        bet = 1 / tautom;
      }
      const double tb = theta / deltal / G.w1[j];
      L.t1[j] = c20 * G.c2[j] * (tb - .5);
      if (j + 1 < NTH_N) L.t2[j + 1] = c20 * G.c2[j] * (tb + .5);
      L.t3[j] = G.x3[j] * (tautom * bet);
      L.bet[j] = bet;
      L.d[j] = w * ((j <= q.ne && q.ne >= 1) ? G.dph[j] : 0.0);
    }
  }
  __syncthreads();
  if (tid < 64 && n > 0) {
    const int m = (n + 63) / 64, lane = tid;
    const int lo = 1 + lane * m, hi = min(lo + m, jmax - 1);  // this lane's rows [lo, hi)
    // pivots: s -> (A s + B) / (C s + D) over the lane's rows, then over the lanes
    double A = 1., B = 0., C = 0., D = 1.;
    for (int j = lo; j < hi; j++) {
      const double t1 = L.t1[j], t2 = L.t2[j], t3 = L.t3[j];
      const double r = 1. / (t1 + t2 + t3);  // (a common factor: entries of order one)
      const double p = t2 * r, qq = t3 * r, e = (t1 + t3) * r;
      const double a0 = p * A + qq * C, b0 = p * B + qq * D;
      C = p * A + e * C;
      D = p * B + e * D;
      A = a0;
      B = b0;
    }
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
      const double a = nth_shfl_up(A, s), bb = nth_shfl_up(B, s), c = nth_shfl_up(C, s), e = nth_shfl_up(D, s);
      if (lane >= s) {
        const double a0 = A * a + B * c, b0 = A * bb + B * e, c0 = C * a + D * c, d0 = C * bb + D * e;
        const double mx = fmax(fmax(fabs(a0), fabs(b0)), fmax(fabs(c0), fabs(d0)));
        const int k = (mx > 0. && mx < INFINITY) ? -ilogb(mx) : 0;  // (only ratios matter)
        A = ldexp(a0, k);
        B = ldexp(b0, k);
        C = ldexp(c0, k);
        D = ldexp(d0, k);
      }
    }
    double sg = nth_shfl_up(B, 1) / nth_shfl_up(D, 1);
    if (lane == 0) sg = 0.;
    // the lane's pivots (into t3) and its part of the downward sweep
    // y_j = (d_j + t1_{j-1} y_{j-1}) / b_j
    double al = 1., be = 0.;
    for (int j = lo; j < hi; j++) {
      const double s = L.t3[j] + L.t2[j] * sg;
      const double bp = L.t1[j] + s;
      sg = s / bp;
      L.t3[j] = bp;
      const double k = (j > 1 ? L.t1[j - 1] : 0.) / bp;
      al = k * al;
      be = k * be + L.d[j] / bp;
    }
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
      const double a = nth_shfl_up(al, s), bb = nth_shfl_up(be, s);
      if (lane >= s) {
        be = al * bb + be;
        al = al * a;
      }
    }
    double v = nth_shfl_up(be, 1);
    if (lane == 0) v = 0.;
    for (int j = lo; j < hi; j++) {
      v = (L.d[j] + (j > 1 ? L.t1[j - 1] : 0.) * v) / L.t3[j];
      L.d[j] = v;
    }
    // the upward sweep u_j = y_j + (t2_{j+1} / b_j) u_{j+1}
    al = 1.;
    be = 0.;
    for (int j = hi - 1; j >= lo; j--) {
      const double k = (j < jmax - 2 ? L.t2[j + 1] : 0.) / L.t3[j];
      al = k * al;
      be = k * be + L.d[j];
    }
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
      const double a = nth_shfl_down(al, s), bb = nth_shfl_down(be, s);
      if (lane + s < 64) {
        be = al * bb + be;
        al = al * a;
      }
    }
    v = nth_shfl_down(be, 1);
    if (lane == 63) v = 0.;
    for (int j = hi - 1; j >= lo; j--) {
      v = L.d[j] + (j < jmax - 2 ? L.t2[j + 1] : 0.) / L.t3[j] * v;
      L.t3[j] = v;
    }
    if (lane == 0) L.t3[0] = L.t2[1] / L.t1[0] * L.t3[1];
  }
  __syncthreads();
  // escaping photons and E F_E (:297-300, :630-636), into t1
  for (int j = tid; j < NTH_N; j += nt) {
    double v = 0.0;
    if (j < jmax - 1) {
      const double dphesc = L.x[j] * L.x[j] * L.t3[j] * L.bet[j] * tautom;
      v = dphesc * (L.x[j] * L.x[j]);
    }
    L.t1[j] = v;
  }
  __syncthreads();
  return jmax;
}

// The photon energies are log-spaced from the same x_0 in every solve, so a
// bracket comes from one logarithm, corrected to the exact comparison (at most
// a step or two; the searches it replaces took 10 dependent reads).
__device__ __forceinline__ int nth_guess(double v511) {  // about (j with x_j 511 = v511), at least -1
  constexpr float lg0 = -17.6096405f;   // log2(511 x_0) = log2(1e-4 NTH_KTBB)
  constexpr float scale = 15.0514998f;  // 1 / (0.02 log2(10))
  return (int)fminf(fmaxf((__log2f((float)v511) - lg0) * scale, -1.0f), (float)NTH_N);
}

// E F_E of a solution at x (f_spp__, src/donthcomp.c:651-681): the first
// index ih >= 1 with x_ih >= x (at most nth - 1), linear in [x_{ih-1}, x_ih].
__device__ inline double nthcomp_spp(const double *x, const double *spt, int nth, double xx) {
#pragma clang fp contract(off)
  int ih = max(1, min(nth_guess(xx * 511.) + 1, nth - 1));
  while (ih > 1 && !(xx > x[ih - 1])) ih--;
  while (ih < nth - 1 && xx > x[ih]) ih++;
  const int il = ih - 1;
  return spt[il] + (spt[ih] - spt[il]) * (xx - x[il]) / (x[ih] - x[il]);
}

// E F_E at the grid edge ear (keV) for redshift z (c_donthcomp, :757-774):
// the reference walks j up while x_{j-1} 511 < ear (z + 1); the bracket is
// the first such failure, j in [1, nth], else nth + 1.
__device__ inline double nthcomp_edge(const double *x, const double *spt, int nth, double ear, double z) {
#pragma clang fp contract(off)
  const double v = ear * (z + 1);
  int j = max(1, min(nth_guess(v) + 2, nth + 1));
  while (j > 1 && !(x[j - 2] * 511. < v)) j--;
  while (j <= nth && x[j - 1] * 511. < v) j++;
  if (j > nth) return 0.0;
  if (j == 1) return spt[0];
  const int jl = j - 1;
  return spt[jl - 1] + (ear / 511. * (z + 1) - x[jl - 1]) * (spt[jl] - spt[jl - 1]) / (x[jl] - x[jl - 1]);
}

// the normalisation of c_donthcomp (:747-756): E F_E(1 keV, source) = 1
__device__ inline double nthcomp_normfac(const double *x, const double *spt, int nth, double z) {
#pragma clang fp contract(off)
  const double xn = (z + 1) / 511.;
  return 1 / nthcomp_spp(x, spt, nth, 1 / (1 / xn));
}

// photons in the bin [e0, e1] from the edge values p0, p1 (E F_E) with the
// normalisation normfac
__device__ inline double nthcomp_bin(double e0, double e1, double p0, double p1, double normfac) {
#pragma clang fp contract(off)
  return (p1 / (e1 * e1) + p0 / (e0 * e0)) * .5 * (e1 - e0) * normfac;
}

}  // namespace rx
