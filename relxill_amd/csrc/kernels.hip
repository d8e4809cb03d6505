// kernels.hip -- CDNA4 (gfx950) kernels of the relativistic smearing path.
//
//   k_begin      clears the run's counters, fetches a call's request block
//   k_setup      one workgroup per request: (a, mu0) bilinear table
//                interpolation (interpol_relTable, src/Relprofile.cpp:141-303),
//                fine radial grid, emissivity (src/Rellp.cpp:518-564), energy
//                windows and the request's work items (radius chunk x bin
//                segment)
//   k_dist       one wavefront per (request, 64 radii): the emission-angle
//                distribution (src/Relprofile.cpp:908-938)
//   k_integrate  persistent 64-lane wavefronts over the work items: lane =
//                fine radius, loop over the segment's bins, fixed-order wave
//                sum per bin (calc_relline_profile, src/Relprofile.cpp:857-900)
//   k_fixup      FP64 re-check of FP32 Romberg stop tests in the guard band
//   k_finalize   one workgroup per request: photons per bin and
//                renormalisation (src/Relprofile.cpp:749-796)
//   k_conv       one workgroup per convolution request: rebin onto the
//                convolution grid, real FFT convolution held in LDS with the
//                1 keV rotation and E/dE weighting, band normalisation, rebin
//                back and zeroing outside 0.01-1000 keV
//                (src/Relbase.cpp:93-289)
//   k_deliver    counters, statuses and a call's outputs to the host
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "rx_engine.h"
#include "rx_math.h"
#include "rx_nthcomp.h"

namespace rx {

namespace {

constexpr int FINAL_THREADS = 256;
constexpr int CONV_THREADS = 256;      // smallest convolution workgroup
constexpr int XILL_THREADS = 256;
constexpr int XILL_BINS = 4;    // table bins per k_xill thread, one-zone requests
constexpr int XILL_BINS_Z = 2;  // the same for requests of LP_ZONES zones (ten accumulators per bin)
constexpr int PRIM_THREADS = 256;
constexpr int CONV_THREADS_MAX = 1024;  // n/8 threads: 512 for 4096 bins, 1024 for 8192

// spec_cutoffpl (src/Xillspec.cpp:215-241): photons of the cut-off power law
// exp(1/Ecut) E^-Gamma exp(-E/Ecut) dE in [e0, e1] at E = (e0 + e1) / 2, as
// one exponential of ln_en = ln E (precomputed per grid bin): it differs from
// the product of the three factors by a few ulp of the exponent
__device__ inline double cutoffpl_bin(double e0, double e1, double ln_en, double ecut, double gam) {
  const double en = 0.5 * (e0 + e1);
  return exp(1.0 / ecut - gam * ln_en - en / ecut) * (e1 - e0);
}

// spec_blackbody (src/Xillspec.cpp:255-268): photons of E^2 / (kT^4 (exp(E/kT) - 1))
// dE in [e0, e1] at E = (e0 + e1) / 2
__device__ inline double bbody_bin(double e0, double e1, double kt) {
  const double en = 0.5 * (e0 + e1);
  return en * en / (pow(kt, 4) * (exp(en / kt) - 1)) * (e1 - e0);
}

// 1e15 / (4 pi): the xillver tables' incident flux normalisation (src/Xillspec.cpp:203)
constexpr double NORM_XILLVER_TABLE = 1e15 / 4.0 / 3.14159265358979323846;

// A xillver table value as the reference holds it after renorm_xill_spec
// (src/xilltable.c:478-486): the resident rows are divided by 10^logXi; rows
// of a table without a density axis are also divided by dens_div =
// 10^(logN - 15) (rounded to float, as the reference's float array), unless
// logN is 15 (dens_div 0).  The quotient by the request's one divisor takes its
// correctly rounded reciprocal and one correction step (the remainder in one
// fma), which rounds as the division does, in 3 operations instead of about 10.
struct DensDiv {
  double d, r;
};
__device__ __forceinline__ DensDiv dens_of(double dens_div) {
  return DensDiv{dens_div, dens_div != 0.0 ? 1.0 / dens_div : 0.0};
}
__device__ __forceinline__ double xval(float v, const DensDiv &dd) {
  if (dd.d == 0.0) return (double)v;
  const double q = (double)v * dd.r;
  return (double)(float)fma(fma(-dd.d, q, (double)v), dd.r, q);
}

// This thread's part of calcNormWrtXillverTableSpec's sum (src/Xillspec.cpp:179-205)
// for the cut-off power law on the 500-bin 0.1-1000 keV grid ce.
__device__ inline double xill_norm_part(const DevConvGrid &cg, double ecut, double gam, int tid, int nt) {
  double sp = 0.0;
  for (int k = tid; k < N_ENER_COARSE; k += nt) {
    const double e0 = cg.coarse[k], e1 = cg.coarse[k + 1];
    if (e0 >= 0.1 && e0 <= 1000.0)
      sp += cutoffpl_bin(e0, e1, cg.coarse_ln[k], ecut, gam) * 0.5 * (e0 + e1) * 1e20 * 1.602177e-09;
  }
  return sp;
}

// The same sum for the blackbody of kT_bb kt.
__device__ inline double bbody_norm_part(const DevConvGrid &cg, double kt, int tid, int nt) {
  double sp = 0.0;
  for (int k = tid; k < N_ENER_COARSE; k += nt) {
    const double e0 = cg.coarse[k], e1 = cg.coarse[k + 1];
    if (e0 >= 0.1 && e0 <= 1000.0) sp += bbody_bin(e0, e1, kt) * 0.5 * (e0 + e1) * 1e20 * 1.602177e-09;
  }
  return sp;
}

// bsearch_asc by a whole wavefront: the same bracket of an ascending array from
// one load a lane (binary search: a dependent load a step, 0.5 us each)
template <class T, class V>
__device__ inline int wave_bracket(const T *arr, int n, V val, int lane) {
  int cnt = 0;  // values that are not above val
  for (int k = 0; k < n; k += 64) cnt += __popcll(__ballot(k + lane < n && !(arr[min(k + lane, n - 1)] > val)));
  return min(max(cnt - 1, 0), n - 2);
}

// get_ipol_factor (src/relutility.c:419-423): float quotient
__device__ inline double ipol_fac(float value, const float *arr, int ind) {
  return (double)((value - arr[ind]) / (arr[ind + 1] - arr[ind]));
}

struct LpFine {
  double emis, del_emit, del_inc;
  int err;
};

// rebin_emisprofile_on_radial_grid for one fine radius (src/Rellp.cpp:120-175):
// the table walk reduces to kk = clamp(#{jet_rad <= r} - 1, 0, n-2).
__device__ inline LpFine lp_on_fine(double re, const double *jr, const double *je,
                                    const double *jd, const double *ji, int ntr) {
  LpFine o;
  o.err = 0;
  int lo = 0, hi = ntr;
  while (lo < hi) {
    int mid = (lo + hi) >> 1;
    if (jr[mid] <= re) lo = mid + 1; else hi = mid;
  }
  int kk = lo - 1;
  if (kk < 0) kk = 0;
  if (kk >= ntr - 1) {
    if (!(re - 1000.0 <= 1e-6)) o.err = 22;
    kk = ntr - 2;
  }
  double inter_r;
  if (jd[kk] / PI * 180.0 <= 75.0) {  // get_ipol_factor_radius, src/relutility.c:407-417
    inter_r = (re - jr[kk]) / (jr[kk + 1] - jr[kk]);
  } else {
    inter_r = (log(re) - log(jr[kk])) / (log(jr[kk + 1]) - log(jr[kk]));
  }
  o.emis = exp(inter_r * log(je[kk + 1]) + (1.0 - inter_r) * log(je[kk]));
  o.del_emit = lerp1(inter_r, jd[kk], jd[kk + 1]);
  o.del_inc = lerp1(inter_r, ji[kk], ji[kk + 1]);
  return o;
}

// g = E/E_i for the lamp post (src/Relphysics.cpp:163-207)
__device__ inline double gi_potential_lp(double r, double a, double h, double bet, double del) {
  double ut_d = ((r * sqrt(r) + a) / (sqrt(r) * sqrt(r * r - 3 * r + 2 * a * sqrt(r))));
  double ut_h = sqrt((h * h + a * a) / (h * h - 2 * h + a * a));
  double gi = ut_d / ut_h;
  if (fabs(bet) < 1e-6) return gi;
  double gam = 1.0 / sqrt(1.0 - bet * bet);
  double sgn = (del > PI / 2) ? -1.0 : 1.0;
  double delta_eq = h * h - 2 * h + a * a;
  double sd = sin(del);
  double hh = h * h + a * a;
  double q2 = (sd * sd) * (hh * hh / delta_eq) - a * a;
  double beta_fac = sqrt(hh * hh - delta_eq * (q2 + a * a));
  beta_fac = gam * (1.0 + sgn * beta_fac / hh * bet);
  return gi / beta_fac;
}

// lamp-post emissivity of a fine radius with the flux boost (src/Rellp.cpp:249-253,
// src/Relphysics.cpp:301-311); *err is set where the table does not reach
__device__ __forceinline__ double lp_emis_at(const ReqParams &rq, double re, const double *jr, const double *je,
                                    const double *jd, const double *ji, int ntr, int *err) {
  LpFine f = lp_on_fine(re, jr, je, jd, ji, ntr);
  if (f.err) *err = f.err;
  double boost = pow(gi_potential_lp(re, rq.a, rq.height, rq.beta, f.del_emit), rq.gamma);
  if (rq.beta > 1e-6) {
    const double d = sqrt(1.0 - rq.beta * rq.beta) / (1.0 + rq.beta * cos(f.del_emit));
    boost *= d * d;
  }
  return f.emis * boost;
}

__device__ inline double relat_abberation(double del, double beta) {
  return acos((cos(del) - beta) / (1 - beta * cos(del)));
}

// corrected_gshift_fluxboost_factor (src/Relreturn_Corona.cpp:39-83): the flux
// boost of the xillver reflection under the energy shift g, from its boost
// ratio c to a power law at g = 1.5 (a parabola through 0 for c < 1, a line
// otherwise; at most 1 below g = 1, never negative)
__device__ inline double gshift_boost(double c, double g, double gamma) {
  const double g0 = 2. / 3;
  double corr;
  if (c < 1) {
    const double a = (c / g0 - 1) / (g0 - 1);
    const double b = 1 - a;
    corr = (g >= 1) ? 1. / g * (1. / g * a + b) : g * (g * a + b);
  } else {
    const double alin = (c - 1) / (g0 - 1);
    const double blin = 1 - alin;
    corr = (g >= 1) ? (1. / g * alin + blin) : (g * alin + blin);
  }
  double boost = pow(g, gamma) * corr;
  if (g < 1 && boost > 1) boost = 1;
  if (boost < 0) boost = 0;
  return boost;
}

// interpol_lptable (src/Rellp.cpp:219-247) of one request into the block's
// LDS rows: radius (lerped in spin), intensity, emission and incidence angle
// ((1 - f_a) lerp_h(spin lo) + f_a lerp_h(spin hi), float factors) at the
// table's n_r radii.  Called by every thread of the block (two barriers).
__device__ inline void lp_rows(const DevLpTable &L, const ReqParams &rq, double *jr, double *je, double *jd,
                               double *ji, int tid, int nt) {
  __shared__ int s_i[3];
  __shared__ double s_f[3];
  if (tid < 64) {
    // the searches are float (src/relutility.c:419-423)
    const float a = (float)rq.a, h = (float)rq.height;
    const int lia = wave_bracket(L.a, L.n_a, a, tid);
    const float *hl = L.h + (size_t)lia * L.n_h, *hu = hl + L.n_h;
    const int h0 = wave_bracket(hl, L.n_h, h, tid), h1 = wave_bracket(hu, L.n_h, h, tid);
    const double lfa = ipol_fac(a, L.a, lia), fh0 = ipol_fac(h, hl, h0), fh1 = ipol_fac(h, hu, h1);
    s_i[0] = lia;
    s_i[1] = h0;
    s_i[2] = h1;
    s_f[0] = lfa;
    s_f[1] = fh0;
    s_f[2] = fh1;
  }
  __syncthreads();
  const int ntr = L.n_r;
  const int lia = s_i[0], h0 = s_i[1], h1 = s_i[2];
  const double lfa = s_f[0], fh0 = s_f[1], fh1 = s_f[2];
  for (int ii = tid; ii < ntr; ii += nt) {
    jr[ii] = lerp1(lfa, (double)L.rad[(size_t)lia * ntr + ii], (double)L.rad[(size_t)(lia + 1) * ntr + ii]);
    const size_t l0 = ((size_t)lia * L.n_h + h0) * ntr + ii;
    const size_t u0 = ((size_t)lia * L.n_h + h0 + 1) * ntr + ii;
    const size_t l1 = ((size_t)(lia + 1) * L.n_h + h1) * ntr + ii;
    const size_t u1 = ((size_t)(lia + 1) * L.n_h + h1 + 1) * ntr + ii;
    je[ii] = (1.0 - lfa) * lerp1(fh0, L.intens[l0], L.intens[u0]) + (lfa)*lerp1(fh1, L.intens[l1], L.intens[u1]);
    jd[ii] = (1.0 - lfa) * lerp1(fh0, L.del[l0], L.del[u0]) + (lfa)*lerp1(fh1, L.del[l1], L.del[u1]);
    ji[ii] = (1.0 - lfa) * lerp1(fh0, L.del_inc[l0], L.del_inc[u0]) + (lfa)*lerp1(fh1, L.del_inc[l1], L.del_inc[u1]);
  }
  __syncthreads();
}

// The fine radii around r: the largest i in 0 .. nr - 2 with re(i) > r, or 0
// (the radii descend; r1, r2: fine_radius_r1 of rout and rin).  The grid's own
// formula gives the index to the rounding; the comparisons decide.
__device__ inline int fine_above(double r1, double r2, double r, int nr) {
  int i = (int)((1.0 / sqrt(r) - r1) / (r2 - r1) * (nr - 1));
  i = min(max(i, 0), nr - 2);
  while (i > 0 && !(fine_radius_at(r1, r2, i, nr) > r)) i--;
  while (i < nr - 2 && fine_radius_at(r1, r2, i + 1, nr) > r) i++;
  return i;
}

// One radial zone of a relxill request (IonGradient, src/IonGradient.cpp:
// 182-209, :421-430): its centre, for the lamp post the emission angle there
// (inv_rebin_mean of the fine grid's angles, src/relutility.c:636-663), the
// source -> disk energy shift and the Ecut the zone sees with its xillver
// bracket (float factor, clamps, ensure_ecut_within_boundarys,
// src/xilltable.c:1054-1125).  *ect receives that Ecut (lamp post).
__device__ inline ZoneRec zone_record(const DevXillTable &xt, const ReqParams &rq, int z, bool lp, const double *jr,
                                      const double *je, const double *jd, const double *ji, int ntr, int nr,
                                      double *ect) {
  const double *zg = rq.zgrid;
  ZoneRec o;
  o.rmean = 0.5 * (zg[z] + zg[z + 1]);
  o.del_emit = 0.0;
  o.shift = 1.0;
  o.ncf = 1.0;
  o.ect_ind = xt.ect_dim >= 0 ? rq.xind[xt.ect_dim] : 0;
  o.ect_fac = xt.ect_dim >= 0 ? rq.xfac[xt.ect_dim] : 0.0;
  o.lxi_ind = xt.lxi_dim >= 0 ? rq.xind[xt.lxi_dim] : 0;
  o.lxi_fac = xt.lxi_dim >= 0 ? rq.xfac[xt.lxi_dim] : 0.0;
  *ect = rq.xect_src;
  if (rq.ion_grad == 1 && xt.lxi_dim >= 0) {
    // the power-law gradient (calc_ion_grad_pl, src/IonGradient.cpp:174-182)
    // from the input logXi in the zones' mean radius, kept within 0-4.7
    // (adjust_parameter_to_be_within_xillver_bounds, :36-44, :388), and its
    // bracket on the table's logXi axis as the request's parameters get
    // theirs (float value, clamped into the table, float factor)
    const double rm0 = 0.5 * (zg[0] + zg[1]);
    double lxi = exp(rq.xlxi0) * pow(o.rmean / rm0, -1.0 * rq.ion_index);
    lxi = log(lxi);
    if (lxi < 0.0) lxi = 0.0;
    else if (lxi > 4.7) lxi = 4.7;
    const float *vals = xt.lxi_vals;
    const int n = xt.n_lxi;
    float v = (float)lxi;
    int ind = bsearch_asc(vals, n, v);
    if (ind < 0) ind = 0;
    else if (ind > n - 2) ind = n - 2;
    if (v < vals[0]) v = vals[0];
    else if (v > vals[n - 1]) v = vals[n - 1];
    const float num = v - vals[ind];
    const float den = vals[ind + 1] - vals[ind];
    o.lxi_ind = ind;
    o.lxi_fac = (float)(num / den);
  }
  if (lp) {
    const double q1 = fine_radius_r1(rq.rout), q2 = fine_radius_r1(rq.rin);
    const int lo = fine_above(q1, q2, o.rmean, nr);
    const double r0 = fine_radius_at(q1, q2, lo, nr), r1 = fine_radius_at(q1, q2, lo + 1, nr);
    const LpFine f0 = lp_on_fine(r0, jr, je, jd, ji, ntr);
    const LpFine f1 = lp_on_fine(r1, jr, je, jd, ji, ntr);
    o.del_emit = lerp1((o.rmean - r1) / (r0 - r1), f1.del_emit, f0.del_emit);
    o.shift = gi_potential_lp(o.rmean, rq.a, rq.height, rq.beta, o.del_emit);
    *ect = rq.xect_src * o.shift;
    if (xt.ect_dim >= 0) {
      const float *vals = xt.ect_vals;
      const int n = xt.n_ect;
      float v = (float)*ect;
      int ind = bsearch_asc(vals, n, v);
      if (ind < 0) ind = 0;
      else if (ind > n - 2) ind = n - 2;
      if (v < vals[0]) v = vals[0];
      else if (v > vals[n - 1]) v = vals[n - 1];
      const float num = v - vals[ind];
      const float den = vals[ind + 1] - vals[ind];
      double fac = (float)(num / den);
      if (*ect <= xt.q_vals[0]) fac = 0.0;
      if (*ect >= xt.q_vals[xt.n_q - 1]) fac = 1.0;
      o.ect_ind = ind;
      o.ect_fac = fac;
    }
  }
  return o;
}

// Where a request's profile accumulates: the caller output for line models,
// the convolution-grid profile for convolution models.
__device__ inline double *profile_acc(const BatchDev &b, const ReqParams &rq) {
  return (rq.prof_off >= 0) ? b.prof + rq.prof_off : b.out + rq.flux_off;
}

// Index guess for an ascending grid that is close to log-spaced (every grid
// here is): e0[k] ~ e0[0] exp(k dlog).
struct GridGuess {
  float lg0, scale;  // log2(e0[0]), n0 / log2(e0[n0] / e0[0])
  double first, last;
};

__device__ __forceinline__ GridGuess grid_guess(const double *e0, int n0) {
  GridGuess g;
  g.first = e0[0];
  g.last = e0[n0];
  g.lg0 = __log2f((float)g.first);
  g.scale = (float)n0 / (__log2f((float)g.last) - g.lg0);
  return g;
}

// cnt(x) = #{k in [0, n0] : e0(k) <= x}: the log-spaced guess, exact
// correction by at most two steps, else bisection (any ascending grid).
template <class E>
__device__ __forceinline__ int count_le(E e0, int n0, double x, const GridGuess &g) {
  if (!(x >= g.first)) return 0;
  if (x >= g.last) return n0 + 1;
  int k = (int)((__log2f((float)x) - g.lg0) * g.scale);
  k = min(max(k, 0), n0 - 1);
#pragma unroll
  for (int it = 0; it < 3; it++) {
    if (e0(k) > x) {
      if (k == 0) return 0;  // cannot happen: x >= e0[0]
      k--;
    } else if (e0(k + 1) <= x) {
      k++;
    } else {
      return k + 1;
    }
  }
  int lo = 0, hi = n0 + 1;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (e0(mid) <= x) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// Guessed bracket of x (the first guess of count_le), clamped to [0, n0 - 1].
__device__ __forceinline__ int guess_index(double x, const GridGuess &g, int n0) {
  const int k = (int)((__log2f((float)x) - g.lg0) * g.scale);
  return min(max(k, 0), n0 - 1);
}

// count_le when the edges a = e0(k), b = e0(k + 1) around the guess k are
// already loaded: the exact search only when the guess misses.
template <class E>
__device__ __forceinline__ int count_le_at(E e0, int n0, double x, const GridGuess &g, int k, double a, double b) {
  if (!(x >= g.first)) return 0;
  if (x >= g.last) return n0 + 1;
  if (a <= x && x < b) return k + 1;
  return count_le(e0, n0, x, g);
}

template <int CTRL>
__device__ inline int dpp_int(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
}

template <int CTRL>
__device__ inline int dpp_i(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
}

template <int CTRL>
__device__ inline double dpp_d(double v) {
  const int lo = dpp_i<CTRL>(__double2loint(v));
  const int hi = dpp_i<CTRL>(__double2hiint(v));
  return __hiloint2double(hi, lo);
}

__device__ inline double readlane_d(double v, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                          __builtin_amdgcn_readlane(__double2loint(v), l));
}

// Sum over the 64 lanes in a fixed order (pairs, quads, half rows, rows, then
// the four rows); every lane must be active.
__device__ inline double wave_sum(double v) {
  v += dpp_d<0xB1>(v);   // quad_perm [1,0,3,2]
  v += dpp_d<0x4E>(v);   // quad_perm [2,3,0,1]
  v += dpp_d<0x141>(v);  // row_half_mirror
  v += dpp_d<0x140>(v);  // row_mirror
  return (readlane_d(v, 0) + readlane_d(v, 16)) + (readlane_d(v, 32) + readlane_d(v, 48));
}

// maximum over the 64 lanes; every lane must be active
__device__ inline double wave_max_d(double v) {
  v = fmax(v, dpp_d<0xB1>(v));
  v = fmax(v, dpp_d<0x4E>(v));
  v = fmax(v, dpp_d<0x141>(v));
  v = fmax(v, dpp_d<0x140>(v));
  return fmax(fmax(readlane_d(v, 0), readlane_d(v, 16)), fmax(readlane_d(v, 32), readlane_d(v, 48)));
}

// What one lane wrote to LDS is there for the other lanes of its wavefront behind
// this (the hardware keeps a wavefront's LDS operations in order; the fence keeps
// the compiler from moving them across).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// min / max over the 64 lanes (quad, half-row and row exchanges, then the rows);
// every lane must be active
__device__ inline int wave_min_i(int v) {
  v = min(v, dpp_int<0xB1>(v));
  v = min(v, dpp_int<0x4E>(v));
  v = min(v, dpp_int<0x141>(v));
  v = min(v, dpp_int<0x140>(v));
  return min(min(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
             min(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

__device__ inline int wave_max_i(int v) {
  v = max(v, dpp_int<0xB1>(v));
  v = max(v, dpp_int<0x4E>(v));
  v = max(v, dpp_int<0x141>(v));
  v = max(v, dpp_int<0x140>(v));
  return max(max(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
             max(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

// 1/x to within an ulp or two: hardware estimate and two Newton steps
// (cheaper than the IEEE division sequence; the rebin weights need ~1e-15).
__device__ __forceinline__ double rcp64(double x) {
  double r = __builtin_amdgcn_rcp(x);
  double e = fma(-x, r, 1.0);
  r = fma(r, e, r);
  e = fma(-x, r, 1.0);
  return fma(r, e, r);
}

// _rebin_spectrum (src/relutility.c:549-601), value of one output bin
// [elo_, ehi_] from the counts clo = cnt(elo_), chi = cnt(ehi_) of input
// edges at or below each end, cnt(x) = #{k : e0(k) <= x}: the reference's
// sequential search gives imin = max(clo-1, 0), imax = max(min(chi, n0)-1, 0);
// an overlap of zero width at the top edge gives 0.
template <class E, class F>
__device__ __forceinline__ double rebin_bin(double elo_, double ehi_, int clo, int chi, E e0, int n0, F f0) {
  const int imin = clo > 0 ? clo - 1 : 0;
  if (!((e0(0) <= ehi_) && (e0(n0) >= elo_)) || imin >= n0) return 0.0;
  int imax = chi < n0 ? chi : n0;
  if (imax > 0) imax--;
  double elo = elo_, ehi = ehi_;
  const double a0 = e0(imin), a1 = e0(imin + 1);
  if (elo < a0) elo = a0;
  const double b0 = e0(imax), b1 = e0(imax + 1);
  if (ehi > b1) ehi = b1;
  const double ra = rcp64(a1 - a0);
  if (imax == imin) return (ehi - elo) * ra * f0(imin);
  const double dmin = (a1 - elo) * ra;
  const double dmax = (ehi - b0) * rcp64(b1 - b0);
  double v = 0.0;
  v += f0(imin) * dmin + f0(imax) * dmax;
  for (int jj = imin + 1; jj <= imax - 1; jj++) v += f0(jj);
  return v;
}

// A fine radius' lerp factor between the node radii K+1 (lo) and K (hi) and
// its g window, lerped between the nodes' g_min and g_max (src/Relprofile.cpp:
// 249-300).  k_setup, k_integrate and k_fixup all take them from here (k_setup
// from its LDS copy of the node arrays, the others from the request's node
// arrays in global memory), so that the three agree bit for bit.
struct RadGeo {
  double ifac_r, gmin, gmax;
};
__device__ inline RadGeo rad_geo(const double *tre, const double *tgmin, const double *tgmax, double re, int K) {
#pragma clang fp contract(off)
  RadGeo o;
  o.ifac_r = (re - tre[K + 1]) / (tre[K] - tre[K + 1]);
  o.gmin = lerp1(o.ifac_r, tgmin[K + 1], tgmin[K]);
  o.gmax = lerp1(o.ifac_r, tgmax[K + 1], tgmax[K]);
  return o;
}

// block-wide deterministic sum (fixed tree order)
__device__ inline double block_sum(double v, double *red) {
  const int tid = threadIdx.x;
  red[tid] = v;
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if (tid < s) red[tid] += red[tid + s];
    __syncthreads();
  }
  double r = red[0];
  __syncthreads();
  return r;
}

}  // namespace

// ---------------------------------------------------------------------------
// setup
// ---------------------------------------------------------------------------
// NZ: the most zones of a request in the batch (LP_ZONES, or MAX_ZONES with
// an ionisation gradient), which sizes the zone arrays in LDS.  NT: threads.
// Bound: latency, of the table loads, of a fine radius' chain (a search over
// the node radii, the emissivity's pow, two bracket searches over the energy
// grid) and of the barriers between the phases; so what one thread did in turn
// (table and radius searches, the lamp post's reflection fraction, the list of
// windows) is done by a wavefront at once, and sums cross the wavefronts in one
// step.  Batches that leave the chip idle get workgroups of 512 threads, which
// take the 1000 radii in two rounds instead of four.  Measured before and after:
// relline call 24 -> 15 us, relline_lp call 43 -> 27 us, relxilllp call 62 -> 31
// us, 256 relline_lp requests 50 -> 33 us, 4096 relconv requests 176 -> 131 us.
template <int NZ, int NT>
__global__ __launch_bounds__(NT, NT == 256 ? 3 : 1) void k_setup(BatchDev b) {
  constexpr int NW = NT / 64;
  const int req = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const ReqParams &rq = b.req[req];
  const DevRelTable &T = b.rt;
  const int nr = b.nr_fine;
  const int n_r = T.n_r;
  if (rq.pre_status != 0) return;  // status already set by the host
  if (rq.model == MOD_XILLVER) {
    // the xillver models (LocalModel::xillver_model, src/LocalModel.cpp:
    // 104-128) have no relativistic part: the angle distribution carries the
    // inclination's bracket, so that k_xill's sum over angles is the
    // interpolation in the inclination (interp_5d_tab, src/xilltable.c:878-995);
    // k_primary rebins and adds the primary
    double *d = b.dist + rq.dist_off;
    for (int a = tid; a < rq.n_incl; a += NT)
      d[a] = (a == rq.xinc_ind) ? 1.0 - rq.xinc_fac : ((a == rq.xinc_ind + 1) ? rq.xinc_fac : 0.0);
    return;
  }
  __shared__ double s_tre[MAX_NR_TAB], s_tgmin[MAX_NR_TAB], s_tgmax[MAX_NR_TAB];
  __shared__ double s_jr[MAX_LP_R], s_je[MAX_LP_R], s_jd[MAX_LP_R], s_ji[MAX_LP_R];
  __shared__ double s_rr_rad[MAX_RR], s_rr_ret[MAX_RR];
  __shared__ double s_sum[NW], s_max[NW];
  // statuses of the three stages, each tested behind a barrier of its own and not
  // written after it (a wavefront may still be at the test of the one before)
  __shared__ int s_st, s_st_edge, s_st_rad, s_st_refl;
  __shared__ int s_ia, s_im, s_rmin;
  __shared__ double s_fa, s_fm;
  constexpr int MAX_RC = MAX_NR_FINE / RAD_CHUNK;
  // energy window of each (radius chunk, zone): bins [s_ulo, s_uhi]
  __shared__ int s_ulo[MAX_RC * NZ], s_uhi[MAX_RC * NZ];
  __shared__ int s_pref[MAX_RC * NZ], s_prefs[MAX_RC * NZ];
  __shared__ int s_base, s_bases, s_jlo, s_jhi;
  const int n_rc = (nr + RAD_CHUNK - 1) / RAD_CHUNK;
  const int nz = rq.n_zones;
  const double *zg = rq.zgrid;
  const bool lp = (rq.emis_type == EMIS_LP);
  const DevLpTable &L = b.lp;
  const int ntr = L.n_r;

  // the (a, mu0) bracket, one wavefront; meanwhile the others begin with the grid
  if (wave == 0) {
    const float a = (float)rq.a, mu0 = (float)cos(rq.incl);
    const int ia = wave_bracket(T.a, T.n_a, a, lane), im = wave_bracket(T.mu0, T.n_mu0, mu0, lane);
    const float fa = (a - T.a[ia]) / (T.a[ia + 1] - T.a[ia]);
    const float fm = (mu0 - T.mu0[im]) / (T.mu0[im + 1] - T.mu0[im]);
    int st = 0;
    if (!(rq.rout > rq.rin) || !(rq.rin >= rq.rms)) st = 10;
    if (!(fm >= 0 && fm <= 1 && fa >= 0 && fa <= 1)) st = 11;
    if (lane == 0) {
      s_st = st;
      s_st_rad = s_st_refl = 0;
      s_ia = ia;
      s_im = im;
      s_fa = fa;
      s_fm = fm;
    }
  }
  for (int c = tid; c < n_rc * NZ; c += NT) {
    s_ulo[c] = 0x7fffffff;
    s_uhi[c] = -1;
  }
  if (rq.model == MOD_RELXILL || rq.model == MOD_RELXILLLP) {
    // the zones' convolutions add into the output (k_conv)
    double *out = b.out + rq.flux_off;
    for (int j = tid; j < rq.n_in; j += NT) out[j] = 0.0;
  }
  if (rq.n_incl > 0) {  // k_dist adds into the angle distribution
    const int nd = rq.n_incl * nz;  // [zone][angle bin]
    for (int k = tid; k < nd; k += NT) b.dist[rq.dist_off + k] = 0.0;
  }
  // profile grid: caller grid shifted to line-energy units (XspecSpectrum.h:61-76)
  const double *E;
  if (rq.pgrid_off >= 0) {
    double *pg = b.pgrid + rq.pgrid_off;
    const double *ein = b.ener_in + rq.ener_off;
    for (int k = tid; k <= rq.n_in; k += NT) {
      double e = ein[k];
      if (rq.z > 0) e *= (1 + rq.z);
      pg[k] = e / rq.lineE;
    }
    E = pg;
  } else {
    E = b.cg.ener;
  }
  __syncthreads();
  if (s_st) {
    if (tid == 0) b.status[req] = s_st;
    return;
  }
  const int ia = s_ia, im = s_im;
  const double fa = s_fa, fm = s_fm;
  const size_t n00 = (size_t)ia * T.n_mu0 + im, n10 = (size_t)(ia + 1) * T.n_mu0 + im;
  const size_t n01 = (size_t)ia * T.n_mu0 + im + 1, n11 = (size_t)(ia + 1) * T.n_mu0 + im + 1;
  // node radii: lerp in a only (src/Relprofile.cpp:190-193); node values:
  // bilinear in (a, mu0) (interpol_a_mu0, :39-80)
  for (int ir = tid; ir < n_r; ir += NT) {
    s_tre[ir] = lerp1(fa, (double)T.r[n00 * n_r + ir], (double)T.r[n10 * n_r + ir]);
    s_tgmin[ir] = lerp2f(fa, fm, T.gmin[n00 * n_r + ir], T.gmin[n10 * n_r + ir],
                         T.gmin[n01 * n_r + ir], T.gmin[n11 * n_r + ir]);
    s_tgmax[ir] = lerp2f(fa, fm, T.gmax[n00 * n_r + ir], T.gmax[n10 * n_r + ir],
                         T.gmax[n01 * n_r + ir], T.gmax[n11 * n_r + ir]);
  }
  // lamp-post table node (interpol_lptable, src/Rellp.cpp:219-247)
  if (lp) lp_rows(L, rq, s_jr, s_je, s_jd, s_ji, tid, NT);
  // returning radiation: the zones' centres and returning emissivity (k_rrad)
  const bool rrad = lp && rq.return_rad != 0;
  const int rr_n = rq.rr_n;
  if (rrad) {
    const double *rr = b.rret + (size_t)rq.rr_slot * (2 * MAX_RR);
    for (int i = tid; i < rr_n; i += NT) {
      s_rr_rad[i] = rr[i];
      s_rr_ret[i] = rr[MAX_RR + i];
    }
  }
  __syncthreads();
  if (wave == 0) {
    // ISCO snap (src/Relprofile.cpp:195-200)
    const double rms = rq.rms;
    if (lane == 0 && (s_tre[n_r - 1] > rms) && ((s_tre[n_r - 1] - rms) / s_tre[n_r - 1] < 1e-3)) s_tre[n_r - 1] = rms;
    wave_lds_fence();  // (the other lanes read the node)
    int c_in = 0, c_out = 0;  // nodes not below Rin / Rout (bsearch_desc, src/relutility.c:195-211)
    for (int k = 0; k < n_r; k += 64) {
      const bool v = k + lane < n_r;
      const double t = s_tre[min(k + lane, n_r - 1)];
      c_in += __popcll(__ballot(v && !(t < rq.rin)));
      c_out += __popcll(__ballot(v && !(t < rq.rout)));
    }
    const int ind_rmin = min(max(c_in - 1, 0), n_r - 2), ind_rmax = min(max(c_out - 1, 0), n_r - 2);
    if (lane == 0) {
      int st = 0;
      // 1000 rg snap (:235-238)
      if (s_tre[ind_rmax] < 1000.0 && s_tre[ind_rmax] * 1.01 > 1000.0) s_tre[ind_rmax] = 1000.0;
      if (!(ind_rmin > 0) || !(s_tre[ind_rmin + 1] <= rq.rin) || !(s_tre[ind_rmin] >= rq.rin) ||
          !(s_tre[ind_rmax + 1] <= rq.rout) || !(s_tre[ind_rmax] >= rq.rout) ||
          !(ind_rmax <= ind_rmin) || !(rq.rout <= 1000.0)) {
        st = 12;
      }
      s_rmin = ind_rmin;
      s_st_edge = st;
    }
  }
  __syncthreads();
  if (s_st_edge) {
    if (tid == 0) b.status[req] = s_st_edge;
    return;
  }
  {  // the node arrays the radius records are rebuilt from (rad_geo)
    double *gn = b.rnode + (size_t)req * RAD_NODE_ARRAYS * n_r;
    for (int ir = tid; ir < n_r; ir += NT) {
      gn[ir] = s_tre[ir];
      gn[n_r + ir] = s_tgmin[ir];
      gn[2 * n_r + ir] = s_tgmax[ir];
    }
  }
  const double r1g = fine_radius_r1(rq.rout), r2g = fine_radius_r1(rq.rin);
  auto fr = [&](int ii) { return fine_radius_at(r1g, r2g, ii, nr); };

  // reflection fractions (calc_refl_frac, src/Rellp.cpp:36-89): lane 0 takes the
  // inner edge, lane 1 the outer one (the wavefront with the fewest radii)
  if (lp && wave == NW - 1) {
    const double edge = lane == 0 ? rq.rin : rq.rout;
    int klo = lane == 0 ? nr - 2 : 0;  // what the search below finds on a descending grid
    const bool plain = lane == 0 ? !(fr(klo) < edge) : (fr(1) < edge);
    if (!plain && lane < 2) {
      klo = 0;
      int khi = nr - 1;
      while (khi - klo > 1) {
        const int k = (khi + klo) / 2;
        if (fr(k) < edge) khi = k; else klo = k;
      }
    }
    double del = lp_on_fine(fr(klo), s_jr, s_je, s_jd, s_ji, ntr).del_emit;
    double dmax = s_jd[ntr - 1];
    if (dmax < PI / 2.0) dmax = PI / 2.0;
    if (rq.beta > 1e-6) del = relat_abberation(del, -1. * rq.beta);
    const double cdel = cos(del);
    const double cos_bh = readlane_d(cdel, 0), cos_ad = readlane_d(cdel, 1);
    LpRefl o;
    o.f_bh = 0.5 * (1.0 - cos_bh);
    o.f_ad = 0.5 * (cos_bh - cos_ad);
    o.f_inf_rest = 0.5 * (1.0 + cos(dmax));
    o.f_inf = (rq.beta > 1e-6) ? 0.5 * (1.0 + cos(relat_abberation(dmax, -1. * rq.beta))) : o.f_inf_rest;
    o.refl_frac = o.f_ad / o.f_inf;
    if (lane == 0) {
      if (!(o.f_inf + o.f_ad < 1.0)) s_st_refl = 20;
      b.refl[req] = o;
    }
  }

  // fine radii: node -> fine map (:249-300), emissivity, energy window (:859-878)
  RadRec *rad = b.rad + (size_t)req * nr;
  const GridGuess gE = grid_guess(E, rq.n_e);
  auto ge = [&](int k) { return E[k]; };
  const double e_lo = E[0], e_hi = E[rq.n_e];
  double area = 0.0;
  double cmax = 0.0;  // largest weight of a radius with a window
  int err = 0;
  for (int ii0 = 0; ii0 < nr; ii0 += NT) {  // same trip count in every wavefront
    const int ii = ii0 + tid;
    int wlo = 0x7fffffff, whi = -1;
    int izone = -1;
    if (ii < nr) {
    const double re = fr(ii);
    const double rprev = (ii > 0) ? fr(ii - 1) : 0.0;
    const double rnext = (ii < nr - 1) ? fr(ii + 1) : 0.0;
    // K = largest k <= ind_rmin with tre[k] > re: the walk of :250-265 starts
    // at the Rin bracket and only moves outwards, so a fine radius rounded
    // just below the innermost node extrapolates that bracket (ifac_r < 0)
    int lo = 0, hi = n_r;
    while (lo < hi) {
      int mid = (lo + hi) >> 1;
      if (s_tre[mid] > re) lo = mid + 1; else hi = mid;
    }
    int K = min(lo - 1, s_rmin);
    if (K < 0) {  // (re beyond the outermost node: the request fails, K stays in bounds)
      if (!(re - 1000.0 <= 1e-6)) err = 13;
      K = 0;
    }
    if (K >= n_r - 1) {  // cannot happen for rin >= tre[n_r-1]; keep in bounds
      K = n_r - 2;
      err = 13;
    }
    const RadGeo geo = rad_geo(s_tre, s_tgmin, s_tgmax, re, K);
    const double ifac_r = geo.ifac_r;
    if (ifac_r > 1.0 && K > 0) err = 14;
    const double gmin = geo.gmin;
    const double gmax = geo.gmax;
    const double tz = trapez_half(rprev, re, rnext, ii, nr);
    const double weight = tz / 2;
    double emis;
    if (!lp) {  // broken power law (get_emis_bkn, src/Rellp.cpp:421-437)
      const double alpha = (re > rq.rbr) ? rq.emis2 : rq.emis1;
      emis = pow(re / rq.rbr, -alpha);
      area += emis * (tz * 2);
    } else {
      emis = lp_emis_at(rq, re, s_jr, s_je, s_jd, s_ji, ntr, &err);
      if (rrad) {
        // the returning emissivity at this radius (rebin_emisprofile_on_radial_grid,
        // src/Rellp.cpp:120-175: linear radius factor, log-interpolated values)
        const int kk = min(max(bsearch_asc(s_rr_rad, rr_n, re), 0), rr_n - 2);
        const double f = (re - s_rr_rad[kk]) / (s_rr_rad[kk + 1] - s_rr_rad[kk]);
        const double er = exp(f * log(s_rr_ret[kk + 1]) + (1.0 - f) * log(s_rr_ret[kk]));
        emis = (rq.return_rad == 1) ? emis + er : er;
      }
    }
    // energy window
    double egmin = gmin, egmax = gmax;
    int ielo = 1, iehi = 0;
    if ((egmax > e_lo) && (egmin < e_hi)) {
      if (egmin < e_lo) egmin = e_lo;
      if (egmax > e_hi) egmax = e_hi;
      // binary_search (src/relutility.c:155-171) on [E0, E_n]: count - 1, at most n-1
      ielo = min(count_le(ge, rq.n_e, egmin, gE) - 1, rq.n_e - 1);
      iehi = min(count_le(ge, rq.n_e, egmax, gE) - 1, rq.n_e - 1);
    }
    // zone of the radius (binary_search on the zone edges, src/Relprofile.cpp:874)
    izone = (nz > 1) ? bsearch_asc(zg, nz + 1, re) : 0;
    const double coef = emis / (gmax - gmin) * weight;  // times ReqNorm.fac
    rad[ii] = rad_pack(coef, K, izone, ielo, iehi);
    if (ielo <= iehi) {
      wlo = ielo;
      whi = iehi;
      cmax = fmax(cmax, fabs(coef));
    }
    }  // ii < nr
    // energy window of the radius chunk (this wavefront's 64 consecutive
    // radii), per zone present in the chunk
    const int zlo = wave_min_i(ii < nr ? izone : 0x7fffffff);
    const int zhi = wave_max_i(ii < nr ? izone : -1);
    for (int z = zlo; z <= zhi; z++) {
      const int zl = wave_min_i(izone == z ? wlo : 0x7fffffff);
      const int zh = wave_max_i(izone == z ? whi : -1);
      if (lane == 0) {
        s_ulo[(ii / RAD_CHUNK) * NZ + z] = zl;
        s_uhi[(ii / RAD_CHUNK) * NZ + z] = zh;
      }
    }
  }
  if (err) atomicMax(&s_st_rad, err);
  // BKN normalisation: sum emis * 2 pi r dr (norm_emis_profile, src/Rellp.cpp:91-109),
  // applied through ReqNorm instead of a second pass over the records
  const double area_w = wave_sum(area), cmax_w = wave_max_d(cmax);
  if (lane == 0) {
    s_sum[wave] = area_w;
    s_max[wave] = cmax_w;
  }
  __syncthreads();
  if (const int st = s_st_rad ? s_st_rad : s_st_refl) {
    if (tid == 0) b.status[req] = st;
    return;
  }
  // work items: the window of each (radius chunk, zone) cut into segments
  // of seg_bins; the item's chunk and zone share its rc field.  An item's
  // time grows with its bins, so segments of at least S / 4 bins go to the
  // front of the list and the shorter last segments of windows to its back:
  // k_integrate hands out the long ones first and the wavefronts finish
  // together on short ones.  One wavefront lists the windows (64 at a time,
  // their numbers of segments summed across the lanes) and reserves the
  // request's places; another one writes the request's norms.
  const int S = b.seg_bins;
  const int thr = max(1, S / 4);
  const int n_cz = n_rc * nz;  // pairs q = c nz + z; their windows sit at c NZ + z
  if (wave == 0) {
    int jlo = 0x7fffffff, jhi = -1, tot = 0, tots = 0;
    for (int q0 = 0; q0 < n_cz; q0 += 64) {
      const int q = q0 + lane;
      int nlong = 0, nshort = 0;
      if (q < n_cz) {
        const int w = (q / nz) * NZ + q % nz;
        const int lo = s_ulo[w], hi = s_uhi[w];
        if (hi >= lo) {
          jlo = min(jlo, lo);
          jhi = max(jhi, hi);
          const int len = hi - lo + 1;
          const int nseg = (len + S - 1) / S;
          nlong = nseg - 1 + (len - (nseg - 1) * S >= thr ? 1 : 0);
          nshort = nseg - nlong;
        }
      }
      int pl = nlong, ps = nshort;  // inclusive sums over the lanes
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int ul = __shfl_up(pl, d, 64), us = __shfl_up(ps, d, 64);
        if (lane >= d) {
          pl += ul;
          ps += us;
        }
      }
      if (q < n_cz) {
        s_pref[q] = tot + pl - nlong;
        s_prefs[q] = tots + ps - nshort;
      }
      tot += __builtin_amdgcn_readlane(pl, 63);
      tots += __builtin_amdgcn_readlane(ps, 63);
    }
    jlo = wave_min_i(jlo);
    jhi = wave_max_i(jhi);
    if (lane == 0) {
      static_assert(CTR_ITEMS % 2 == 0 && CTR_ITEMS_S == CTR_ITEMS + 1, "one aligned 64-bit word");
      unsigned long long *ctr = reinterpret_cast<unsigned long long *>(&b.ctr[CTR_ITEMS]);
      int base, bases;
      bool first_out;
      // the host sizes the list for the bins that the table's radii reach
      // (reach_bins); a request that it does not hold all the same fails, and its
      // neighbours' items stay whole
      if (!reserve_items([&](uint64_t v) { return (uint64_t)atomicAdd(ctr, (unsigned long long)v); }, tot, tots,
                         b.item_cap, base, bases, first_out)) {
        atomicOr(&b.ctr[CTR_ITEMS_OVF], 1);
        if (first_out) {
          b.ctr[CTR_FIT] = base;
          b.ctr[CTR_FIT_S] = bases;
        }
        base = -1;
      }
      s_base = base;
      s_bases = bases;
      s_jlo = jlo;
      s_jhi = jhi;
      b.reach[req] = BinRange{jlo, jhi};
    }
  } else if (wave == 1 && lane == 0) {
    double total = s_sum[0], cmax_all = s_max[0];
    for (int w = 1; w < NW; w++) {
      total += s_sum[w];
      cmax_all = fmax(cmax_all, s_max[w]);
    }
    ReqNorm n;
    n.fac = lp ? 1.0 : 1.0 / total;
    n.fa = fa;
    n.fm = fm;
    n.ia = ia;
    n.im = im;
    n.r1 = r1g;
    n.r2 = r2g;
    const double m = cmax_all * n.fac;
    int k = 0;
    if (m > 0.0 && m < INFINITY) k = min(1000, max(-1000, -ilogb(m)));
    n.cmul = ldexp(n.fac, k);
    n.cinv = ldexp(1.0, -k);
    b.rnorm[req] = n;
  }
  __syncthreads();
  // the profile accumulates with atomic adds: clear the bins any window
  // reaches (k_finalize writes zeros elsewhere); every zone's profile over the
  // union of the windows.  (No window reaches the grid: jlo = INT_MAX > jhi =
  // -1, nothing to clear; jlo + tid must not be formed then, it would overflow.)
  const int jlo = s_jlo, jhi = s_jhi;
  double *acc = profile_acc(b, rq);
  if (jlo <= jhi)
    for (int z = 0; z < nz; z++)
      for (int j = jlo + tid; j <= jhi; j += NT) acc[(size_t)z * rq.n_e + j] = 0.0;
  if (s_base >= 0) {
    // SEG_LANES lanes a window, a lane per segment (all but the last are S bins
    // long): one lane a window took 2-9 us for segments of one bin
    constexpr int SEG_LANES = 16;
    for (int q = tid / SEG_LANES; q < n_cz; q += NT / SEG_LANES) {
      const int c = q / nz, z = q % nz, w = c * NZ + z;
      const int k = s_base + s_pref[q], ks = s_bases + s_prefs[q];
      const int uhi = s_uhi[w];
      int i = tid % SEG_LANES;
      for (int64_t j0 = s_ulo[w] + (int64_t)i * S; j0 <= uhi; j0 += SEG_LANES * (int64_t)S, i += SEG_LANES) {
        WorkItem it;
        it.req = req;
        it.rc = c | (z << 16);
        it.j0 = (int)j0;
        it.j1 = (int)min((int64_t)uhi + 1, j0 + S);
        if (it.j1 - it.j0 >= thr) b.items[k + i] = it;
        else b.items[b.item_cap - 1 - ks] = it;
      }
    }
  }
  if (tid == 0) b.status[req] = s_base >= 0 ? 0 : ST_WORKLIST;
}

// Radial zones of the relxill and xillver requests (IonGradient,
// src/IonGradient.cpp:182-209, :421-430): the zone record (centre, and for the
// lamp post the emission angle, energy shift and xillver brackets the zone
// sees) and, for the lamp post, the normalisation change of the incident
// spectrum (src/Xillspec.cpp:408-435), one wavefront per (request, zone).  The
// change is a ratio of two sums over the 500-bin grid (the cut-off power law; 8
// exponentials a lane and sum) or of two nthcomp norms (k_nth, which runs
// before).  Zone 0's wavefront keeps the norm of the primary at the source
// (calcNormWrtXillverTableSpec on the 500-bin grid, src/PrimarySource.h:238-292)
// and its energy boost for k_primary.
// Bound: the latency of the table rows and the sums, 15 us alone, 20 us for 1280
// zones (inside k_setup, zone after zone with tree sums: 18 us and 22 us, but
// after the returning radiation that reads the records).
constexpr int ZONE_LDS = 4 * MAX_LP_R;  // doubles
// (nt threads; the first wavefront's do the work behind the lamp post's rows)
__device__ __forceinline__ void zone_unit(const BatchDev &b, const XillWork wk, int lane, int nt, double *lds) {
  double *s_jr = lds, *s_je = lds + MAX_LP_R, *s_jd = lds + 2 * MAX_LP_R, *s_ji = lds + 3 * MAX_LP_R;
  const int req = wk.req, z = wk.zone;
  const ReqParams &rq = b.req[req];
  if (rq.pre_status != 0) return;  // uniform over the block
  const DevXillTable &xt = b.xt[rq.prim];
  const bool lp = rq.emis_type == EMIS_LP;
  const double gam = rq.xgam;
  double ect = rq.xect_src;
  ZoneRec zr;
  if (rq.model == MOD_XILLVER) {  // no relativistic part: the request's brackets
    zr = ZoneRec();
    zr.shift = 1.0;
    zr.ect_ind = xt.ect_dim >= 0 ? rq.xind[xt.ect_dim] : 0;
    zr.ect_fac = xt.ect_dim >= 0 ? rq.xfac[xt.ect_dim] : 0.0;
    zr.lxi_ind = xt.lxi_dim >= 0 ? rq.xind[xt.lxi_dim] : 0;
    zr.lxi_fac = xt.lxi_dim >= 0 ? rq.xfac[xt.lxi_dim] : 0.0;
  } else {
    if (lp) lp_rows(b.lp, rq, s_jr, s_je, s_jd, s_ji, lane, nt);
    if (lane >= 64) return;
    zr = zone_record(xt, rq, z, lp, s_jr, s_je, s_jd, s_ji, b.lp.n_r, b.nr_fine, &ect);
  }
  if (lane >= 64) return;
  zr.ncf = 1.0;
  zr.pe = 0.0;
  if (rq.prim == PRIM_NTHCOMP) {
    const NthRes *n = b.nth + rq.nth_off;
    zr.nf = n[0].nf;
    if (lp) {
      zr.ncf = n[1 + z].nf / n[0].nf;
      zr.pe = n[1 + z].pe;
    }
  } else {
    const double part = rq.prim == PRIM_BBODY ? bbody_norm_part(b.cg, rq.xktbb, lane, 64)
                                              : xill_norm_part(b.cg, rq.xect_src, gam, lane, 64);
    zr.nf = 1. / (wave_sum(part) / NORM_XILLVER_TABLE);
    if (lp) {
      const double disk = 1. / (wave_sum(xill_norm_part(b.cg, ect, gam, lane, 64)) / NORM_XILLVER_TABLE);
      zr.ncf = disk / zr.nf;
      // energy flux of the zone's normalised primary in 0.1-1000 keV
      // (get_xillver_fluxcorr, src/Xillspec.cpp:344-362)
      double pe = 0.0;
      if (rq.rr_corr) {
        for (int k = lane; k < N_ENER_COARSE; k += 64) {
          const double e0 = b.cg.coarse[k], e1 = b.cg.coarse[k + 1];
          if (e0 >= 0.1 && e1 <= 1000.0)
            pe += cutoffpl_bin(e0, e1, b.cg.coarse_ln[k], ect, gam) * disk * 0.5 * (e0 + e1);
        }
      }
      zr.pe = wave_sum(pe);
    }
  }
  zr.boost = 1.0;
  if (lp) {  // flux_boost_source_to_observer, src/PrimarySource.h:84-93
    zr.boost = pow(rq.g_so, gam);
    if (rq.beta > 1e-4) {
      const double dop = sqrt(1.0 - rq.beta * rq.beta) / (1.0 + rq.beta * cos(M_PI - rq.incl));
      zr.boost *= pow(dop, 2);
    }
  }
  if (lane == 0) b.zone[rq.zone_off + z] = zr;
}

__global__ __launch_bounds__(64) void k_zone(BatchDev b, const XillWork *__restrict__ work) {
  __shared__ double s_lds[ZONE_LDS];
  zone_unit(b, work[blockIdx.x], threadIdx.x, 64, s_lds);
}

// The eight corners of a request's xillver table row on the interpolated axes
// other than zax (zax index 0), each with its weight, in rows of ni
// inclinations; one step on zax moves a row by *stride rows.
__device__ inline void corners8(const DevXillTable &xt, const ReqParams &rq, int zax, double *w8, unsigned *cb,
                                unsigned *stride) {
  unsigned st = 1;
#pragma unroll
  for (int k = 0; k < 4; k++)
    if (k > zax) st *= (unsigned)xt.n_val[k];
#pragma unroll
  for (int c = 0; c < 8; c++) {
    double w = 1.0;
    unsigned r = 0;
    int bit = 2;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      int idx = 0;
      if (k != zax) {
        const int o = (c >> bit) & 1;
        bit--;
        w *= o ? rq.xfac[k] : (1.0 - rq.xfac[k]);
        idx = rq.xind[k] + o;
      }
      r = r * (unsigned)xt.n_val[k] + (unsigned)idx;
    }
    w8[c] = w;
    cb[c] = r * (unsigned)xt.n_incl;
  }
  *stride = st;
}

// relxilllp's returning radiation above spin 0: the band sums behind the
// zones' xillver correction factors (calc_rrad_corr_factors,
// src/Relxill.cpp:164-182, with get_xillver_fluxcorrection_factors,
// src/Xillspec.cpp:500-526).  A zone's xillver spectra for every inclination
// are averaged with the weights of calc_angle_averaged_xill_spec (:109-126:
// 0.5 cos(i) / n_incl with the table's inclination, in degrees, read as
// radians); of the average this takes
//   [0] the energy flux in 0.1-1000 keV (:344-362),
//   [1] the photon flux in 0.15-500 keV,
//   [2] the photon flux there of the average shifted 1.5 times lower in energy
//       (rebinned, times 2/3; :454-487): the bins of the band are contiguous,
//       so their shares of the average add up to its photons in the band's
//       shifted ends [xt.rr_lo, xt.rr_hi], and no bin is searched for.
// All three are linear in the average, and the zones differ only in their
// bracket (i_z, f_z) on the Ecut axis: so the sums are taken once per Ecut
// node that some zone's bracket touches, and zone z gets those of nodes i_z and
// i_z + 1 (k_rrad weights them).  An ionisation gradient gives every zone its
// own logXi bracket too; then each zone takes its own 16 corners.
// One workgroup per (request, RRA_THREADS table bins), one bin a thread; the
// partial sums go to rrpart[zone][node][chunk][3].
// Bound: L2 / HBM reads of 80 rows per Ecut node.  One workgroup per (request,
// zone) with 160 rows a zone and the shift's rebin took 144 us for one request (362 us with a density
// division, 696 us for 64 of those); this takes 16 us (16 us, 28 us), with the brackets from
// the lamp post's rows 24 us, but beside the zone records.
// The brackets are taken from the lamp post's rows here too, so that the sums
// need nothing of k_zone or k_nth and run beside them (k_before_rrad).
struct RradLds {
  double rows[ZONE_LDS];
  double wa[MAX_INCL];
  double w[3][RRA_THREADS / 64];
  double ect_fac[MAX_ZONES], lxi_fac[MAX_ZONES];
  int ect_ind[MAX_ZONES], lxi_ind[MAX_ZONES];
};
__device__ __forceinline__ void rrad_sums(const BatchDev &b, int req, int chunk, int tid, RradLds &S) {
  double *s_wa = S.wa, (*s_w)[RRA_THREADS / 64] = S.w;
  int *s_ind = S.ect_ind;
  const ReqParams &rq = b.req[req];
  const DevXillTable xt = b.xt[rq.prim];
  const int chunks = rrad_chunks(xt.n_ener);  // of this request's table
  if (rq.pre_status != 0 || chunk >= chunks) return;  // uniform over the block
  const DensDiv dd = dens_of(rq.xdens_div);
  const int nz = rq.n_zones, ni = xt.n_incl, ne = xt.n_ener;
  const int zax = xt.ect_dim >= 0 ? xt.ect_dim : 3;
  const bool grad = rq.ion_grad == 1 && xt.lxi_dim >= 0;
  for (int a = tid; a < ni; a += RRA_THREADS) {
    const double incl_deg = (double)xt.incl_vals[a] * 180 / PI;
    s_wa[a] = 0.5 * cos(incl_deg * PI / 180) / ni;
  }
  if (xt.ect_dim >= 0 || grad) {
    double *jr = S.rows, *je = jr + MAX_LP_R, *jd = je + MAX_LP_R, *ji = jd + MAX_LP_R;
    lp_rows(b.lp, rq, jr, je, jd, ji, tid, RRA_THREADS);
    if (tid < nz) {
      double ect;
      const ZoneRec zr = zone_record(xt, rq, tid, true, jr, je, jd, ji, b.lp.n_r, b.nr_fine, &ect);
      s_ind[tid] = xt.ect_dim >= 0 ? zr.ect_ind : rq.xind[3];
      S.ect_fac[tid] = zr.ect_fac;
      S.lxi_ind[tid] = zr.lxi_ind;
      S.lxi_fac[tid] = zr.lxi_fac;
    }
  } else if (tid < nz) {
    s_ind[tid] = rq.xind[3];
  }
  __syncthreads();
  const int e = chunk * RRA_THREADS + tid;
  const bool in = e < ne;
  const size_t eb = in ? e : 0;  // a valid address; bins beyond the table weigh nothing
  const double e0 = xt.ener[eb], e1 = xt.ener[eb + 1];
  const double we = (in && e0 >= 0.1 && e1 <= 1000.0) ? 0.5 * (e0 + e1) : 0.0;
  const double wp = (in && e0 >= 0.15 && e1 <= 500.0) ? 1.0 : 0.0;
  const double zlo = fmax(e0, xt.rr_lo), zhi = fmin(e1, xt.rr_hi);
  const double wz = (in && zhi > zlo) ? (zhi - zlo) / (e1 - e0) * (2. / 3.) : 0.0;
  double *part = b.rrpart + rq.rr_corr_off;
  // the block's sums of a spectrum with value avg in this thread's bin, to nodes
  // [n0, n1] of zone z
  double sums[3];
  auto reduce = [&](double avg) {
    const double v[3] = {wave_sum(avg * we), wave_sum(avg * wp), wave_sum(avg * wz)};
    __syncthreads();  // the last sums have been read
    if ((tid & 63) == 0)
      for (int k = 0; k < 3; k++) s_w[k][tid >> 6] = v[k];
    __syncthreads();
    for (int k = 0; k < 3; k++) {
      sums[k] = 0.0;
      for (int w = 0; w < RRA_THREADS / 64; w++) sums[k] += s_w[k][w];
    }
  };
  auto store = [&](int z, int node) {
    if (tid < 3) part[((size_t)(2 * z + node) * chunks + chunk) * 3 + tid] = sums[tid];
  };
  const int n_o = xt.n_out > 1 ? 2 : 1;
  const size_t nel = (size_t)ne;
  if (!grad) {
    int elo = s_ind[0], ehi = s_ind[0];
    for (int z = 1; z < nz; z++) {
      elo = min(elo, s_ind[z]);
      ehi = max(ehi, s_ind[z]);
    }
    double w8[8];
    unsigned cb[8], stride;
    corners8(xt, rq, zax, w8, cb, &stride);
    for (int nd = elo; nd <= ehi + 1; nd++) {
      bool used = false;
      for (int z = 0; z < nz; z++) used |= nd == s_ind[z] || nd == s_ind[z] + 1;
      if (!used) continue;  // uniform
      double avg = 0.0;
      for (int a = 0; a < ni; a++) {
        const unsigned po = (unsigned)nd * stride * (unsigned)ni + (unsigned)a;
        double sv = 0.0;
        for (int o = 0; o < n_o; o++) {  // (a six-parameter table: both brackets of its first axis)
          const double wo = n_o == 1 ? 1.0 : (o ? rq.xo_fac : 1.0 - rq.xo_fac);
          const size_t ob = (size_t)(rq.xo_ind + o) * xt.outer_rows;
          double so = 0.0;
#pragma unroll
          for (int c = 0; c < 8; c++) so += w8[c] * xval(xt.spec[(ob + cb[c] + po) * nel + eb], dd);
          sv += wo * so;
        }
        avg += s_wa[a] * sv;
      }
      reduce(avg);
      for (int z = 0; z < nz; z++) {
        if (s_ind[z] == nd) store(z, 0);
        if (s_ind[z] + 1 == nd) store(z, 1);
      }
    }
    return;
  }
  for (int z = 0; z < nz; z++) {
    const double zef = S.ect_fac[z], zlf = S.lxi_fac[z];
    const int zei = S.ect_ind[z], zli = S.lxi_ind[z];
    double avg = 0.0;
    for (int c = 0; c < 16; c++) {  // the zone's own Ecut and logXi brackets
      double w = 1.0;
      unsigned r = 0;
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const bool ie = (k == xt.ect_dim), il = (k == xt.lxi_dim);
        const int o = (c >> (3 - k)) & 1;
        const double f = ie ? zef : (il ? zlf : rq.xfac[k]);
        w *= o ? f : (1.0 - f);
        r = r * (unsigned)xt.n_val[k] + (unsigned)((ie ? zei : (il ? zli : rq.xind[k])) + o);
      }
      for (int o = 0; o < n_o; o++) {
        const double wo = n_o == 1 ? w : w * (o ? rq.xo_fac : 1.0 - rq.xo_fac);
        const size_t row = (size_t)(rq.xo_ind + o) * xt.outer_rows + (size_t)r * ni;
        double sa = 0.0;
        for (int a = 0; a < ni; a++) sa += s_wa[a] * xval(xt.spec[(row + a) * nel + eb], dd);
        avg += wo * sa;
      }
    }
    reduce(avg);
    store(z, 0);
    store(z, 1);
  }
}

// Returning radiation (add_returnrad_emis, src/Rellp.cpp:483-507, with
// get_rrad_emis_corona, src/Relreturn_Corona.cpp:291-321): the returning
// emissivity of a request's table zones, sum_re frac_g g^(Gamma-1) tf_r
// emis(re) (calc_rrad_emis_corona, :119-151), which k_setup log-interpolates
// onto the fine radii.  One wavefront per incident zone (RR_ZONES to a
// workgroup), its lanes the emitting zones (at most 64); the direct emissivity
// at a zone's centre is interpolated between the two fine radii around it
// (inv_rebin_mean, src/relutility.c:636-663).  The frac_g weight is
// g^(Gamma-1), or with a g-shift factor off 1 by more than 1e-3 of the emitting
// zone its corrected boost over g (calc_rrad_emis_zone, :87-108); the sum times
// the incident zone's flux factor.
// Bound: FP64 issue of a pow per (incident, emitting zone, energy-shift bin),
// 50 x 50 x 20 a request, and before it the latency of the emissivity's chain:
// about 180 us on the one CU of the request's k_setup workgroup (239 -> 59 us
// without it), 24 us over the CUs of its 13 workgroups here (29 us with both
// emissivities of a zone and the search for its radii on one thread); 270 us
// and 57 us for 64 requests.
// SPLIT: a workgroup's wavefronts share one incident zone's energy-shift bins,
// for few requests, which leave the chip idle (1 request 14 us).
constexpr int RR_ZONES = 4;
template <int SPLIT>
__global__ __launch_bounds__(64 * RR_ZONES) void k_rrad(BatchDev b, const int *__restrict__ reqs) {
  constexpr int NT = 64 * RR_ZONES, PER = SPLIT ? 1 : RR_ZONES, GROUPS = MAX_RR / PER;
  __shared__ double s_jr[MAX_LP_R], s_je[MAX_LP_R], s_jd[MAX_LP_R], s_ji[MAX_LP_R];
  __shared__ double s_rad[MAX_RR], s_in[MAX_RR], s_cf[MAX_RR], s_cg[MAX_RR], s_corr[2];
  __shared__ double s_zf[MAX_ZONES], s_zg[MAX_ZONES], s_e[2][MAX_RR], s_r[2][MAX_RR];
  __shared__ double s_term[RR_ZONES][64];
  const int req = reqs[blockIdx.x / GROUPS], i0 = (blockIdx.x % GROUPS) * PER;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const ReqParams &rq = b.req[req];
  const int rr_n = rq.rr_n, nr = b.nr_fine, nz = rq.n_zones;
  if (rq.pre_status != 0 || i0 >= rr_n) return;  // uniform over the block
  const DevLpTable &L = b.lp;
  lp_rows(L, rq, s_jr, s_je, s_jd, s_ji, tid, NT);
  const DevRradTable &R = b.rr;
  const int nt = R.n_rad, k = rq.rr_k, klo = rq.rr_klo;
  const double *rlo_t = R.rlo + (size_t)k * nt, *rhi_t = R.rhi + (size_t)k * nt;
  const double rin_f = fine_radius(rq.rin, rq.rout, nr - 1, nr), rout_f = fine_radius(rq.rin, rq.rout, 0, nr);
  // wavefronts 0 and 1: the emissivity at the fine radius outside and inside
  // each table zone's centre; 2: the end zones; 3: the relxill zones' factors
  auto centre = [&](int i) {
    const double lo = (i == 0) ? rin_f : rlo_t[klo + i];
    const double hi = (i == rr_n - 1) ? rout_f : rhi_t[klo + i];
    return 0.5 * (lo + hi);
  };
  if (wave < 2) {
    if (lane < rr_n) {
      int err = 0;  // (k_setup evaluates and flags every fine radius)
      const double q1 = fine_radius_r1(rq.rout), q2 = fine_radius_r1(rq.rin);
      const int a = fine_above(q1, q2, centre(lane), nr) + wave;
      const double r = fine_radius_at(q1, q2, a, nr);
      s_r[wave][lane] = r;
      s_e[wave][lane] = lp_emis_at(rq, r, s_jr, s_je, s_jd, s_ji, L.n_r, &err);
    }
  } else if (wave == 2) {  // ring-area corrections of the end zones (src/Relreturn_Table.cpp:415-435)
    if (lane < 2) {
      const int i = (lane == 0) ? 0 : rr_n - 1;
      double rl = rlo_t[klo + i];
      if (klo + i == 0 && rl > rq.rms) rl = rq.rms;
      const double rh = rhi_t[klo + i];
      const double lo = (i == 0) ? rin_f : rlo_t[klo + i];
      const double hi = (i == rr_n - 1) ? rout_f : rhi_t[klo + i];
      s_corr[lane] = (0.5 * (lo + hi) * (hi - lo)) / (0.5 * (rl + rh) * (rh - rl));
    }
  } else if (rq.rr_corr && lane < nz) {
    // the correction factors of relxill zone lane from its band sums (rrad_sums):
    //   flux factor = energy flux over that of the zone's normalised primary
    //   (k_zone); g factor = photon flux over the shifted one's, over 1.5^Gamma
    const ZoneRec zr = b.zone[rq.zone_off + lane];
    const DevXillTable &xt = b.xt[rq.prim];
    const double f = xt.ect_dim >= 0 ? zr.ect_fac : rq.xfac[3];
    const int chunks = rrad_chunks(xt.n_ener);
    const double *part = b.rrpart + rq.rr_corr_off + (size_t)(2 * lane) * chunks * 3;
    double s[3] = {0.0, 0.0, 0.0};
#pragma unroll 4
    for (int c = 0; c < chunks; c++)
      for (int j = 0; j < 3; j++) s[j] += (1.0 - f) * part[c * 3 + j] + f * part[(chunks + c) * 3 + j];
    s_zf[lane] = s[0] / zr.pe;
    s_zg[lane] = s[1] / s[2] / pow(1.5, rq.xgam);
  }
  __syncthreads();
  if (tid < rr_n) {
    const double rm = centre(tid);
    s_rad[tid] = rm;
    // relxilllp above spin 0: the correction factors of the relxill zone
    // the table zone's centre falls in (rebin_corrfactors_to_rradtable_grid,
    // src/Relreturn_Corona.cpp:248-289; a centre beyond the last edge takes
    // the last zone)
    double cf = 1.0, cg = 1.0;
    if (rq.rr_corr) {
      const double *zg = rq.zgrid;
      int ind = bsearch_asc(zg, nz + 1, rm);
      if (rm < zg[0]) ind = 0;
      else if (rm > zg[nz] || ind > nz - 1) ind = nz - 1;
      cf = s_zf[ind];
      cg = s_zg[ind];
    }
    s_cf[tid] = cf;
    s_cg[tid] = cg;
    const double r0 = s_r[0][tid], r1 = s_r[1][tid];
    s_in[tid] = lerp1((rm - r1) / (r0 - r1), s_e[1][tid], s_e[0][tid]);
  }
  __syncthreads();
  const int i = SPLIT ? i0 : i0 + wave, j = lane, ng = R.n_g;
  if (i >= rr_n) return;  // (SPLIT: not reached; else no barrier below)
  double term = 0.0;
  if (j < rr_n) {
    const size_t t = (size_t)k * nt * nt + (size_t)(klo + i) * nt + (klo + j);
    const double gmin = R.gmin[t], gmax = R.gmax[t];
    const double cgj = s_cg[j];
    double ez = 0.0;
    for (int jj = SPLIT ? wave : 0; jj < ng; jj += SPLIT ? RR_ZONES : 1) {
      const double g = (jj + 0.5) / ng * (gmax - gmin) + gmin;  // get_gfac_grid (src/Relreturn_Datastruct.cpp:51-59)
      double v = R.frac_g[t * ng + jj];
      if (fabs(cgj - 1) > 1e-3) v *= gshift_boost(cgj, g, rq.gamma) / g;
      else if (fabs(g - 1) > 1e-3) v *= pow(g, rq.gamma - 1);
      ez += v;
    }
    double tf = R.tf_r[t];
    if (j == 0 && i < rr_n - 1) tf *= s_corr[0];
    if (j == rr_n - 1 && i < rr_n - 2) tf *= s_corr[1];
    term = ez * tf * s_in[j];
  }
  if constexpr (SPLIT) {
    s_term[wave][lane] = term;
    __syncthreads();
    if (wave > 0) return;
    term = 0.0;
    for (int w = 0; w < RR_ZONES; w++) term += s_term[w][lane];
  }
  const double sum = wave_sum(term);
  if (lane == 0) {
    double *o = b.rret + (size_t)rq.rr_slot * (2 * MAX_RR);
    o[i] = s_rad[i];
    o[MAX_RR + i] = sum * s_cf[i];
  }
}

// relxill models with the nthcomp primary (relxillCp, relxilllpCp): one
// Kompaneets solve per (request, j) of work, j = 0 for the source's kTe (the
// nthcomp models keep kTe in the source frame, src/Relxill.cpp:197-200),
// j = 1 + z for the kTe lamp-post zone z sees (kTe times the zone's source ->
// disk energy shift, src/IonGradient.cpp:196-209, from zone_record).  Each solve writes its normalisation nf on the
// 500-bin grid and the energy flux of the normalised spectrum in 0.1-1000 keV
// (calc_xillver_normalization_change_source_to_disk, src/Xillspec.cpp:408-435;
// get_xillver_fluxcorr, :344-362); the source's also keeps its solution for
// k_primary.  First in a run: k_zone reads the results.
constexpr int NTH_THREADS_R = 256;

struct NthJobLds {
  NthLds L;
  double red[NTH_THREADS_R];
  double kte;
};
__device__ __forceinline__ void nth_job(const BatchDev &b, const XillWork wk, int tid, NthJobLds &S) {
  NthLds &L = S.L;
  double *s_red = S.red;
  const int req = wk.req, j = wk.zone;
  const ReqParams &rq = b.req[req];
  if (rq.pre_status != 0) return;  // uniform over the block
  if (j == 0) {
    if (tid == 0) S.kte = rq.xect_src;
  } else {
    // the lamp-post rows in the solve's arrays (the solve overwrites them)
    lp_rows(b.lp, rq, L.t1, L.t2, L.t3, L.d, tid, NTH_THREADS_R);
    if (tid == 0) {
      double ect;
      (void)zone_record(b.xt[rq.prim], rq, j - 1, true, L.t1, L.t2, L.t3, L.d, b.lp.n_r, b.nr_fine, &ect);
      S.kte = ect;
    }
  }
  __syncthreads();
  const double kte = S.kte;
  const int nth = nth_solve(L, nth_grid_tab(b.nth_tab), kte, rq.xgam, tid, NTH_THREADS_R);
  // the spectrum on the 500-bin grid (spec_nthcomp at z = 0), per bin in t2
  const double nfac = nthcomp_normfac(L.x, L.t1, nth, 0.0);
  const double *ce = b.cg.coarse;
  double sp = 0.0;
  for (int k = tid; k < N_ENER_COARSE; k += NTH_THREADS_R) {
    const double e0 = ce[k], e1 = ce[k + 1];
    const double f = nthcomp_bin(e0, e1, nthcomp_edge(L.x, L.t1, nth, e0, 0.0), nthcomp_edge(L.x, L.t1, nth, e1, 0.0),
                                 nfac);
    L.t2[k] = f;
    if (e0 >= 0.1 && e0 <= 1000.0) sp += f * 0.5 * (e0 + e1) * 1e20 * 1.602177e-09;
  }
  const double nf = 1. / (block_sum(sp, s_red) / NORM_XILLVER_TABLE);
  double pe = 0.0;
  for (int k = tid; k < N_ENER_COARSE; k += NTH_THREADS_R) {
    const double e0 = ce[k], e1 = ce[k + 1];
    if (e0 >= 0.1 && e1 <= 1000.0) pe += L.t2[k] * nf * 0.5 * (e0 + e1);
  }
  const double s_pe = block_sum(pe, s_red);
  if (tid == 0) b.nth[rq.nth_off + j] = NthRes{nf, s_pe};
  if (j == 0) {
    double *xo = b.nth_x + (size_t)rq.nth_sol * (NTH_N + 1);
    double *so = b.nth_s + (size_t)rq.nth_sol * NTH_N;
    for (int i = tid; i <= nth; i += NTH_THREADS_R) xo[i] = L.x[i];
    for (int i = tid; i < NTH_N; i += NTH_THREADS_R) so[i] = L.t1[i];
    if (tid == 0) b.nth_n[rq.nth_sol] = nth;
  }
}

__global__ __launch_bounds__(NTH_THREADS_R) void k_nth(BatchDev b, const XillWork *__restrict__ work) {
  __shared__ NthJobLds s_job;
  nth_job(b, work[blockIdx.x], threadIdx.x, s_job);
}

// Before k_rrad, side by side: the xillver band sums, and the nthcomp solves
// (NTH) or the zone records.  One after the other zones and sums were 17 us and
// 16 us of a relxilllp call, solves, zones and sums 23 us, 10 us and 16 us of a
// relxilllpCp call; 24 us, and 24 us and 10 us, here.
template <int NTH>
__global__ __launch_bounds__(RRA_THREADS) void k_before_rrad(BatchDev b, const XillWork *__restrict__ work, int n_work,
                                                             const int *__restrict__ reqs, int n_chunk) {
  static_assert(RRA_THREADS == NTH_THREADS_R, "one workgroup size");
  constexpr size_t LDS = NTH ? (sizeof(NthJobLds) > sizeof(RradLds) ? sizeof(NthJobLds) : sizeof(RradLds))
                             : sizeof(RradLds);
  __shared__ __align__(16) char s_raw[LDS];
  const int tid = threadIdx.x;
  if ((int)blockIdx.x < n_work) {
    if constexpr (NTH) nth_job(b, work[blockIdx.x], tid, *reinterpret_cast<NthJobLds *>(s_raw));
    else zone_unit(b, work[blockIdx.x], tid, RRA_THREADS, reinterpret_cast<double *>(s_raw));
    return;
  }
  const int k = blockIdx.x - n_work;
  rrad_sums(b, reqs[k / n_chunk], k % n_chunk, tid, *reinterpret_cast<RradLds *>(s_raw));
}

// First in a run: clears its counters and, for an evaluation call, copies the
// request block (parameters, work lists, grids, input) from pinned host memory:
// the launch graph of a call on one grid then holds its transfers too, and a
// call makes one launch and one wait where it made about nine copies of 5-10 us
// each before the kernels and three after them.
constexpr int COPY_THREADS = 256;
__global__ __launch_bounds__(COPY_THREADS) void k_begin(int *ctr, const uint4 *__restrict__ src,
                                                        uint4 *__restrict__ dst, int64_t n16) {
  if (blockIdx.x == 0)
    for (int i = threadIdx.x; i < N_COUNTERS; i += COPY_THREADS) ctr[i] = 0;
  for (int64_t i = (int64_t)blockIdx.x * COPY_THREADS + threadIdx.x; i < n16; i += (int64_t)gridDim.x * COPY_THREADS)
    dst[i] = src[i];
}

// What a request's last workgroup delivers where a run's last kernel has one
// workgroup a request (k_finalize for line models, k_conv for one zone): its
// status and, the first workgroup's, the counters.  A launch of k_deliver less:
// relline call 63 us and 59 us, relconv call 92 us and 87 us, relxill call 100
// us and 92 us.
__device__ inline void deliver_words(const BatchDev &b, const Deliver &dl, int req, int tid) {
  if (!dl.res) return;
  if (tid == 0) dl.res[RES_CTR + req] = b.status[req];
  if (blockIdx.x == 0 && tid < RES_CTR) dl.res[tid] = b.ctr[tid];
}

// Last in a run: counters, statuses and (calls, server) outputs to pinned host
// memory, where the host reads them once the stream is done.
__global__ __launch_bounds__(COPY_THREADS) void k_deliver(BatchDev b, int *__restrict__ res,
                                                          double *__restrict__ res_out, int64_t n_out) {
  const int64_t i0 = (int64_t)blockIdx.x * COPY_THREADS + threadIdx.x, step = (int64_t)gridDim.x * COPY_THREADS;
  if (i0 < RES_CTR) res[i0] = b.ctr[i0];
  for (int64_t i = i0; i < b.n_req; i += step) res[RES_CTR + i] = b.status[i];
  const double2 *o2 = reinterpret_cast<const double2 *>(b.out);
  double2 *r2 = reinterpret_cast<double2 *>(res_out);
  for (int64_t i = i0; i < n_out / 2; i += step) r2[i] = o2[i];
  if ((n_out & 1) && i0 == 0) res_out[n_out - 1] = b.out[n_out - 1];
}

// ---------------------------------------------------------------------------
// integrate: the hot loop (calc_relline_profile, src/Relprofile.cpp:857-900)
// ---------------------------------------------------------------------------
namespace {

// One row of a fine radius (2 n_g values), lerped from its two node rows into
// LDS; 8 values per round, so that a round's 16 loads are in flight together.
template <class TV>
__device__ inline void lerp_row(double ifac, const double *lo, const double *hi, int nq, TV *dst) {
  for (int q0 = 0; q0 < nq; q0 += 8) {
    double a[8], c[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const int q = min(q0 + k, nq - 1);
      a[k] = lo[q];
      c[k] = hi[q];
    }
#pragma unroll
    for (int k = 0; k < 8; k++)
      if (q0 + k < nq) dst[q0 + k] = (TV)lerp1_(ifac, a[k], c[k]);
  }
}

// A request's (a, mu0)-interpolated node rows (interpol_a_mu0,
// src/Relprofile.cpp:39-80), read from the table's four corners: row ir,
// column c (g* column c >> 1, branch c & 1) of the transfer function or of
// the emission-angle cosines.  k_integrate, k_fixup and the angle distributions
// all build their rows from it, so every consumer sees the same bits.
struct NodeSrc {
  const float *a1, *a2;  // branch 0 and 1 arrays
  size_t s00, s10, s01, s11;
  double fa, fm;
  int ng;
};

__device__ inline NodeSrc node_src(const DevRelTable &T, const ReqNorm &rn, bool cos) {
  NodeSrc s;
  s.a1 = cos ? T.cosne1 : T.trff1;
  s.a2 = cos ? T.cosne2 : T.trff2;
  const size_t nq = (size_t)T.n_r * T.n_g;
  s.s00 = ((size_t)rn.ia * T.n_mu0 + rn.im) * nq;
  s.s10 = ((size_t)(rn.ia + 1) * T.n_mu0 + rn.im) * nq;
  s.s01 = ((size_t)rn.ia * T.n_mu0 + rn.im + 1) * nq;
  s.s11 = ((size_t)(rn.ia + 1) * T.n_mu0 + rn.im + 1) * nq;
  s.fa = rn.fa;
  s.fm = rn.fm;
  s.ng = T.n_g;
  return s;
}

// (the branch arrays are taken into locals before the select: a select
// between two members' addresses would put the struct in scratch memory)
__device__ inline double node_value(const NodeSrc &s, int ir, int c) {
  const float *a1 = s.a1, *a2 = s.a2;
  const float *arr = (c & 1) ? a2 : a1;
  const size_t q = (size_t)ir * s.ng + (c >> 1);
  return lerp2f(s.fa, s.fm, arr[s.s00 + q], arr[s.s10 + q], arr[s.s01 + q], arr[s.s11 + q]);
}

// Node rows kb .. kb + tot / nq - 1 (nq = 2 n_g values each, contiguous) built
// into LDS by the whole wavefront: every lane loads the four corners of PER
// values per round (4 PER loads in flight), then interpolates them; at most
// STAGE_MAX values.
constexpr int STAGE_MAX = 640;
template <int PER>
__device__ inline void stage_table_rows(const NodeSrc &s, int kb, int tot, int nq, double *dst, int lane) {
  int row = kb + lane / nq, col = lane % nq;
  const float *a1 = s.a1, *a2 = s.a2;
  for (int k0 = 0; k0 < STAGE_MAX / 64 && 64 * k0 < tot; k0 += PER) {
    float c00[PER], c10[PER], c01[PER], c11[PER];
#pragma unroll
    for (int k = 0; k < PER; k++) {
      if (lane + 64 * (k0 + k) < tot) {
        const float *arr = (col & 1) ? a2 : a1;
        const size_t q = (size_t)row * s.ng + (col >> 1);
        c00[k] = arr[s.s00 + q];
        c10[k] = arr[s.s10 + q];
        c01[k] = arr[s.s01 + q];
        c11[k] = arr[s.s11 + q];
      }
      col += 64;
      while (col >= nq) {
        col -= nq;
        row++;
      }
    }
#pragma unroll
    for (int k = 0; k < PER; k++) {
      const int idx = lane + 64 * (k0 + k);
      if (idx < tot) dst[idx] = lerp2f(s.fa, s.fm, c00[k], c10[k], c01[k], c11[k]);
    }
  }
}

// k_fixup: an entry's FP64 row values, straight from the table, for the g*
// brackets that the FP64 integral of the bin [e0, e1] reads (its points lie
// between the bin's clamped ends, whose brackets bound theirs; one bracket of
// margin either side) and for the brackets of the two edge norms; the other
// columns of the row are not read.  Lane l of the entry's FIX_LANES takes every
// FIX_LANES-th column.
constexpr int FIX_LANES = 8;
__device__ inline void load_radius_table(const BatchDev &b, const ReqNorm &rn, const RadGeo &r, int K, int limb,
                                         double e0, double e1, double *myT, double *myC, RadiusView &v, int l) {
  v.gmin = r.gmin;
  v.gmax = r.gmax;
  v.del_g = 1. / (r.gmax - r.gmin);  // set_str_relbf, src/Relprofile.cpp:733
  v.limb = limb;
  const int ng = b.rt.n_g;
  auto bracket = [&](double e) {
    const double g = fmin(fmax((e - v.gmin) * v.del_g, GFAC_H), 1.0 - GFAC_H);
    return g_bracket(g, ng, v.gs_step, v.inv_step);
  };
  const NodeSrc ts = node_src(b.rt, rn, false);
  const NodeSrc cs = node_src(b.rt, rn, true);
  auto put = [&](int c) {
    myT[c] = lerp1_(r.ifac_r, node_value(ts, K + 1, c), node_value(ts, K, c));
    if (limb) myC[c] = lerp1_(r.ifac_r, node_value(cs, K + 1, c), node_value(cs, K, c));
  };
  const int ia = max(0, bracket(e0) - 1), ib = min(ng - 2, bracket(e1) + 1);
#pragma unroll 4
  for (int c = 2 * ia + l; c <= 2 * ib + 3; c += FIX_LANES) put(c);
  // four columns of each edge bracket
  static_assert(FIX_LANES == 8, "a lane per column of the two edge brackets");
  put(2 * edge_point(l >= 4, v).ind + (l & 3));
}

__device__ inline const double *profile_grid(const BatchDev &b, const ReqParams *rq) {
  const int64_t off = rq->pgrid_off;
  return (off >= 0) ? b.pgrid + off : b.cg.ener;
}

// The bin edges of a work item in turn: one scalar load a bin ahead, or (ONE) the
// edges of SUM_BINS bins per load, a group ahead.
template <int ONE>
struct EdgeWalk {
  const double *E;
  double first, next, grp;
  __device__ void start(const double *grid, const WorkItem &it, int lane) {
    E = grid;
    first = E[it.j0];
    next = E[min(it.j0 + 1 + (ONE ? lane : 0), it.j1)];
  }
  __device__ void group(const WorkItem &it, int jg, int lane) {  // bins [jg, jg + SUM_BINS)
    if constexpr (ONE) {
      grp = next;  // lane l: the upper edge of the group's bin l
      next = E[min(jg + SUM_BINS + 1 + lane, it.j1)];
    }
  }
  __device__ double upper(const WorkItem &it, int j, int jj) {  // of bin j, jj-th of its group
    if constexpr (ONE) return readlane_d(grp, jj);
    const double e = next;
    next = E[min(j + 2, it.j1)];
    return e;
  }
};

}  // namespace

// Emission-angle distribution of the requests with one (src/Relprofile.cpp:
// 908-938), one wavefront per (request, chunk of 64 fine radii), after k_setup.
// Lane = fine radius; the node rows of the chunk's radii (transfer function
// and cosines) are built in LDS from the table corners, DIST_STAGE values of
// each at a time, and each lane walks the g* columns, both branches of a
// column at once (16-byte LDS reads).  Neighbouring columns mostly fall into
// one angle bin, so a lane sums in a register while its bin stays and adds to
// the LDS bins when it changes; the wavefront's last bins go as one wave sum
// when all lanes share the bin.  By itself (k_dist) or as workgroups of
// k_integrate.
// The chunk's sums are added to the request's distribution in HBM (cleared by
// k_setup, left unnormalised: its readers scale by its sum).
// Bound: FP64 issue, 1000 radii x 2 n_g columns x ~60 operations a request,
// which one CU takes 16 us for: inside k_setup (one workgroup a request) it
// was 61 us of a single relxill call (k_setup 87 us) and 165 us of a batch of
// 1024 (237 us); the 16 wavefronts a request take 12 us and 70 us (92 us with
// staging areas of 640 values, which halved the wavefronts per CU).
constexpr int DIST_STAGE = 320;  // staged values of each of the two arrays (2 rows of 2 MAX_NG at least)
__host__ __device__ constexpr int dist_lds(int n_zones) {  // doubles
  return 2 * DIST_STAGE + 2 * MAX_NG + n_zones * MAX_INCL;
}
__device__ __forceinline__ void dist_chunk(const BatchDev &b, int req, int c, int lane, double *lds) {
  double *s_t = lds, *s_c = lds + DIST_STAGE;
  double2 *s_g = reinterpret_cast<double2 *>(lds + 2 * DIST_STAGE);
  double *s_dist = lds + 2 * DIST_STAGE + 2 * MAX_NG;  // [zone][angle bin]
  if (b.status[req] != 0) return;  // uniform over the block
  const ReqParams &rq = b.req[req];
  const ReqNorm rn = b.rnorm[req];
  const int n_incl = rq.n_incl, ng = b.rt.n_g, nr = b.nr_fine, nq = 2 * ng;
  const int ii = c * RAD_CHUNK + lane;
  RadRec rec = rad_pack(0.0, 0, 0, 1, 0);
  if (ii < nr) rec = b.rad[(size_t)req * nr + ii];
  const bool live = ii < nr && rad_ielo(rec) <= rad_iehi(rec);
  if (__ballot(live) == 0) return;
  const int K = rad_K(rec), zone = rad_zone(rec);
  double amp = 0.0;  // re (2 pi re)^2 emis weight: what a radius' columns share
  RadGeo r = {0.0, 0.0, 0.0};
  if (live) {
    const double *gn = b.rnode + (size_t)req * RAD_NODE_ARRAYS * b.rt.n_r;
    const double re = fine_radius_at(rn.r1, rn.r2, ii, nr);
    r = rad_geo(gn, gn + b.rt.n_r, gn + 2 * b.rt.n_r, re, K);
    const double pr = 2 * PI * re;
    amp = re * (pr * pr) * (rec.coef * (r.gmax - r.gmin) * rn.fac);
  }
  const int zlo = wave_min_i(live ? zone : INT_MAX), zhi = wave_max_i(live ? zone : -1);
  for (int k = zlo * n_incl + lane; k < (zhi + 1) * n_incl; k += 64) s_dist[k] = 0.0;
  // per g*: the node value and d_gstar / sqrt(g* (1 - g*))
  const double step = (1.0 - 2 * GFAC_H) / (ng - 1);
  const double gs0 = gstar_node(step, 0), gs1 = gstar_node(step, 1);
  for (int g = lane; g < ng; g += 64) {
    const double gs = gstar_node(step, g);
    const double dgs = (g == 0 || g == ng - 1) ? 0.5 * (gs1 - gs0) + GFAC_H : gs1 - gs0;
    s_g[g] = make_double2(gs, dgs / sqrt(gs - gs * gs));
  }
  const int kmin = wave_min_i(live ? K : INT_MAX), kmax = wave_max_i(live ? K : -1);
  const NodeSrc ts = node_src(b.rt, rn, false), cs = node_src(b.rt, rn, true);
  const int stage_rows = DIST_STAGE / nq;  // at least 2 (n_g <= MAX_NG)
  int derr = 0;
  auto put = [&](int k, double sum) {  // one lane's sum over columns of angle bin k
    const double v = sum * amp;
    if (v != v) derr = max(derr, 41);
    else atomicAdd(&s_dist[zone * n_incl + k], v);
  };
  for (int kb = kmin; kb <= kmax; kb += stage_rows - 1) {
    const int ke = min(kmax, kb + stage_rows - 2);
    const int tot = (ke - kb + 2) * nq;
    stage_table_rows<5>(ts, kb, tot, nq, s_t, lane);
    stage_table_rows<5>(cs, kb, tot, nq, s_c, lane);
    __syncthreads();
    const bool mine = live && K >= kb && K <= ke;
    const int olo = (mine ? K + 1 - kb : 0) * nq, ohi = (mine ? K - kb : 0) * nq;
    const double2 *tlo = reinterpret_cast<const double2 *>(s_t + olo), *thi = reinterpret_cast<const double2 *>(s_t + ohi);
    const double2 *clo = reinterpret_cast<const double2 *>(s_c + olo), *chi = reinterpret_cast<const double2 *>(s_c + ohi);
    int cur[2] = {-1, -1};
    double acc[2] = {0.0, 0.0};
    for (int g = 0; g < ng; g++) {
      const double2 t0 = tlo[g], t1 = thi[g], c0 = clo[g], c1 = chi[g], gg = s_g[g];
      const double trff[2] = {lerp1(r.ifac_r, t0.x, t1.x), lerp1(r.ifac_r, t0.y, t1.y)};
      const double cosne[2] = {lerp1(r.ifac_r, c0.x, c1.x), lerp1(r.ifac_r, c0.y, c1.y)};
      const double gv = gg.x * (r.gmax - r.gmin) + r.gmin;
      const double gw = gv * gv * gg.y;
#pragma unroll
      for (int br = 0; br < 2; br++) {
        const int imu = ((int)(n_incl * (1 - cosne[br]) + 1)) - 1;
        if (!mine) continue;
        if (imu < 0 || imu >= n_incl) {
          derr = 40;
          continue;
        }
        if (imu != cur[br]) {
          if (cur[br] >= 0) put(cur[br], acc[br]);
          cur[br] = imu;
          acc[br] = 0.0;
        }
        acc[br] += gw * trff[br];
      }
    }
#pragma unroll
    for (int br = 0; br < 2; br++) {
      const int bin = cur[br] >= 0 ? zone * n_incl + cur[br] : -1;
      const unsigned long long m_ok = __ballot(bin >= 0);
      if (m_ok == 0) continue;
      const int first = __ffsll((long long)m_ok) - 1;
      const int k0 = __builtin_amdgcn_readlane(bin, first);
      if (__ballot(bin >= 0 && bin != k0) == 0) {
        const double v = bin >= 0 ? acc[br] * amp : 0.0;
        if (v != v) derr = max(derr, 41);
        const double sum = wave_sum(v);
        if (lane == first) atomicAdd(&s_dist[k0], sum);
      } else if (bin >= 0) {
        put(cur[br], acc[br]);
      }
    }
    __syncthreads();  // the next rows overwrite the staged ones
  }
  derr = wave_max_i(derr);
  if (derr && lane == 0) atomicMax(&b.status[req], derr);
  __syncthreads();
  for (int k = zlo * n_incl + lane; k < (zhi + 1) * n_incl; k += 64)
    if (s_dist[k] != 0.0) unsafeAtomicAdd(&b.dist[rq.dist_off + k], s_dist[k]);
}

__global__ __launch_bounds__(64) void k_dist(BatchDev b, const int *__restrict__ reqs, int n_rc) {
  extern __shared__ __align__(16) double s_lds[];
  dist_chunk(b, reqs[blockIdx.x / n_rc], blockIdx.x % n_rc, threadIdx.x, s_lds);
}

// Byte offset of k_integrate's coefficient slots and bin buffer (FP64 path)
// behind the lane rows (rows: 64 or 128 of 2 n_g + 1 values).
__host__ __device__ inline size_t integrate_rows_bytes(int ng, bool cos_rows, size_t elem) {
  const size_t b = (size_t)(cos_rows ? 2 : 1) * 64 * (2 * ng + 1) * elem;
  return (b + 15) & ~(size_t)15;
}

// Persistent wavefronts pull work items (request, chunk of 64 fine radii, bin
// segment) from the per-XCD ranges of the work list until every range is
// exhausted.  Lane l owns
// fine radius 64 rc + l: its transfer-function row sits in LDS and its window,
// weight and edge norms in registers.  For every bin of the segment each lane
// integrates the bin at its radius (zero outside its window) and parks the
// value in LDS; every SUM_BINS bins the wavefront turns round: 8 lanes per bin
// each sum 8 radii in FP64 (fixed order), a 3-step DPP tree adds the 8 partial
// sums and one lane per bin adds the result to the request's profile with one
// FP64 atomic.
//   MODE 0 (FP64): the parked values are the FP64 bin integrals; the
//   turn-round multiplies them by the radii's weights (64 slots in LDS).
//   MODE 1 (FP32 integrand, FP64 decisions and edges): each lane parks its
//   integral times its weight times the request's power of two
//   (ReqNorm.cmul) as FP32, and the atomic adds the sum times ReqNorm.cinv.
//   Bins whose Romberg stop test fell in the guard band are queued for the
//   FP64 re-check (k_fixup).
//   Item set-up: the node rows that the chunk's radii lerp between (nodes
//   kmin .. kmax + 1) are built in LDS from the table's four (a, mu0)
//   corners by the whole wavefront, stage_rows at a time, in one round of
//   loads each; each lane then lerps its row and the FP64 values of its edge
//   norms from LDS.  The staging area is the parked-value area, which is free
//   between items.
//   COS: the batch holds emission-angle rows (a request with limb
//   darkening); COS == 0 compiles the limb factors out.
//   ONE: one workgroup per item of the list's capacity, and no hand-out: for
//   short lists, where a wavefront takes one item anyway and the walk over the
//   range counters (one atomic each, 8 when it finds them all empty) would be a
//   third of the kernel's time.  It also loads an item's edges a group ahead.
//   A single relconv call (segments of 4 bins): 34 us with the counters, 22 us
//   without (FP32 36 and 15 us); with the segments of 64 bins that every batch
//   had by default 64 us (43 us).
//   ONE also takes the angle distribution's chunks and, where nothing before
//   reads them, the zone records along as its first workgroups (side): they and
//   the items need nothing of each other and leave the chip idle between them.
//   As launches of their own they were 12 us and 5-17 us of every relxill call
//   (relxill 120 us, 109 us with them here; 128 relxilllp requests 566 us, 554 us).
template <int MODE, int COS, int ONE>
__global__ __launch_bounds__(64, MODE == 0 ? 1 : 3) void k_integrate(BatchDev b_arg, int stage_rows, SideWork side) {
  // The argument is read through a pointer that every item renews, so that the
  // compiler reads its fields where an item uses them: kept across the item
  // loop they took 28 scalar registers more than there are, spilled to vector
  // lanes and read back for every bin (4096 relconv requests: 1259 us, 1250 us
  // without the spills, FP64 3700 us and 3535 us).
  typedef const __attribute__((address_space(4))) BatchDev KArg;
  KArg *bp = (KArg *)__builtin_amdgcn_kernarg_segment_ptr();
  const BatchDev &b = *(const BatchDev *)bp;
  constexpr int cos_rows = COS;
  using TV = typename std::conditional<MODE == 0, double, float>::type;
  extern __shared__ __align__(16) double s_dyn[];
  const int lane = threadIdx.x;
  int one_item = blockIdx.x;
  if constexpr (ONE) {
    const int n_chunk = side.n_ang * side.n_rc;
    if (one_item < n_chunk) {
      dist_chunk(b, side.ang[one_item / side.n_rc], one_item % side.n_rc, lane, s_dyn);
      return;
    }
    one_item -= n_chunk;
    if (one_item < side.n_zone) {
      zone_unit(b, side.zone[one_item], lane, 64, s_dyn);
      return;
    }
    one_item -= side.n_zone;
  }
  const int ng = b.rt.n_g;
  const int RS = 2 * ng + 1;  // odd row stride: lanes' rows start in distinct banks
  TV *rows = reinterpret_cast<TV *>(s_dyn);
  TV *myT = rows + lane * RS;
  TV *myC = cos_rows ? rows + (64 + lane) * RS : myT;
  // behind the rows: MODE 0 the 64 weights then the parked doubles, MODE 1 the parked floats
  double *s_coef = reinterpret_cast<double *>(reinterpret_cast<char *>(s_dyn) +
                                              integrate_rows_bytes(ng, cos_rows != 0, sizeof(TV)));
  TV *s_bins = (MODE == 0) ? reinterpret_cast<TV *>(s_coef + 64) : reinterpret_cast<TV *>(s_coef);
  // long items at [0, n_long), short ones at the back of the list
  const int asked = b.ctr[CTR_ITEMS], asked_s = b.ctr[CTR_ITEMS_S], fit = b.ctr[CTR_FIT], fit_s = b.ctr[CTR_FIT_S];
  const bool ovf = b.ctr[CTR_ITEMS_OVF] != 0;
  const int n_long = ovf ? fit : asked, n_short = ovf ? fit_s : asked_s;
  const int nr = b.nr_fine;
  // turn-round roles: SUM_LANES lanes per bin; lane (col, part) sums radii
  // SUM_BINS part .. SUM_BINS part + SUM_BINS - 1 of bin col
  constexpr int SUM_LANES = 64 / SUM_BINS;
  const int col = lane / SUM_LANES, part = lane % SUM_LANES;
  RadiusView v;
  v.ng = ng;
  v.gs_step = (1.0 - 2 * GFAC_H) / (ng - 1);
  v.inv_step = 1.0 / v.gs_step;
  v.guard = b.guard;
  v.T64 = nullptr;
  v.C64 = nullptr;
  v.T32 = nullptr;
  v.C32 = nullptr;
  v.limb = 0;
  if (MODE == 0) {
    v.T64 = reinterpret_cast<const double *>(myT);
    v.C64 = reinterpret_cast<const double *>(myC);
  } else {
    v.T32 = reinterpret_cast<const float *>(myT);
    v.C32 = reinterpret_cast<const float *>(myC);
  }
  int xq = blockIdx.x % N_XQ, exhausted = 0;
  for (;;) {
    // next item of range xq (its share of the long items, then its share of
    // the short ones); an empty range sends the wavefront to the next one,
    // and once all N_XQ have been found empty it is done
    int k = -1;
    if constexpr (ONE) {
      const int kk = one_item;
      if (kk >= n_long + n_short) return;
      k = kk < n_long ? kk : b.item_cap - 1 - (kk - n_long);
    }
    while (!ONE && exhausted < N_XQ) {
      const int lo = (int)((int64_t)n_long * xq / N_XQ), hi = (int)((int64_t)n_long * (xq + 1) / N_XQ);
      const int los = (int)((int64_t)n_short * xq / N_XQ), his = (int)((int64_t)n_short * (xq + 1) / N_XQ);
      int kk = 0;
      if (lane == 0) kk = atomicAdd(&b.ctr[CTR_XQ + xq * XQ_STRIDE], 1);
      kk = __builtin_amdgcn_readfirstlane(kk);
      if (kk < hi - lo) {
        k = lo + kk;
        break;
      }
      if (kk < (hi - lo) + (his - los)) {
        k = b.item_cap - 1 - (los + kk - (hi - lo));
        break;
      }
      exhausted++;
      xq = (xq + 1) % N_XQ;
    }
    if (k < 0) break;
    if constexpr (!ONE) asm volatile("" : "+s"(bp));
    const BatchDev &b = *(const BatchDev *)bp;
    const WorkItem it = b.items[k];
    const ReqParams *rq = b.req + it.req;
    const ReqNorm rn = b.rnorm[it.req];
    const int limb = COS ? rq->limb : 0;
    const int i = (it.rc & 0xffff) * RAD_CHUNK + lane;
    const int zone = it.rc >> 16;
    // the lane's radius: the stored record, and its geometry rebuilt from the
    // request's node arrays
    int rK = 0, ielo = 1, iehi = 0;
    double coef = 0.0;
    if (i < nr) {
      const RadRec pr = b.rad[(size_t)it.req * nr + i];
      if (rad_zone(pr) == zone) {  // (else a radius of another zone of the chunk)
        ielo = rad_ielo(pr);
        iehi = rad_iehi(pr);
      }
      rK = rad_K(pr);
      coef = pr.coef;
    }
    EdgeWalk<ONE> ew;
    if constexpr (ONE) ew.start(profile_grid(b, rq), it, lane);
    const bool has_win = ielo <= iehi;
    RadGeo r = {0.0, 0.0, 0.0};
    if (has_win) {
      const double *gn = b.rnode + (size_t)it.req * RAD_NODE_ARRAYS * b.rt.n_r;
      r = rad_geo(gn, gn + b.rt.n_r, gn + 2 * b.rt.n_r, fine_radius_at(rn.r1, rn.r2, i, nr), rK);
    }
    const int kmin = wave_min_i(has_win ? rK : INT_MAX);
    const int kmax = wave_max_i(has_win ? rK : -1);
    if (kmax >= 0) {
      // the lanes' rows from node rows kb .. ke + 1 built in LDS, stage_rows
      // at a time (lanes with K in [kb, ke] are served per round), for the
      // transfer function and then (limb) the cosines; the FP64 values at the
      // edge brackets are kept for the edge norms
      const int nq = 2 * ng;
      double *stage = reinterpret_cast<double *>(s_bins);
      const NodeSrc ts = node_src(b.rt, rn, false);
      const NodeSrc cs = node_src(b.rt, rn, true);
      EdgePt pL{}, pU{};
      if (has_win) {
        v.gmin = r.gmin;
        v.gmax = r.gmax;
        v.del_g = 1. / (r.gmax - r.gmin);  // set_str_relbf, src/Relprofile.cpp:733
        v.limb = limb;
        pL = edge_point(false, v);
        pU = edge_point(true, v);
      }
      for (int kb = kmin; kb <= kmax; kb += stage_rows - 1) {
        double tL[4] = {0, 0, 0, 0}, tU[4] = {0, 0, 0, 0}, cL[4] = {0, 0, 0, 0}, cU[4] = {0, 0, 0, 0};
        const int ke = min(kmax, kb + stage_rows - 2);
        const bool mine = has_win && rK >= kb && rK <= ke;
        const int tot = (ke - kb + 2) * nq;
        const int klo = mine ? rK + 1 - kb : 1, khi = mine ? rK - kb : 0;
        const double *lo = stage + (size_t)klo * nq;
        const double *hi = stage + (size_t)khi * nq;
        stage_table_rows<5>(ts, kb, tot, nq, stage, lane);
        __syncthreads();  // one wavefront: orders the staged rows before the lanes read them
        if (mine) {
          lerp_row<TV>(r.ifac_r, lo, hi, nq, myT);
#pragma unroll
          for (int k = 0; k < 4; k++) {
            tL[k] = lerp1_(r.ifac_r, lo[pL.ind * 2 + k], hi[pL.ind * 2 + k]);
            tU[k] = lerp1_(r.ifac_r, lo[pU.ind * 2 + k], hi[pU.ind * 2 + k]);
          }
        }
        __syncthreads();  // the next rows (or the bins) overwrite the staging area
        if (COS && limb) {
          stage_table_rows<5>(cs, kb, tot, nq, stage, lane);
          __syncthreads();
          if (mine) {
            lerp_row<TV>(r.ifac_r, lo, hi, nq, myC);
#pragma unroll
            for (int k = 0; k < 4; k++) {
              cL[k] = lerp1_(r.ifac_r, lo[pL.ind * 2 + k], hi[pL.ind * 2 + k]);
              cU[k] = lerp1_(r.ifac_r, lo[pU.ind * 2 + k], hi[pU.ind * 2 + k]);
            }
          }
          __syncthreads();
        }
        if (mine) {
          v.normL = edge_norm_at(pL, v, tL, cL);
          v.normU = edge_norm_at(pU, v, tU, cU);
          v.eL = (float)(2 * v.normL * (v.gmax - v.gmin));
          v.eU = (float)(2 * v.normU * (v.gmax - v.gmin));
        }
      }
    }
    const double w64 = has_win ? coef * rn.fac : 0.0;   // MODE 0 weight
    const double w32 = has_win ? coef * rn.cmul : 0.0;  // MODE 1 scaled weight
    const float w32f = (float)w32;
    if constexpr (MODE == 0) s_coef[lane] = w64;
    if constexpr (!ONE) ew.start(profile_grid(b, rq), it, lane);
    double *acc = profile_acc(b, *rq) + (size_t)zone * rq->n_e;
    double ehi = ew.first;
    double ghi = (ehi - v.gmin) * v.del_g;  // unclamped g* of the bin's upper edge, carried
    EdgePair<TV> cy;  // integrand pair at the next bin's lower edge, when a Romberg bin left it
    cy.ok = false;
    for (int jg = it.j0; jg < it.j1; jg += SUM_BINS) {
      const int jn = min(SUM_BINS, it.j1 - jg);
      ew.group(it, jg, lane);
      for (int jj = 0; jj < jn; jj++) {
        const int j = jg + jj;
        const double elo = ehi, glo = ghi;
        ehi = ew.upper(it, j, jj);
        ghi = (ehi - v.gmin) * v.del_g;
        TV val = 0;
        if (j >= ielo && j <= iehi) {
          if constexpr (MODE == 0) {
            val = integ_bin_g<0>(elo, ehi, glo, ghi, v, nullptr, &cy);
          } else {
            bool need64 = false;
            val = integ_bin32(elo, ehi, glo, ghi, v, &need64, &cy) * w32f;
            if (need64) {
              const int slot = atomicAdd(&b.ctr[CTR_FIX], 1);
              if (slot < b.fix_cap) {
                FixEntry fe;
                fe.req = it.req;
                fe.rad = i;
                fe.bin = j;
                fe.pad = 0;
                fe.v32 = (double)val * rn.cinv;  // this radius' share of the bin's atomic
                b.fix[slot] = fe;
              } else {
                atomicOr(&b.ctr[CTR_FIX_OVF], 1);
              }
            }
          }
        } else {
          cy.ok = false;
        }
        s_bins[jj * SUM_STRIDE + lane] = val;
      }
      __syncthreads();  // one wavefront: orders the parked values before the turn-round
      // FP64 sum over the 64 radii of bin jg + col: SUM_BINS radii per lane,
      // then the SUM_LANES lanes of the bin in a fixed DPP tree
      const TV *src = s_bins + col * SUM_STRIDE + part * SUM_BINS;
      double sum = 0.0;
      if constexpr (MODE == 0) {
        const double *cf = s_coef + part * SUM_BINS;
#pragma unroll
        for (int q = 0; q < SUM_BINS; q++) sum = fma(src[q], cf[q], sum);
      } else {
#pragma unroll
        for (int q = 0; q < SUM_BINS; q++) sum += (double)src[q];
      }
      sum += dpp_d<0xB1>(sum);   // quad_perm [1,0,3,2]
      sum += dpp_d<0x4E>(sum);   // quad_perm [2,3,0,1]
      sum += dpp_d<0x141>(sum);  // row_half_mirror: every lane of a half row holds its sum
      if constexpr (SUM_LANES == 16) sum += dpp_d<0x140>(sum);  // row_mirror: the whole row
      if (MODE == 1) sum *= rn.cinv;
      if (part == 0 && col < jn) unsafeAtomicAdd(&acc[jg + col], sum);
      __syncthreads();  // the next bins overwrite the parked values
    }
    if constexpr (ONE) return;
  }
}

// FP64 re-check of guarded FP32 bins, FIX_LANES lanes an entry, the entries
// spread over the workgroups.  Bound: latency, of the entry's records, its table
// columns and its integral.  One lane an entry read up to 2 n_g columns in turn,
// 8 corner loads each, in wavefronts of 64 neighbouring entries: 1 entry 6.5 us,
// 577 entries 19 us, 3017 wide bins of convolutions 30 us, 12354 30 us; with the
// columns over the lanes 3.5 us, 8.5 us, 17 us and 20 us (26 us with 1024
// workgroups).
__global__ __launch_bounds__(64) void k_fixup(BatchDev b, int cos_rows) {
  extern __shared__ __align__(16) double s_dyn[];
  constexpr int PER = 64 / FIX_LANES;  // entries per wavefront
  const int sub = threadIdx.x / FIX_LANES, l = threadIdx.x % FIX_LANES;
  const int ng = b.rt.n_g;
  const int RS = 2 * ng + 1;
  double *myT = s_dyn + sub * RS;
  double *myC = cos_rows ? s_dyn + (PER + sub) * RS : myT;
  const int n = min(b.ctr[CTR_FIX], b.fix_cap);
  RadiusView v;
  v.ng = ng;
  v.gs_step = (1.0 - 2 * GFAC_H) / (ng - 1);
  v.inv_step = 1.0 / v.gs_step;
  v.guard = b.guard;
  v.T64 = myT;
  v.C64 = myC;
  v.T32 = nullptr;
  v.C32 = nullptr;
  for (int e0 = blockIdx.x; e0 < n; e0 += gridDim.x * PER) {  // (uniform: the barriers are met by all)
    const int e = e0 + sub * gridDim.x;
    const bool live = e < n;
    const FixEntry fe = b.fix[live ? e : e0];
    const ReqParams *rq = b.req + fe.req;
    const RadRec pr = b.rad[(size_t)fe.req * b.nr_fine + fe.rad];
    const double *gn = b.rnode + (size_t)fe.req * RAD_NODE_ARRAYS * b.rt.n_r;
    const ReqNorm &rn = b.rnorm[fe.req];
    const double *E = profile_grid(b, rq);
    const double elo = E[fe.bin], ehi = E[fe.bin + 1];
    const RadGeo r = rad_geo(gn, gn + b.rt.n_r, gn + 2 * b.rt.n_r, fine_radius_at(rn.r1, rn.r2, fe.rad, b.nr_fine),
                             rad_K(pr));
    load_radius_table(b, rn, r, rad_K(pr), rq->limb, elo, ehi, myT, myC, v, l);
    __syncthreads();  // one wavefront: the entry's columns before its lanes read them
    v.normL = edge_norm64(false, v);
    v.normU = edge_norm64(true, v);
    const double val = integ_bin<0>(elo, ehi, v) * (pr.coef * rn.fac);
    if (live && l == 0)
      unsafeAtomicAdd(&profile_acc(b, *rq)[(size_t)rad_zone(pr) * rq->n_e + fe.bin], val - fe.v32);
    __syncthreads();  // the next entry's columns overwrite them
  }
}

// ---------------------------------------------------------------------------
// finalize: renormalisation (renorm_relline_profile, src/Relprofile.cpp:749-796)
// ---------------------------------------------------------------------------
// Line models only: a convolution's profile and angle distribution are sums that
// their readers (k_conv, k_xill) scale themselves, each by one factor.  While
// the distributions were normalised here, ten zones' block sums one after the
// other took 12-14 us of a relxilllp call, one zone's 4.6 us.
__global__ __launch_bounds__(FINAL_THREADS) void k_finalize(BatchDev b, Deliver dl) {
  __shared__ double s_red[FINAL_THREADS];
  const int req = blockIdx.x;
  const int tid = threadIdx.x;
  const ReqParams &rq = b.req[req];
  if (rq.prof_off >= 0 || rq.model == MOD_XILLVER) return;
  const int n_e = rq.n_e;
  double *dst = profile_acc(b, rq);
  double *host = dl.out ? dl.out + rq.flux_off : nullptr;
  deliver_words(b, dl, req, tid);
  const int st = b.status[req];
  if (st != 0) {
    for (int j = tid; j < n_e; j += FINAL_THREADS) {
      dst[j] = 0.0;
      if (host) host[j] = 0.0;
    }
    return;
  }
  const double *E = b.pgrid + rq.pgrid_off;
  const BinRange rc = b.reach[req];
  double loc = 0.0;
  for (int j = tid; j < n_e; j += FINAL_THREADS) {
    double v = 0.0;
    if (j >= rc.lo && j <= rc.hi) v = dst[j] / (0.5 * (E[j] + E[j + 1]));
    dst[j] = v;
    if (host && !rq.do_renorm) host[j] = v;
    loc += v;
  }
  const double sum = block_sum(loc, s_red);
  if (rq.do_renorm) {
    const double f = rq.norm / sum;
    for (int j = tid; j < n_e; j += FINAL_THREADS) {
      const double v = dst[j] * f;
      dst[j] = v;
      if (host) host[j] = v;
    }
  }
}

// ---------------------------------------------------------------------------
// convolution
// ---------------------------------------------------------------------------
namespace {

// LDS index of complex element i: one pad slot every 16 elements, so that the
// strided writes of the passes spread over the banks.
__device__ inline int P(int i) { return i + (i >> 4); }

__device__ inline double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ inline double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ inline double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
// a * (S i), S = -1 (forward) or +1 (inverse)
template <int S>
__device__ inline double2 mul_si(double2 a) {
  return S > 0 ? make_double2(-a.y, a.x) : make_double2(a.y, -a.x);
}

// exp(S 2 pi i M / 16), M known at compile time
template <int S, int M>
__device__ inline double2 w16() {
  constexpr double c[5] = {1.0, 0.92387953251128675613, 0.70710678118654752440, 0.38268343236508977173, 0.0};
  constexpr int q = (M & 15) >> 2, r = M & 3;
  constexpr double cs = q == 0 ? c[r] : q == 1 ? -c[4 - r] : q == 2 ? -c[r] : c[4 - r];
  constexpr double sn = q == 0 ? c[4 - r] : q == 1 ? c[r] : q == 2 ? -c[4 - r] : -c[r];
  return make_double2(cs, S * sn);
}

template <int S>
__device__ __forceinline__ void dft4(double2 &a0, double2 &a1, double2 &a2, double2 &a3) {
  const double2 s02 = cadd(a0, a2), d02 = csub(a0, a2);
  const double2 s13 = cadd(a1, a3), d13 = mul_si<S>(csub(a1, a3));
  a0 = cadd(s02, s13);
  a2 = csub(s02, s13);
  a1 = cadd(d02, d13);
  a3 = csub(d02, d13);
}

template <int S, int N2, int K1>
__device__ inline void tw16(double2 &x) {
  if (N2 * K1 != 0) x = cmul(x, w16<S, N2 * K1>());
}

// In-register DFT of length R (2, 4 or 8), natural order in and out.
template <int R, int S>
__device__ __forceinline__ void dft(double2 *v) {
  if (R == 2) {
    const double2 t = v[0];
    v[0] = cadd(t, v[1]);
    v[1] = csub(t, v[1]);
  } else if (R == 4) {
    dft4<S>(v[0], v[1], v[2], v[3]);
  } else {
    static_assert(R == 2 || R == 4 || R == 8, "the passes' radices");
    // n = 2 n1 + n2, k = k1 + 4 k2: two DFT4 (even, odd), twiddle, butterflies
    dft4<S>(v[0], v[2], v[4], v[6]);
    dft4<S>(v[1], v[3], v[5], v[7]);
    tw16<S, 1, 2>(v[3]);
    tw16<S, 1, 4>(v[5]);
    tw16<S, 1, 6>(v[7]);
    const double2 e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
    const double2 o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
    v[0] = cadd(e0, o0);
    v[4] = csub(e0, o0);
    v[1] = cadd(e1, o1);
    v[5] = csub(e1, o1);
    v[2] = cadd(e2, o2);
    v[6] = csub(e2, o2);
    v[3] = cadd(e3, o3);
    v[7] = csub(e3, o3);
  }
}

// The twiddles of this thread's first value in a radix-R pass (at most 7).
__device__ __forceinline__ void load_twiddles(double2 *w, int R, int N, int Ns, const double2 *twp) {
  const int j = threadIdx.x;
  if (j >= N / R) return;
  const int k = j & (Ns - 1);
#pragma unroll
  for (int r = 1; r < 8; r++)
    if (r < R) w[r - 1] = twp[r * Ns + k];
}

// Radix of the pass with N / Ns left.
__device__ __forceinline__ int fft_radix(int left) { return left % 8 == 0 ? 8 : left % 4 == 0 ? 4 : 2; }

// One Stockham radix-R pass over N complex values in LDS (padded layout):
// thread j loads x[j + r N/R] r = 0..R-1, twiddles by w^(r (j mod Ns)),
// w = exp(S 2 pi i / (Ns R)) (table twp[r Ns + k], forward sign, conjugated
// for S = +1), transforms, and stores at (j / Ns) Ns R + j mod Ns + r Ns.
// PER j values per thread; reads finish before any write.  w holds the first
// j's twiddles, and receives the next pass' before the barriers, so that their
// reads (L2) are in flight meanwhile (1 unit 30.8 us and 29.6 us, 256 units 46 us
// and 41 us, 4096 units 350 us and 342 us).
template <int R, int S, int PER>
__device__ __forceinline__ void fft_pass(double2 *buf, int N, int Ns, const double2 *twp, double2 *w) {
  const int J = N / R;
  double2 v[PER][R];
  const int lgNs = __ffs(Ns) - 1;  // Ns is a power of two
#pragma unroll
  for (int u = 0; u < PER; u++) {
    const int j = threadIdx.x + u * blockDim.x;
    if (j < J) {
      const int k = j & (Ns - 1);
#pragma unroll
      for (int r = 0; r < R; r++) {
        double2 x = buf[P(j + r * J)];
        if (r > 0) {
          double2 t = u == 0 ? w[r - 1] : twp[r * Ns + k];
          if (S > 0) t.y = -t.y;
          x = cmul(x, t);
        }
        v[u][r] = x;
      }
      dft<R, S>(v[u]);
    }
  }
  if (Ns * R < N) load_twiddles(w, fft_radix(N / (Ns * R)), N, Ns * R, twp + R * Ns);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < PER; u++) {
    const int j = threadIdx.x + u * blockDim.x;
    if (j < J) {
      const int k = j & (Ns - 1);
      const int base = ((j >> lgNs) << lgNs) * R + k;
#pragma unroll
      for (int r = 0; r < R; r++) buf[P(base + r * Ns)] = v[u][r];
    }
  }
  __syncthreads();
}

// The block has at least N/8 threads, so a pass holds at most 8 values per
// thread: PER = 1 (R = 8), <= 2 (R = 4), <= 4 (R = 2).
template <int R, int S>
__device__ __forceinline__ void fft_pass_any(double2 *buf, int N, int Ns, const double2 *twp, double2 *w) {
  const int per = (N / R + blockDim.x - 1) / blockDim.x;
  if (per <= 1) fft_pass<R, S, 1>(buf, N, Ns, twp, w);
  else if (R <= 4 && per <= 2) fft_pass<R, S, (R <= 4 ? 2 : 1)>(buf, N, Ns, twp, w);
  else fft_pass<R, S, (R <= 2 ? 4 : 1)>(buf, N, Ns, twp, w);
}

// Unnormalised complex FFT of N (power of two, 2..8192) values in LDS,
// natural order in and out; radix-8 passes, then one of radix 4 or 2 (the
// block has at least N/8 threads).  twp holds the passes' tables one after
// the other (R Ns entries each), in the same plan as the host builds them (the
// first pass' twiddles are all 1).
template <int S>
__device__ __forceinline__ void lds_fft(double2 *buf, int N, const double2 *twp) {
  double2 w[7];
#pragma unroll
  for (int r = 0; r < 7; r++) w[r] = make_double2(1.0, 0.0);
  int Ns = 1;
  while (Ns < N) {
    const int R = fft_radix(N / Ns);
    if (R == 8) fft_pass_any<8, S>(buf, N, Ns, twp, w);
    else if (R == 4) fft_pass_any<4, S>(buf, N, Ns, twp, w);
    else fft_pass_any<2, S>(buf, N, Ns, twp, w);
    twp += R * Ns;
    Ns *= R;
  }
}

// Block sum in a fixed order: FP64 wave trees, then the waves in order.
__device__ inline double block_sum4(double v, double *s_w) {
  const double w = wave_sum(v);
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) s_w[wave] = w;
  __syncthreads();
  double t = 0.0;
  for (int k = 0; k < (int)(blockDim.x >> 6); k++) t += s_w[k];
  __syncthreads();
  return t;
}

// N block sums at once (one pair of barriers).
template <int N>
__device__ inline void block_sums(const double *v, double *out, double (*s_w)[CONV_THREADS_MAX / 64]) {
  const int wave = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < N; i++) {
    const double w = wave_sum(v[i]);
    if ((threadIdx.x & 63) == 0) s_w[i][wave] = w;
    out[i] = 0.0;
  }
  __syncthreads();
  for (int k = 0; k < (int)(blockDim.x >> 6); k++)
#pragma unroll
    for (int i = 0; i < N; i++) out[i] += s_w[i][k];
  __syncthreads();
}

// The power of two at or below a normal v > 0; 0 for every other v.
__device__ inline double pow2_of(double v) {
  const long long e = __double_as_longlong(v) & 0x7ff0000000000000ll;
  return v > 0 && e != 0x7ff0000000000000ll ? __longlong_as_double(e) : 0.0;
}

// Sum of one zone's angle distribution as k_dist leaves it.
__device__ inline double dist_sum(const double *d, int n) {
  double s = 0.0;
  for (int k = 0; k < n; k++) s += d[k];
  return s;
}

// calcFFTNormFactor band (src/Relbase.cpp:205): bins with E_lo >= 0.01 and
// E_hi < 1000, a contiguous index range of the convolution grid
__device__ inline bool in_band(const DevConvGrid &cg, int i) { return i >= cg.band_lo && i < cg.band_hi; }



}  // namespace

// Convolution of one request (relconv_kernel minus relbase, src/Relbase.cpp:257-289).
// One complex FFT carries both real inputs (input spectrum in the real part,
// rotated profile in the imaginary part); their spectra are separated, multiplied
// and inverted with a half-length complex FFT.  Grid-walking phases give each
// wavefront a contiguous run of bins, one bin per lane, so that neighbouring
// lanes read neighbouring addresses.
// WIDE: launch_conv's form for few units.  ANG: relxill_conv requests (resident
// reflection spectra weighted by the angle distribution) are among the units;
// ANG == 0 compiles them out, which frees the scalar registers that were spilled
// (4096 relconv units 356 us and 350 us).
// Bound: the latency of the phases between the barriers for few units, LDS
// traffic and FP64 issue for many (two workgroups a CU: 70 KB of LDS each).
template <int WIDE, int ANG>
__global__ __launch_bounds__(CONV_THREADS_MAX) void k_conv(BatchDev b, const XillWork *__restrict__ work, Deliver dl) {
  extern __shared__ double2 s_buf[];  // P(n) complex
  __shared__ double s_w[3][CONV_THREADS_MAX / 64];
  const int NT = blockDim.x;
  const int req = work[blockIdx.x].req;
  const int zone = work[blockIdx.x].zone;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6, nwave = NT >> 6;
  const ReqParams rq = b.req[req];
  const DevConvGrid cg = b.cg;
  const int n = cg.n;
  const int m = n >> 1;
  double *out = b.out + rq.flux_off;
  // output grid: the caller's (for relxill already redshifted on the host)
  const double *eo = b.ener_in + rq.ener_off;
  const int n_o = rq.n_in;
  double *host = nullptr;
  if constexpr (WIDE) {
    host = dl.out ? dl.out + rq.flux_off : nullptr;
    deliver_words(b, dl, req, tid);
  }
  if (b.status[req] != 0) {
    for (int j = tid; j < n_o; j += NT) {
      out[j] = 0.0;
      if (host) host[j] = 0.0;
    }
    return;
  }
  const double *Ec = cg.ener;
  const double *cf = cg.cfac;
  const double2 *tw = reinterpret_cast<const double2 *>(cg.tw);
  const bool angular = ANG && rq.model == MOD_RELXILL_CONV;
  const bool relxill = (rq.model == MOD_RELXILL || rq.model == MOD_RELXILLLP);
  // input: the caller's spectrum, or for relxill each zone's angle-weighted
  // xillver spectrum on the table grid (k_xill)
  const double *ein = relxill ? b.xt[rq.prim].ener : eo;
  const int n_in = relxill ? b.xt[rq.prim].n_ener : n_o;
  const DevReflSet *rs = angular ? &b.refl_sets[rq.refl_set] : nullptr;
  auto ge_in = [&](int k) { return ein[k]; };
  const BinRange rc = b.reach[req];
  // relxill: the reflection's scale (add_primary_spectrum,
  // src/PrimarySource.cpp:66-125): |refl_frac| for the broken power law; for
  // the lamp post |refl_frac| (times the lamp post's own reflection fraction
  // when refl_frac is a boost) over that fraction.  The primary is added by
  // k_primary.
  double refl_scale = 1.0;
  if (relxill) {
    if (rq.emis_type != EMIS_LP) {
      refl_scale = fabs(rq.refl_frac);
    } else {
      const LpRefl lr = b.refl[req];
      double rfi = rq.refl_frac;
      if (rq.xboost) rfi *= lr.refl_frac;
      refl_scale = (fabs(rfi)) / lr.refl_frac;
    }
  }
  auto o_at = [&](int i) -> double & {
    double2 &z = s_buf[P(i >> 1)];
    return (i & 1) ? z.y : z.x;
  };

  // this block's zone (relxill requests have one block per zone)
  const double *prof = b.prof + rq.prof_off + (size_t)zone * n;
  const double *fin = relxill ? b.xspec + rq.xspec_off + (size_t)zone * n_in : b.flux_in + rq.flux_off;
  const double *dist = b.dist + rq.dist_off + (size_t)zone * rq.n_incl;
  // 1. x = rebinned input * E/dE (real part), y = rotated profile * E/dE (imag part)
  double sx = 0.0, sxa = 0.0;  // band sum, sum of the magnitudes
  const int nb = n / nwave;  // bins per wavefront (a multiple of 64)
  if (!angular) {
    // _rebin_spectrum of the input, 4 conv bins per lane at a time: the edges
    // around the guessed brackets of all 4 are loaded together, then their
    // end fluxes; the exact search runs only where a guess misses
    const GridGuess gi = grid_guess(ein, n_in);
    for (int q0 = 0; q0 < nb; q0 += 4 * 64) {
      double elo[4], ehi[4], al[4], bl[4], ah[4], bh[4];
      int kl[4], kh[4], i4[4];
      bool use[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const bool valid = q0 + 64 * u < nb;
        i4[u] = wave * nb + (valid ? q0 + 64 * u : 0) + lane;
        elo[u] = Ec[i4[u]];
        ehi[u] = Ec[i4[u] + 1];
        // overlap with the input grid (the first test of _rebin_spectrum)
        use[u] = valid && gi.first <= ehi[u] && gi.last >= elo[u];
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        kl[u] = guess_index(elo[u], gi, n_in);
        kh[u] = guess_index(ehi[u], gi, n_in);
        if (use[u]) {
          al[u] = ein[kl[u]];
          bl[u] = ein[kl[u] + 1];
          ah[u] = ein[kh[u]];
          bh[u] = ein[kh[u] + 1];
        }
      }
      int imin[4], imax[4];
      double fa[4], fb[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        if (!use[u]) continue;
        const int clo = count_le_at(ge_in, n_in, elo[u], gi, kl[u], al[u], bl[u]);
        const int chi = count_le_at(ge_in, n_in, ehi[u], gi, kh[u], ah[u], bh[u]);
        imin[u] = clo > 0 ? clo - 1 : 0;
        imax[u] = chi < n_in ? chi : n_in;
        if (imax[u] > 0) imax[u]--;
        if (imin[u] >= n_in) {
          use[u] = false;
          continue;
        }
        if (imin[u] != kl[u]) {  // a missed guess or a clipped end: the edges of imin
          al[u] = ein[imin[u]];
          bl[u] = ein[imin[u] + 1];
        }
        if (imax[u] != kh[u]) {
          ah[u] = ein[imax[u]];
          bh[u] = ein[imax[u] + 1];
        }
        fa[u] = fin[imin[u]];
        fb[u] = fin[imax[u]];
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        if (q0 + 64 * u >= nb) continue;
        double xr = 0.0;
        if (use[u]) {  // rebin_bin with the edges and end fluxes in registers
          const double el = (elo[u] < al[u]) ? al[u] : elo[u];
          const double eh = (ehi[u] > bh[u]) ? bh[u] : ehi[u];
          const double ra = rcp64(bl[u] - al[u]);
          if (imax[u] == imin[u]) {
            xr = (eh - el) * ra * fa[u];
          } else {
            const double dmin = (bl[u] - el) * ra;
            const double dmax = (eh - ah[u]) * rcp64(bh[u] - ah[u]);
            xr += fa[u] * dmin + fb[u] * dmax;
            for (int jj = imin[u] + 1; jj <= imax[u] - 1; jj++) xr += fin[jj];
          }
        }
        const int i = i4[u];
        if (elo[u] >= 0.01 && ehi[u] < 1000.0) sx += xr;  // calcFFTNormFactor band (src/Relbase.cpp:205)
        sxa += fabs(xr);
        s_buf[P(i)].x = xr * cf[i];
      }
    }
  } else {
    for (int i = tid; i < n; i += NT) s_buf[P(i)].x = 0.0;
  }
  // the profile as photons per bin, renormalised (renorm_relline_profile,
  // src/Relprofile.cpp:757-779); bins no window reaches are zero
  const int per = n / NT;  // <= 8: the block has at least n/8 threads
  double ph[8];
  double sph = 0.0;
#pragma unroll
  for (int q = 0; q < 8; q++) {
    const int i = tid + q * NT;
    ph[q] = (q < per && i >= rc.lo && i <= rc.hi) ? prof[i] * cg.inv_emid[i] : 0.0;
    sph += ph[q];
  }
  const double p2[3] = {sx, sph, sxa};
  double s2[3];
  block_sums<3>(p2, s2, s_w);
  double sum_xill = readlane_d(s2[0], 0);
  // The profile's renormalisation: as a power of two, which is exact in every bin
  // and brings the profile to the input's scale (the two inputs of one complex
  // transform, whose rounding errors reach both: an input of 1e-12 a bin beside a
  // profile of 1 came out 1.6e-5 of the maximum off), times a rest that only the
  // profile's sums carry (the result is normalised by them): against FP64 sums in
  // another order 4e-13 in bins 1e-4 below the maximum, 4e-12 without.  The
  // product of the transforms is brought back by p_scale, so that it does not go
  // with the input's square (an input of 1e-165 a bin underflowed).  4096 units
  // 343 us and 345 us without and with it.
  double f = rq.do_renorm ? rq.norm / s2[1] : 1.0, f_rest = 1.0, p_scale = 1.0;
  const double f1 = pow2_of(f);
  double f2 = f1;
  if (!angular && s2[2] > 0) {
    const double r = pow2_of(s2[2] / s2[1]);
    if (r > 0) f2 = r;
  }
  if (f1 > 0 && f2 > 0) {  // (the same in every lane: kept in scalar registers)
    p_scale = readlane_d(f1 / f2, 0);
    f_rest = readlane_d(f / f2, 0);
    f = f2;
  }
  double sr = 0.0, sa = 0.0;
#pragma unroll
  for (int q = 0; q < 8; q++) {
    const int i = tid + q * NT;
    if (q < per) {
      const double pv = ph[q] * f;
      if (in_band(cg, i)) sr += pv;
      sa += pv;
      const int irot = (i - cg.i1kev + n) & (n - 1);
      s_buf[P(irot)].y = pv * cf[i];
    }
  }
  // (barrier inside: the buffer is complete)
  double sum_rel, sum_prof = 1.0;
  if (angular || relxill) {
    const double p3[2] = {sr, sa};
    double s3[2];
    block_sums<2>(p3, s3, s_w);
    sum_rel = s3[0] * f_rest;
    sum_prof = s3[1] * f_rest;
  } else {
    sum_rel = block_sum4(sr, s_w[0]) * f_rest;
  }
  if (angular) {
    sum_xill = 0.0;
    for (int k = 0; k < rs->n_incl; k++) sum_xill += dist[k] * rs->bandsum[k];
  }
  // a zone whose profile sums below 1e-12 is left out (src/Relxill.cpp:453-456)
  const bool zone_used = !(sum_prof < 1e-12);
  if (relxill && !zone_used) {  // (block-uniform)
    if (host)
      for (int j = tid; j < n_o; j += NT) host[j] = out[j];
    return;
  }
  // 2. forward complex FFT of x + i y
  lds_fft<-1>(s_buf, n, reinterpret_cast<const double2 *>(cg.twp_fwd));
  // 3. X = (W_k + conj W_{n-k})/2, Y = (W_k - conj W_{n-k})/(2i), P = X Y (k = 0..m);
  //    then pack for the half-length inverse real FFT:
  //    Z_k = (P_k + conj P_{m-k}) + i (P_k - conj P_{m-k}) e^{+2 pi i k/n}.
  //    The pair {k, m-k} reads slots k, n-k, m-k, m+k and writes slots k and
  //    m-k, which no other pair touches: no staging across a barrier.
  for (int k = tid; k <= (m >> 1); k += NT) {
    double2 Pk[2];
    const int ks[2] = {k, m - k};
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int kk = ks[u];
      const double2 wk = s_buf[P(kk)];
      const double2 wn = s_buf[P((n - kk) & (n - 1))];
      double2 Y = make_double2(0.5 * (wk.y + wn.y), -0.5 * (wk.x - wn.x));
      double2 X;
      if (angular) {
        X = make_double2(0.0, 0.0);
        for (int a = 0; a < rs->n_incl; a++) {
          const double *F = rs->fft + ((size_t)a * (m + 1) + kk) * 2;
          X.x += dist[a] * F[0];
          X.y += dist[a] * F[1];
        }
      } else {
        X = make_double2(0.5 * (wk.x + wn.x), 0.5 * (wk.y - wn.y));
        X.x *= p_scale;
        X.y *= p_scale;
      }
      Pk[u] = cmul(X, Y);
    }
    if (k == 0) {  // c2r ignores the imaginary parts of P_0 and P_m
      Pk[0].y = 0.0;
      Pk[1].y = 0.0;
    }
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int kk = ks[u];
      if (kk >= m || (u == 1 && kk == k)) continue;  // Z_m is not needed; k = m/2 once
      const double2 p0 = Pk[u], p1 = Pk[1 - u];
      const double2 A = make_double2(p0.x + p1.x, p0.y - p1.y);
      const double2 Bd = make_double2(p0.x - p1.x, p0.y + p1.y);
      double2 w = tw[kk];
      w.y = -w.y;  // e^{+2 pi i kk/n}
      const double2 Bw = cmul(Bd, w);
      s_buf[P(kk)] = make_double2(A.x - Bw.y, A.y + Bw.x);
    }
  }
  __syncthreads();
  // 4. half-length inverse FFT: z_j = out_{2j} + i out_{2j+1}
  lds_fft<+1>(s_buf, m, reinterpret_cast<const double2 *>(cg.twp_inv));
  double sc = 0.0;
#pragma unroll 8
  for (int i = tid; i < n; i += NT) {
    const double v = o_at(i) * cg.cfinv[i];
    o_at(i) = v;
    if (in_band(cg, i)) sc += v;
  }
  const double sum_conv = block_sum4(sc, s_w[0]);
  // normalizeFFTOutput (src/Relbase.cpp:199-222): applied to the rebinned
  // values below (the rebin is linear), which saves a pass over the buffer
  double fnorm = sum_rel * sum_xill / sum_conv;
  if (angular && !zone_used) fnorm = 0.0;
  // the distribution's own sum: a normalised one scales the spectrum and its band
  // sum, whose ratio to the convolution's sum fnorm holds, once each
  if (angular) fnorm /= dist_sum(dist, rs->n_incl);
  if (relxill) fnorm *= refl_scale;
  // the conv grid edges go to the upper part of the buffer, free after the
  // half-length FFT (its values occupy slots below P(m))
  double *s_e = reinterpret_cast<double *>(s_buf + P(m));
#pragma unroll 8
  for (int i = tid; i <= n; i += NT) s_e[i] = Ec[i];
  __syncthreads();
  // 5. rebin onto the caller grid; relconv zeroes outside 0.01-1000 keV;
  // relxill adds its zones up
  const GridGuess gc = grid_guess(Ec, n);
  auto ge_c = [&](int k) { return s_e[k]; };
  const int nbo = (n_o + nwave - 1) / nwave;
  const int jend = min(n_o, (wave + 1) * nbo);
  const bool relconv = !angular && !relxill;
#pragma unroll 2
  for (int q = 0; q < nbo; q += 64) {
    const int jb = wave * nbo + q + lane;
    if (jb < jend) {
      const double elo = eo[jb], ehi = eo[jb + 1];
      const int clo = count_le(ge_c, n, elo, gc);
      const int chi = count_le(ge_c, n, ehi, gc);
      double v = fnorm * rebin_bin(elo, ehi, clo, chi, ge_c, n, [&](int i) { return o_at(i); });
      if (relconv && (ehi < 0.01 || elo > 1000.0)) v = 0.0;
      if (host) {  // (one zone: what is there is the primary, or the cleared output)
        if (relxill) v += out[jb];
        out[jb] = v;
        host[jb] = v;
      } else if (relxill) {
        unsafeAtomicAdd(&out[jb], v);  // the zones add up (k_setup cleared out)
      } else {
        out[jb] = v;
      }
    }
  }
}

// relxill: the primary added to the reflection (add_primary_spectrum,
// src/PrimarySource.cpp:66-125) for refl_frac >= 0: the cut-off power law with
// the source's Ecut shifted to the observer (spec_cutoffpl,
// src/Xillspec.cpp:215-241) on the convolution grid, normalised as the
// xillver incident spectrum at the source (k_zone), times the lamp post's flux
// boost, rebinned onto the caller grid.  One workgroup per
// (request, PRIM_THREADS * per caller bins); prim_work chooses per.  Few relxill
// requests: with k_xill, before k_conv adds to the output; many, and the xillver
// models, which read k_xill's spectra: after k_conv.
// Bound: the latency of the exponential and the grid reads for few requests,
// FP64 issue (an exponential and a division a grid bin) for many.  One
// workgroup a request, with the norm's 500 exponentials and 12 rounds of bins,
// took 28 us for one request of 3000 bins (47 us with the nthcomp primary) and
// 57 us for 1024; now 5.5 us (8 us) and 51 us.
__device__ __forceinline__ void primary_bins(const BatchDev &b, const PrimWork &pw, int block) {
  const int per = pw.per;
  const int req = pw.reqs[block / pw.chunks];
  const int j0 = (block % pw.chunks) * (PRIM_THREADS * per) + threadIdx.x;
  const ReqParams &rq = b.req[req];
  const int j1 = min(rq.n_in, j0 + PRIM_THREADS * per);  // this thread: j0, j0 + PRIM_THREADS, ... below j1
  if (j0 >= j1) return;
  const bool xill = rq.model == MOD_XILLVER;
  if (xill && b.status[req] != 0) {
    for (int jb = j0; jb < j1; jb += PRIM_THREADS) b.out[rq.flux_off + jb] = 0.0;
    return;
  }
  if (!xill && (b.status[req] != 0 || !(rq.refl_frac >= 0))) return;
  const DevConvGrid &cg = b.cg;
  const int n = cg.n;
  const double ect = rq.xect_src, gam = rq.xgam;
  const ZoneRec &z0 = b.zone[rq.zone_off];
  double prim_scale = 1.0;
  if (rq.emis_type == EMIS_LP) prim_scale = b.refl[req].f_inf_rest / 0.5 * z0.boost;
  // nthcomp: the source's solve (k_nth) observed at redshift 1/g - 1
  // (spec_nthcomp, src/Xillspec.cpp:243-253) with the norm of its spectrum
  // at the source
  const bool nth = rq.prim == PRIM_NTHCOMP;
  const int sol = nth ? rq.nth_sol : 0;
  const double *nx = b.nth_x + (size_t)sol * (NTH_N + 1);
  const double *ns = b.nth_s + (size_t)sol * NTH_N;
  const int nn = nth ? b.nth_n[sol] : 0;
  const double zo = 1 / rq.g_so - 1;
  const double nfac = nth ? nthcomp_normfac(nx, ns, nn, zo) : 0.0;
  // the blackbody (relxillNS) takes no energy shift (calc_primary_spectrum,
  // src/Xillspec.cpp:293-295)
  const bool bb = rq.prim == PRIM_BBODY;
  const double nf = z0.nf;
  // the primary on the convolution grid, evaluated where the rebin reads it
  // (one or two grid bins per output bin on caller grids finer than the
  // convolution grid; every grid bin of the output bin, each with its
  // exponential, on coarser ones): no staging buffer
  const double *ce = cg.ener;
  const double *cl = cg.ln_emid;
  const double ect_o = ect * rq.g_so;
  auto prim_at = [&](int i) {
    const double v = nth  ? nthcomp_bin(ce[i], ce[i + 1], nthcomp_edge(nx, ns, nn, ce[i], zo),
                                        nthcomp_edge(nx, ns, nn, ce[i + 1], zo), nfac)
                     : bb ? bbody_bin(ce[i], ce[i + 1], rq.xktbb)
                          : cutoffpl_bin(ce[i], ce[i + 1], cl[i], ect_o, gam);
    return (v * nf) * prim_scale;
  };
  const double *eo = b.ener_in + rq.ener_off;
  double *out = b.out + rq.flux_off;
  if (xill) {
    // the xillver models: the table spectrum times 0.5 cos(Incl)
    // (norm_xillver_spec, src/Xillspec.cpp:536-545) rebinned onto the
    // (redshifted) caller grid, times |refl_frac|, plus the normalised primary
    // evaluated on the caller grid itself for refl_frac >= 0
    // (add_primary_component, src/Relbase.cpp:294-344)
    const DevXillTable &xt = b.xt[rq.prim];
    const int nxt = xt.n_ener;
    const double *xs = b.xspec + rq.xspec_off;
    const double slab = rq.norm, rf = rq.refl_frac;
    const GridGuess gx = grid_guess(xt.ener, nxt);
    auto ge_x = [&](int k) { return xt.ener[k]; };
    auto refl_at = [&](int k) { return xs[k] * slab; };
    for (int jb = j0; jb < j1; jb += PRIM_THREADS) {
      const double elo = eo[jb], ehi = eo[jb + 1];
      const int xlo = count_le(ge_x, nxt, elo, gx);
      const int xhi = count_le(ge_x, nxt, ehi, gx);
      double v = rebin_bin(elo, ehi, xlo, xhi, ge_x, nxt, refl_at) * fabs(rf);
      if (rf >= 0) {
        const double p = nth  ? nthcomp_bin(elo, ehi, nthcomp_edge(nx, ns, nn, elo, 0.0),
                                            nthcomp_edge(nx, ns, nn, ehi, 0.0), nfac)
                         : bb ? bbody_bin(elo, ehi, rq.xktbb)
                              : cutoffpl_bin(elo, ehi, log(0.5 * (elo + ehi)), ect, gam);
        v += p * nf;
      }
      out[jb] = v;
    }
    return;
  }
  const GridGuess gc = grid_guess(ce, n);
  auto ge_c = [&](int k) { return ce[k]; };
  for (int jb = j0; jb < j1; jb += PRIM_THREADS) {
    const double elo = eo[jb], ehi = eo[jb + 1];
    const int clo = count_le(ge_c, n, elo, gc);
    const int chi = count_le(ge_c, n, ehi, gc);
    out[jb] += rebin_bin(elo, ehi, clo, chi, ge_c, n, prim_at);
  }
}

__global__ __launch_bounds__(PRIM_THREADS) void k_primary(BatchDev b, PrimWork pw) { primary_bins(b, pw, blockIdx.x); }

// relxill: the xillver spectrum of the request's parameters for every
// emission angle (interp_5d_tab_incl, src/xilltable.c:812-876: 16 corners of
// the four interpolated parameters, in the reference's order and with its
// weight products) weighted by the angle distribution (calc_xillver_angdep,
// src/Xillspec.cpp:557-573), for one-zone requests.  XILL_BINS bins per
// thread; every table read is coalesced across the block.  Angles with zero
// weight are skipped (they add exactly 0).  The zone's Ecut bracket, angle
// distribution and normalisation change come from its zone record.
// PRIM: the first workgroups are k_primary's (it needs nothing of this kernel's:
// the convolutions add to what it leaves in the output).
template <int PRIM>
__global__ __launch_bounds__(XILL_THREADS, 4) void k_xill1(BatchDev b, const XillWork *__restrict__ work, int chunks,
                                                           PrimWork pw) {
  if (PRIM && (int)blockIdx.x < pw.blocks) {
    primary_bins(b, pw, blockIdx.x);
    return;
  }
  const int block = PRIM ? blockIdx.x - pw.blocks : blockIdx.x;
  const XillWork wk = work[block / chunks];
  const int req = wk.req;
  if (b.status[req] != 0) return;
  const ReqParams &rq = b.req[req];
  const DevXillTable xt = b.xt[rq.prim];
  const DensDiv dd = dens_of(rq.xdens_div);
  // XILL_BINS bins per thread, XILL_THREADS apart: the corner weights and rows
  // are set up once for all of them, and their loads are in flight together
  const int e0 = (block % chunks) * (XILL_THREADS * XILL_BINS) + threadIdx.x;
  if (e0 >= xt.n_ener) return;
  const ZoneRec zr = b.zone[rq.zone_off + wk.zone];
  int i0[4];
  double f[4];
#pragma unroll
  for (int k = 0; k < 4; k++) {  // the zone's own Ecut and logXi brackets
    const bool ect = (k == xt.ect_dim), lxi = (k == xt.lxi_dim);
    i0[k] = ect ? zr.ect_ind : (lxi ? zr.lxi_ind : rq.xind[k]);
    f[k] = ect ? zr.ect_fac : (lxi ? zr.lxi_fac : rq.xfac[k]);
  }
  // corner c has the offsets of bits 3, 2, 1, 0 of kCorner[c] on axes 0..3
  constexpr unsigned char kCorner[16] = {0x0, 0x8, 0x4, 0x2, 0xC, 0xA, 0x6, 0xE,
                                         0x1, 0x9, 0x5, 0x3, 0xD, 0xB, 0x7, 0xF};
  double w[16];
  unsigned row[16];  // first row (inclination 0) of each corner
#pragma unroll
  for (int c = 0; c < 16; c++) {
    int o[4];
    double fk[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      o[k] = (kCorner[c] >> (3 - k)) & 1;
      fk[k] = o[k] ? f[k] : (1.0 - f[k]);
    }
    w[c] = fk[0] * fk[1] * fk[2] * fk[3];
    const unsigned r = (((unsigned)(i0[0] + o[0]) * xt.n_val[1] + (i0[1] + o[1])) * xt.n_val[2] + (i0[2] + o[2])) *
                           xt.n_val[3] + (i0[3] + o[3]);
    row[c] = r * xt.n_incl;
  }
  const double *dist = b.dist + rq.dist_off + (size_t)wk.zone * xt.n_incl;
  const size_t ne = (size_t)xt.n_ener;
  int eb[XILL_BINS];
  bool in[XILL_BINS];
#pragma unroll
  for (int u = 0; u < XILL_BINS; u++) {
    eb[u] = e0 + u * XILL_THREADS;
    in[u] = eb[u] < xt.n_ener;
    if (!in[u]) eb[u] = e0;  // a valid address; the result is not stored
  }
  double acc[XILL_BINS];
#pragma unroll
  for (int u = 0; u < XILL_BINS; u++) acc[u] = 0.0;
  const int n_o = xt.n_out > 1 ? 2 : 1;
  for (int a = 0; a < xt.n_incl; a++) {
    const double d = dist[a];
    if (d == 0.0) continue;
    double s[XILL_BINS];
#pragma unroll
    for (int u = 0; u < XILL_BINS; u++) s[u] = 0.0;
    for (int o = 0; o < n_o; o++) {
      // a six-parameter table: the five-parameter interpolation at both
      // brackets of its first axis, lerped (interp_6d_tab_incl,
      // src/xilltable.c:997-1020); five parameters: one pass with weight 1
      const double wo = n_o == 1 ? 1.0 : (o ? rq.xo_fac : 1.0 - rq.xo_fac);
      const size_t ob = (size_t)(rq.xo_ind + o) * xt.outer_rows;
      double so[XILL_BINS];
#pragma unroll
      for (int u = 0; u < XILL_BINS; u++) so[u] = 0.0;
#pragma unroll
      for (int c = 0; c < 16; c++) {
        const float *src = xt.spec + (ob + row[c] + a) * ne;
#pragma unroll
        for (int u = 0; u < XILL_BINS; u++) so[u] += w[c] * xval(src[eb[u]], dd);
      }
#pragma unroll
      for (int u = 0; u < XILL_BINS; u++) s[u] += wo * so[u];
    }
#pragma unroll
    for (int u = 0; u < XILL_BINS; u++) acc[u] += d * s[u];
  }
  // (the xillver models' weights are no distribution: an inclination bracket)
  const double scale = rq.model == MOD_XILLVER ? zr.ncf : zr.ncf * dist_sum(dist, xt.n_incl);
  double *dst = b.xspec + rq.xspec_off + (size_t)wk.zone * xt.n_ener;
#pragma unroll
  for (int u = 0; u < XILL_BINS; u++)
    if (in[u]) dst[eb[u]] = acc[u] / scale;
}

// relxilllp: the same for the zones of a lamp-post request (src/Relxill.cpp:
// 357-388), which differ only in the Ecut they see and in their angle
// distributions.  One unit per (request, slice of XILL_THREADS * XILL_BINS_Z
// table bins) for all zones, so that a table row is read once however many
// zones use it:
//   zone z = sum_a d_z[a] sum_c w_c row_c(a)
//          = sum_{(e, a)} k_z(e, a) sum_{c8} w_c8 row_{c8, e}(a),
//   k_z(e, a) = d_z[a] (1 - f_z) for e = i_z, d_z[a] f_z for e = i_z + 1, else 0,
// with (i_z, f_z) the zone's bracket on the Ecut axis and c8 the eight
// corners of the other three axes (their weights as the products of the
// reference's factors).  The block first lists the pairs (e, a) that some
// zone weights, with every zone's k_z, in LDS (in windows of XILL_THREADS
// candidates, in a fixed order), then streams the 8 rows of each listed pair.
// Tables without an Ecut axis use the request's bracket on the fourth axis
// for every zone.
// PRIM: as k_xill1's.
template <int NZ, int PRIM>
__global__ __launch_bounds__(XILL_THREADS, 3) void k_xillz(BatchDev b, const XillWork *__restrict__ work, int chunks,
                                                           PrimWork pw) {
  if (PRIM && (int)blockIdx.x < pw.blocks) {
    primary_bins(b, pw, blockIdx.x);
    return;
  }
  const int block = PRIM ? blockIdx.x - pw.blocks : blockIdx.x;
  constexpr int NW = XILL_THREADS / 64;
  __shared__ int s_ind[NZ];
  __shared__ double s_fac[NZ], s_scale[NZ];
  __shared__ unsigned s_off[XILL_THREADS];
  __shared__ double s_k[XILL_THREADS][NZ];
  __shared__ int s_wn[NW];
  const XillWork wk = work[block / chunks];
  const int req = wk.req;
  if (b.status[req] != 0) return;  // uniform over the block
  const ReqParams &rq = b.req[req];
  const DevXillTable xt = b.xt[rq.prim];
  const DensDiv dd = dens_of(rq.xdens_div);
  const int nz = min(rq.n_zones, NZ);
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int zax = xt.ect_dim >= 0 ? xt.ect_dim : 3;
  if (tid < nz) {
    const ZoneRec &zr = b.zone[rq.zone_off + tid];
    s_ind[tid] = xt.ect_dim >= 0 ? zr.ect_ind : rq.xind[3];
    s_fac[tid] = xt.ect_dim >= 0 ? zr.ect_fac : rq.xfac[3];
    s_scale[tid] = zr.ncf * dist_sum(b.dist + rq.dist_off + tid * xt.n_incl, xt.n_incl);
  }
  __syncthreads();
  int elo = s_ind[0], ehi = s_ind[0];
  for (int z = 1; z < nz; z++) {
    elo = min(elo, s_ind[z]);
    ehi = max(ehi, s_ind[z]);
  }
  const int ni = xt.n_incl;
  const int n_o = xt.n_out > 1 ? 2 : 1;
  const int n_cand = (ehi - elo + 2) * ni;  // candidate pairs (e, a), e in [elo, ehi + 1]
  double w8[8];
  unsigned cb[8], stride;
  corners8(xt, rq, zax, w8, cb, &stride);
  const double *dist = b.dist + rq.dist_off;
  const size_t ne = (size_t)xt.n_ener;
  const int e0 = (block % chunks) * (XILL_THREADS * XILL_BINS_Z) + tid;
  int eb[XILL_BINS_Z];
  bool in[XILL_BINS_Z];
#pragma unroll
  for (int u = 0; u < XILL_BINS_Z; u++) {
    eb[u] = e0 + u * XILL_THREADS;
    in[u] = eb[u] < xt.n_ener;
    if (!in[u]) eb[u] = 0;  // a valid address; the result is not stored
  }
  double acc[NZ][XILL_BINS_Z];
#pragma unroll
  for (int z = 0; z < NZ; z++)
#pragma unroll
    for (int u = 0; u < XILL_BINS_Z; u++) acc[z][u] = 0.0;
  for (int q0 = 0; q0 < n_cand; q0 += XILL_THREADS) {
    // list this window's used pairs: thread tid tests candidate q0 + tid
    const int q = q0 + tid;
    const int e = elo + q / ni, a = q % ni;
    auto kz = [&](int z) {  // k_z(e, a); zones beyond nz weigh nothing
      if (z >= nz) return 0.0;
      const double d = dist[z * ni + a];
      const int iz = s_ind[z];
      return e == iz ? d * (1.0 - s_fac[z]) : (e == iz + 1 ? d * s_fac[z] : 0.0);
    };
    bool used = false;
    if (q < n_cand)
      for (int z = 0; z < nz; z++) used |= kz(z) != 0.0;
    const unsigned long long m = __ballot(used);
    if (lane == 0) s_wn[wv] = __popcll(m);
    __syncthreads();
    int slot = __popcll(m & ((1ull << lane) - 1ull)), n_used = 0;
    for (int w = 0; w < NW; w++) {
      if (w < wv) slot += s_wn[w];
      n_used += s_wn[w];
    }
    if (used) {
      s_off[slot] = (unsigned)e * stride * (unsigned)ni + (unsigned)a;
      for (int z = 0; z < NZ; z++) s_k[slot][z] = kz(z);
    }
    __syncthreads();
    if (e0 < xt.n_ener) {
      for (int p = 0; p < n_used; p++) {
        const unsigned po = s_off[p];
        double s8[XILL_BINS_Z];
#pragma unroll
        for (int u = 0; u < XILL_BINS_Z; u++) s8[u] = 0.0;
        for (int o = 0; o < n_o; o++) {  // (a six-parameter table: both brackets of its first axis)
          const double wo = n_o == 1 ? 1.0 : (o ? rq.xo_fac : 1.0 - rq.xo_fac);
          const size_t ob = (size_t)(rq.xo_ind + o) * xt.outer_rows;
          double so[XILL_BINS_Z];
#pragma unroll
          for (int u = 0; u < XILL_BINS_Z; u++) so[u] = 0.0;
#pragma unroll
          for (int c = 0; c < 8; c++) {
            const float *src = xt.spec + (ob + cb[c] + po) * ne;
#pragma unroll
            for (int u = 0; u < XILL_BINS_Z; u++) so[u] += w8[c] * xval(src[eb[u]], dd);
          }
#pragma unroll
          for (int u = 0; u < XILL_BINS_Z; u++) s8[u] += wo * so[u];
        }
#pragma unroll
        for (int z = 0; z < NZ; z++) {
          const double k = s_k[p][z];
#pragma unroll
          for (int u = 0; u < XILL_BINS_Z; u++) acc[z][u] += k * s8[u];
        }
      }
    }
    __syncthreads();  // the list is rewritten by the next window
  }
  if (e0 >= xt.n_ener) return;
#pragma unroll
  for (int z = 0; z < NZ; z++) {
    if (z < nz) {
      const double scale = s_scale[z];
      double *dst = b.xspec + rq.xspec_off + (size_t)z * ne;
#pragma unroll
      for (int u = 0; u < XILL_BINS_Z; u++)
        if (in[u]) dst[eb[u]] = acc[z][u] / scale;
    }
  }
}

// Resident reflection set: per angle, rebin onto the convolution grid, band
// sum, and the real FFT of (spectrum * E/dE), stored for k = 0..n/2.
__global__ __launch_bounds__(CONV_THREADS_MAX) void k_refl_prepare(DevConvGrid cg, const double *refl_ener,
                                                                  const double *refl, int n_refl,
                                                                  double *spec, double *bandsum, double *fft) {
  extern __shared__ double2 s_buf[];
  __shared__ double s_w[CONV_THREADS_MAX / 64];
  const int a = blockIdx.x;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6, nwave = blockDim.x >> 6;
  const int n = cg.n, m = n >> 1;
  const double *f0 = refl + (size_t)a * n_refl;
  const GridGuess gi = grid_guess(refl_ener, n_refl);
  auto ge = [&](int k) { return refl_ener[k]; };
  const int nb = n / nwave;
  double sx = 0.0;
  for (int q = 0; q < nb; q += 64) {
    const int i = wave * nb + q + lane;
    const double elo = cg.ener[i], ehi = cg.ener[i + 1];
    const int clo = count_le(ge, n_refl, elo, gi);
    const int chi = count_le(ge, n_refl, ehi, gi);
    const double xr = rebin_bin(elo, ehi, clo, chi, ge, n_refl, [&](int k) { return f0[k]; });
    spec[(size_t)a * n + i] = xr;
    if (elo >= 0.01 && ehi < 1000.0) sx += xr;
    s_buf[P(i)] = make_double2(xr * cg.cfac[i], 0.0);
  }
  const double s = block_sum4(sx, s_w);
  if (tid == 0) bandsum[a] = s;
  lds_fft<-1>(s_buf, n, reinterpret_cast<const double2 *>(cg.twp_fwd));
  for (int k = tid; k <= m; k += blockDim.x) {
    fft[((size_t)a * (m + 1) + k) * 2 + 0] = s_buf[P(k)].x;
    fft[((size_t)a * (m + 1) + k) * 2 + 1] = s_buf[P(k)].y;
  }
}

// plain streaming copy, used to calibrate the HBM byte counters
__global__ __launch_bounds__(256) void k_copy(const double4 *__restrict__ src, double4 *__restrict__ dst, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    dst[i] = src[i];
  }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static int copy_blocks(int64_t words) {
  return (int)std::max<int64_t>(1, std::min<int64_t>(1024, (words + COPY_THREADS - 1) / COPY_THREADS));
}

int launch_begin(int *ctr, const void *src, void *dst, int64_t n16, void *stream) {
  hipLaunchKernelGGL(k_begin, dim3(copy_blocks(n16)), dim3(COPY_THREADS), 0, (hipStream_t)stream, ctr,
                     (const uint4 *)src, (uint4 *)dst, n16);
  return (int)hipGetLastError();
}

int launch_deliver(const BatchDev &b, int *res, double *res_out, int64_t n_out, void *stream) {
  hipLaunchKernelGGL(k_deliver, dim3(copy_blocks(std::max<int64_t>(b.n_req, n_out / 2))), dim3(COPY_THREADS), 0,
                     (hipStream_t)stream, b, res, res_out, n_out);
  return (int)hipGetLastError();
}

int launch_setup(const BatchDev &b, void *stream) {
  if (b.n_req <= 0) return 0;
  auto go = [&](auto kern, int nt) { hipLaunchKernelGGL(kern, dim3(b.n_req), dim3(nt), 0, (hipStream_t)stream, b); };
  // up to one workgroup a CU the wide form (256 requests: 28 us, 31 us with 256
  // threads); 512 requests: 44 us and 39 us.  1024 threads spill (128 registers)
  // and are no faster than 512 for one request.
  const bool wide = b.n_req <= 256;
  if (b.max_zones > LP_ZONES) wide ? go(k_setup<MAX_ZONES, 512>, 512) : go(k_setup<MAX_ZONES, 256>, 256);
  else wide ? go(k_setup<LP_ZONES, 512>, 512) : go(k_setup<LP_ZONES, 256>, 256);
  return (int)hipGetLastError();
}

// LDS of one k_integrate wavefront: lane rows, then (FP64 path) 64 weight
// slots, then the SUM_BINS x SUM_STRIDE parked values, which double as the
// node-row staging area.  *stage_rows: node rows the staging area takes, as
// many as fit without lowering the wavefronts per CU that the LDS allows (at
// most 12, the VGPR limit of the FP32 path), up to 8 and at least 2.
static size_t integrate_lds(const BatchDev &b, bool cos_rows, size_t elem, int *stage_rows) {
  const size_t rows = integrate_rows_bytes(b.rt.n_g, cos_rows, elem);
  const size_t w = (elem == sizeof(double)) ? 64 * sizeof(double) : 0;
  const size_t park = (size_t)SUM_BINS * SUM_STRIDE * elem;
  const size_t nq = 2 * (size_t)b.rt.n_g;
  // wavefronts per CU that the LDS holds: gfx950 allocates a workgroup's LDS
  // in 1280-byte granules, 128 per CU (160 KB); at most 16 (the VGPRs of the
  // FP32 forms allow four per SIMD)
  auto per_cu = [](size_t lds) { return std::min<size_t>(16, 128 / ((lds + 1279) / 1280)); };
  const size_t base = rows + w + park;
  for (int c = 8; c > 2; c--) {
    if ((size_t)c * nq > (size_t)STAGE_MAX) continue;
    const size_t need = rows + w + std::max(park, (size_t)c * nq * sizeof(double));
    if (per_cu(need) >= per_cu(base)) {
      *stage_rows = c;
      return need;
    }
  }
  *stage_rows = 2;  // the two rows a radius lerps between (2 nq <= STAGE_MAX: n_g <= MAX_NG)
  return rows + w + std::max(park, (size_t)2 * nq * sizeof(double));
}

static int fine_chunks(const BatchDev &b) { return (b.nr_fine + RAD_CHUNK - 1) / RAD_CHUNK; }

int launch_dist(const BatchDev &b, const int *reqs, int n_reqs, void *stream) {
  if (n_reqs <= 0) return 0;
  hipLaunchKernelGGL(k_dist, dim3(n_reqs * fine_chunks(b)), dim3(64), sizeof(double) * dist_lds(b.max_zones),
                     (hipStream_t)stream, b, reqs, fine_chunks(b));
  return (int)hipGetLastError();
}

bool integrate_takes_side(const BatchDev &b, int n_blocks) { return n_blocks >= b.item_cap; }

int launch_integrate(const BatchDev &b, int n_blocks, bool cos_rows, const SideWork *side_in, void *stream) {
  if (b.n_req <= 0 || n_blocks <= 0) return 0;
  hipStream_t st = (hipStream_t)stream;
  int stage = 0;
  size_t lds = integrate_lds(b, cos_rows, b.mode == 0 ? sizeof(double) : sizeof(float), &stage);
  SideWork side = SideWork();
  if (side_in) {
    side = *side_in;
    side.n_rc = fine_chunks(b);
    if (side.n_ang > 0) lds = std::max(lds, sizeof(double) * dist_lds(b.max_zones));
    if (side.n_zone > 0) lds = std::max(lds, sizeof(double) * ZONE_LDS);
  }
  const bool one = integrate_takes_side(b, n_blocks);  // a workgroup for every item there can be
  const int n_side = side.n_ang * side.n_rc + side.n_zone;
  if (n_side > 0 && !one) return (int)hipErrorInvalidValue;
  auto go = [&](auto kern) {
    (void)hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL(kern, dim3(n_side + n_blocks), dim3(64), lds, st, b, stage, side);
  };
  if (b.mode == 0) {
    if (one) cos_rows ? go(k_integrate<0, 1, 1>) : go(k_integrate<0, 0, 1>);
    else cos_rows ? go(k_integrate<0, 1, 0>) : go(k_integrate<0, 0, 0>);
  } else {
    if (one) cos_rows ? go(k_integrate<1, 1, 1>) : go(k_integrate<1, 0, 1>);
    else cos_rows ? go(k_integrate<1, 1, 0>) : go(k_integrate<1, 0, 0>);
  }
  return (int)hipGetLastError();
}

int launch_fixup(const BatchDev &b, bool cos_rows, void *stream) {
  if (b.mode != 1 || b.n_req <= 0) return 0;
  const size_t lds = (size_t)(cos_rows ? 2 : 1) * (64 / FIX_LANES) * (2 * b.rt.n_g + 1) * sizeof(double);
  (void)hipFuncSetAttribute((const void *)k_fixup, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  hipLaunchKernelGGL(k_fixup, dim3(2048), dim3(64), lds, (hipStream_t)stream, b, (int)cos_rows);
  return (int)hipGetLastError();
}

int launch_finalize(const BatchDev &b, const Deliver &dl, void *stream) {
  if (b.n_req <= 0) return 0;
  hipLaunchKernelGGL(k_finalize, dim3(b.n_req), dim3(FINAL_THREADS), 0, (hipStream_t)stream, b, dl);
  return (int)hipGetLastError();
}

static size_t conv_lds(int n) { return (size_t)(n + n / 16) * sizeof(double2); }
// n/8 threads fill a pass of the transforms.
static int conv_threads(int n) { return std::max(CONV_THREADS, n / 8); }

bool conv_delivers(int n_conv_work) { return n_conv_work <= 256; }

int launch_conv(const BatchDev &b, const XillWork *conv_work, int n_conv_work, bool angular, const Deliver &dl,
                void *stream) {
  if (n_conv_work <= 0) return 0;
  const size_t lds = conv_lds(b.cg.n);
  auto go = [&](auto kern, int nt) {
    (void)hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL(kern, dim3(n_conv_work), dim3(nt), lds, (hipStream_t)stream, b, conv_work, dl);
  };
  // where every unit has a CU of its own the most threads (but not more than
  // bins, which a wavefront takes by the 64), so that the phases over the grid
  // take half the rounds: 1 relxill unit of 4096 bins 36 us and 33 us, 256 relconv
  // units 50 us and 45 us; 1024 units 110 us and 127 us (1.2 to 5 us less all of
  // them with the twiddles read ahead)
  if (conv_delivers(n_conv_work)) {
    const int nt = std::min(CONV_THREADS_MAX, b.cg.n);
    angular ? go(k_conv<1, 1>, nt) : go(k_conv<1, 0>, nt);
  } else {
    const int nt = conv_threads(b.cg.n);
    angular ? go(k_conv<0, 1>, nt) : go(k_conv<0, 0>, nt);
  }
  return (int)hipGetLastError();
}

// the larger energy grid of the two xillver tables (units beyond a request's
// own table return at once)
static int xill_n_ener(const BatchDev &b) {
  int n = 0;
  for (int pr = 0; pr < N_PRIM; pr++) n = std::max(n, b.xt[pr].n_ener);
  return n;
}

// k_primary's split of n_reqs requests of up to max_bins caller bins.
static PrimWork prim_work(const int *reqs, int n_reqs, int max_bins) {
  // bins per thread: one until the chip holds no more workgroups at once (1024),
  // then as many as keep it full: a workgroup's fixed part (parameters, grid
  // guesses) costs about two bins.  1024 requests of 3000 bins: 72 us with one
  // bin, 51 us with eleven; 128 requests: 9 us with one, 26 us with twelve.
  PrimWork pw;
  pw.reqs = reqs;
  const int rounds = (max_bins + PRIM_THREADS - 1) / PRIM_THREADS;
  pw.per = (int)std::max<int64_t>(1, std::min<int64_t>(rounds, (int64_t)n_reqs * rounds / 1024));
  pw.chunks = (rounds + pw.per - 1) / pw.per;
  pw.blocks = n_reqs * pw.chunks;
  return pw;
}

// up to 256 requests: one relxill request 109 us and 100 us a call, 128
// relxilllp 554 us and 550 us; with 1024, whose launches fill the chip, 2.09 ms
// and 2.15 ms (k_xill1 loses a wavefront per SIMD to the primary's registers)
int xill_takes_primary(int n_xill, int n_prim) { return n_xill > 0 && n_prim <= 256 ? n_prim : 0; }

int launch_xill(const BatchDev &b, const XillWork *work, int n_single, int n_multi, const int *prim, int n_prim,
                int max_bins, void *stream) {
  static_assert(XILL_THREADS == PRIM_THREADS, "k_primary's workgroups run in k_xill's launches");
  PrimWork pw = prim_work(prim, n_prim, max_bins);
  if (n_single > 0) {
    const int chunks = (xill_n_ener(b) + XILL_THREADS * XILL_BINS - 1) / (XILL_THREADS * XILL_BINS);
    const int grid = pw.blocks + n_single * chunks;
    auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3(grid), dim3(XILL_THREADS), 0, (hipStream_t)stream, b, work, chunks, pw);
    };
    pw.blocks > 0 ? go(k_xill1<1>) : go(k_xill1<0>);
    pw.blocks = 0;  // (taken)
  }
  if (n_multi > 0) {
    const int chunks = (xill_n_ener(b) + XILL_THREADS * XILL_BINS_Z - 1) / (XILL_THREADS * XILL_BINS_Z);
    const int grid = pw.blocks + n_multi * chunks;
    auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3(grid), dim3(XILL_THREADS), 0, (hipStream_t)stream, b, work + n_single, chunks, pw);
    };
    pw.blocks > 0 ? go(k_xillz<LP_ZONES, 1>) : go(k_xillz<LP_ZONES, 0>);
  }
  return (int)hipGetLastError();
}

// the solves' LDS (45 KB) leaves three workgroups a CU: 8 requests' set-up 101 us,
// 111 us with the solves in a launch of their own, 32 requests 121 us and 130 us;
// 64 requests (72 us and 61 us for solves, zones and sums) keep them apart
bool rrad_takes_nth(int n_corr) { return n_corr <= 32; }

int launch_before_rrad(const BatchDev &b, const int *corr_reqs, int n_corr, const XillWork *work, int n_work, bool nth,
                       void *stream) {
  if (n_corr <= 0) return 0;
  const int n_chunk = rrad_chunks(xill_n_ener(b));
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(n_work + n_corr * n_chunk), dim3(RRA_THREADS), 0, (hipStream_t)stream, b, work,
                       n_work, corr_reqs, n_chunk);
  };
  nth ? go(k_before_rrad<1>) : go(k_before_rrad<0>);
  return (int)hipGetLastError();
}

int launch_rrad(const BatchDev &b, const int *reqs, int n_reqs, void *stream) {
  if (n_reqs > 0) {
    auto go = [&](auto kern, int groups) {
      hipLaunchKernelGGL(kern, dim3(n_reqs * groups), dim3(64 * RR_ZONES), 0, (hipStream_t)stream, b, reqs);
    };
    // a workgroup per incident zone repeats the emissivities of all zones, which
    // costs nothing while CUs are idle: 8 requests' set-up 95 us and 102 us, 24
    // requests 117 us and 121 us; 32 requests 127 us and 122 us
    n_reqs <= 24 ? go(k_rrad<1>, MAX_RR) : go(k_rrad<0>, MAX_RR / RR_ZONES);
  }
  return (int)hipGetLastError();
}

int launch_zone(const BatchDev &b, const XillWork *work, int n_work, void *stream) {
  if (n_work <= 0) return 0;
  hipLaunchKernelGGL(k_zone, dim3(n_work), dim3(64), 0, (hipStream_t)stream, b, work);
  return (int)hipGetLastError();
}

int launch_nth(const BatchDev &b, const XillWork *work, int n_work, void *stream) {
  if (n_work <= 0) return 0;
  hipLaunchKernelGGL(k_nth, dim3(n_work), dim3(NTH_THREADS_R), 0, (hipStream_t)stream, b, work);
  return (int)hipGetLastError();
}

int launch_primary(const BatchDev &b, const int *reqs, int n_reqs, int max_bins, void *stream) {
  if (n_reqs <= 0) return 0;
  const PrimWork pw = prim_work(reqs, n_reqs, max_bins);
  hipLaunchKernelGGL(k_primary, dim3(pw.blocks), dim3(PRIM_THREADS), 0, (hipStream_t)stream, b, pw);
  return (int)hipGetLastError();
}

int launch_copy(const void *src, void *dst, size_t bytes, void *stream) {
  const size_t n = bytes / sizeof(double4);
  hipLaunchKernelGGL(k_copy, dim3(2048), dim3(256), 0, (hipStream_t)stream, (const double4 *)src, (double4 *)dst, n);
  return (int)hipGetLastError();
}

int launch_refl_prepare(const DevConvGrid &cg, const double *refl_ener, const double *refl, int n_refl,
                        int n_incl, double *spec, double *bandsum, double *fft, void *stream) {
  const size_t lds = conv_lds(cg.n);
  (void)hipFuncSetAttribute((const void *)k_refl_prepare, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  hipLaunchKernelGGL(k_refl_prepare, dim3(n_incl), dim3(conv_threads(cg.n)), lds, (hipStream_t)stream, cg, refl_ener,
                     refl, n_refl, spec, bandsum, fft);
  return (int)hipGetLastError();
}

}  // namespace rx
