// nthcomp.hip -- the nthcomp primary continuum on the GPU.
//
// spec_nthcomp (src/Xillspec.cpp:243-253): thermal Comptonization of a
// disc-blackbody seed (kT_bb = 0.05 keV, get_nthcomp_param,
// src/relutility.c:625-632) as computed by c_donthcomp (src/donthcomp.c:
// 683-793), with the solve and the bin integrals of rx_nthcomp.h.  Two
// kernels:
//   k_nth_grid       once per device: the photon grid x_j = 1e-4 T_bb 10^(0.02 j),
//                    Cooper's coefficients, the Klein-Nishina ratios and the disc
//                    seed (five-point Gauss per seed bin), which every solve shares;
//   k_nthcomp        one 256-thread workgroup per (Gamma, kTe): the Kompaneets
//                    equation on that grid (<= 899 points, nth_solve), written to
//                    HBM as (x, E F_E, jmax);
//   k_nthcomp_bins   one workgroup per spectrum: E F_E interpolated at every
//                    edge of the caller grid (the bracket of the reference's
//                    monotone walk, from the log-spaced grid), divided by E^2,
//                    trapezoid per bin, times the normalisation E F_E(1 keV,
//                    source) = 1.
// Results differ from the FP64 oracle by the round-off of the reference's
// elimination and by the last-ulp differences of the device pow / exp / log.
#include <hip/hip_runtime.h>

#include "engine.h"
#include "rx_math.h"
#include "rx_nthcomp.h"

namespace rx {

namespace {

constexpr int NTH_THREADS = 256;

// The factors of nth_grid_tab, by one workgroup.
__global__ __launch_bounds__(NTH_THREADS) void k_nth_grid(double *__restrict__ tab) {
#pragma clang fp contract(off)
  __shared__ double s_x[NTH_N + 1], s_a[NTH_N], s_b[NTH_N], s_ph[NTH_N];
  const int tid = threadIdx.x;
  const double tempbb = NTH_KTBB / 511.;
  const double xmin = tempbb * 1e-4;
  const int jmaxth = min(900, (int)(nth_lg10(tempbb * 50. / xmin) / .02)), ne = jmaxth - 2;
  for (int j = tid; j <= NTH_N; j += NTH_THREADS) s_x[j] = xmin * pow(10., j * .02);
  __syncthreads();
  double *x = tab, *w1o = tab + NTH_N + 1, *c2 = w1o + NTH_N, *x3 = c2 + NTH_N, *relo = x3 + NTH_N,
         *dph = relo + NTH_N;
  for (int j = tid; j < NTH_N; j += NTH_THREADS) {
    const double w = s_x[j];
    const double w1 = sqrt(s_x[j] * s_x[j + 1]);
    w1o[j] = w1;
    c2[j] = pow(w1, 4.) / (w1 * 4.6 + 1. + w1 * 1.1 * w1);
    x3[j] = pow(w, 3.);
    double rel;
    if (w <= .05) {
      rel = 1 - w * 2 + w * 26 * w / 5;
    } else {
      const double z1 = (w + 1) / (w * (w * w));
      const double z2 = w * 2 + 1;
      const double z3 = log(z2);
      const double z4 = w * 2 * (w + 1) / z2;
      const double z5 = z3 / 2 / w;
      const double z6 = (w * 3 + 1) / z2 / z2;
      rel = (z1 * (z4 - z3) + z5 - z6) * .75;
    }
    relo[j] = rel;
    s_a[j] = w1 * 511.;  // seed bin centres
    s_ph[j] = 0.0;
  }
  for (int j = tid; j <= NTH_N; j += NTH_THREADS) x[j] = s_x[j];
  __syncthreads();
  const double tin = tempbb * 511.;
  for (int i = 1 + tid; i <= ne; i += NTH_THREADS) {
    const double xn = (s_a[i] - s_a[i - 1]) / 2.0;
    const double xh = xn + s_a[i - 1];
    double ph = 0.0;
    for (int k = 0; k < 5; k++) {
      const double e = xn * c_gl_x[k] + xh;
      ph += c_gl_w[k] * (nth_mcd_shape(e / tin) * tin * tin * 1. / 361.);
    }
    s_b[i - 1] = ph * xn;
  }
  __syncthreads();
  for (int j = 1 + tid; j <= ne; j += NTH_THREADS) s_ph[j] = s_b[j - 1] * 511. / (s_a[j] - s_a[j - 1]);
  __syncthreads();
  for (int j = tid; j < NTH_N; j += NTH_THREADS) dph[j] = s_ph[j == 0 ? 1 : j];
}

// One Kompaneets solve per workgroup, written to HBM as (x, E F_E, jmax).
__global__ __launch_bounds__(NTH_THREADS) void k_nthcomp(const NthJob *__restrict__ jobs, const double *__restrict__ tab,
                                                         double *__restrict__ sol_x,
                                                         double *__restrict__ sol_s, int *__restrict__ sol_n) {
  __shared__ NthLds L;
  const int tid = threadIdx.x;
  const NthJob jb = jobs[blockIdx.x];
  const int jmax = nth_solve(L, nth_grid_tab(tab), jb.kte, jb.gam, tid, NTH_THREADS);
  double *xo = sol_x + (size_t)blockIdx.x * (NTH_N + 1);
  double *so = sol_s + (size_t)blockIdx.x * NTH_N;
  for (int j = tid; j <= jmax; j += NTH_THREADS) xo[j] = L.x[j];
  for (int j = tid; j < NTH_N; j += NTH_THREADS) so[j] = L.t1[j];
  if (tid == 0) sol_n[blockIdx.x] = jmax;
}

__global__ __launch_bounds__(NTH_THREADS) void k_nthcomp_bins(const double *__restrict__ ener, int n,
                                                              const double *__restrict__ shift,
                                                              const double *__restrict__ sol_x,
                                                              const double *__restrict__ sol_s,
                                                              const int *__restrict__ sol_n, double *__restrict__ out) {
#pragma clang fp contract(off)
  const int s = blockIdx.x;
  const double *x = sol_x + (size_t)s * (NTH_N + 1);
  const double *spt = sol_s + (size_t)s * NTH_N;
  const int nth = sol_n[s];
  const double z = 1 / shift[s] - 1;
  const double normfac = nthcomp_normfac(x, spt, nth, z);
  for (int i = threadIdx.x; i < n; i += NTH_THREADS) {
    const double p0 = nthcomp_edge(x, spt, nth, ener[i], z);
    const double p1 = nthcomp_edge(x, spt, nth, ener[i + 1], z);
    out[(size_t)s * n + i] = nthcomp_bin(ener[i], ener[i + 1], p0, p1, normfac);
  }
}

}  // namespace

size_t nth_grid_bytes() { return sizeof(double) * NTH_GRID_DOUBLES; }

int launch_nth_grid(double *tab, void *stream) {
  hipLaunchKernelGGL(k_nth_grid, dim3(1), dim3(NTH_THREADS), 0, (hipStream_t)stream, tab);
  return (int)hipGetLastError();
}

int launch_nthcomp(const NthJob *jobs, int n_jobs, const double *tab, double *sol_x, double *sol_s, int *sol_n, void *stream) {
  if (n_jobs <= 0) return 0;
  hipLaunchKernelGGL(k_nthcomp, dim3(n_jobs), dim3(NTH_THREADS), 0, (hipStream_t)stream, jobs, tab, sol_x, sol_s,
                     sol_n);
  return (int)hipGetLastError();
}

// rx_nthcomp: n_spec spectra on one caller grid (host arrays in and out).
int nthcomp_spectra(const double *ener, int n_flux, int n_spec, const double *kte, const double *gam,
                    const double *ener_shift, double *flux, std::string &err) {
  for (int s = 0; s < n_spec; s++) {
    // the solve's grid needs kTe well above the seed and a finite Thomson depth
    if (!(kte[s] >= 0.1 && kte[s] <= 1e4) || !(gam[s] > 1.0 && gam[s] < 10.0) ||
        !(ener_shift[s] > 0.0 && ener_shift[s] < 1e3)) {
      err = "nthcomp parameters out of range (kTe 0.1-1e4 keV, 1 < Gamma < 10, energy shift > 0)";
      return RX_ERR_ARG;
    }
  }
  for (int k = 0; k < n_flux; k++)
    if (!(ener[k + 1] > ener[k]) || !(ener[k] > 0.0)) {
      err = "energy grid must be positive and ascending";
      return RX_ERR_ARG;
    }
  std::vector<NthJob> jobs(n_spec);
  for (int s = 0; s < n_spec; s++) jobs[s] = NthJob{kte[s], gam[s]};
  DevBuf d_jobs, d_e, d_shift, d_x, d_s, d_n, d_out;
  if (d_jobs.ensure(sizeof(NthJob) * n_spec) || d_e.ensure(sizeof(double) * (n_flux + 1)) ||
      d_shift.ensure(sizeof(double) * n_spec) || d_x.ensure(sizeof(double) * (NTH_N + 1) * n_spec) ||
      d_s.ensure(sizeof(double) * NTH_N * n_spec) || d_n.ensure(sizeof(int) * n_spec) ||
      d_out.ensure(sizeof(double) * (size_t)n_flux * n_spec)) {
    err = "device allocation failed";
    return RX_ERR_NOMEM;
  }
  int e = (int)hipMemcpy(d_jobs.p, jobs.data(), sizeof(NthJob) * n_spec, hipMemcpyHostToDevice);
  e |= (int)hipMemcpy(d_e.p, ener, sizeof(double) * (n_flux + 1), hipMemcpyHostToDevice);
  e |= (int)hipMemcpy(d_shift.p, ener_shift, sizeof(double) * n_spec, hipMemcpyHostToDevice);
  e |= launch_nthcomp(d_jobs.as<NthJob>(), n_spec, G().nth_grid.as<double>(), d_x.as<double>(), d_s.as<double>(), d_n.as<int>(), nullptr);
  hipLaunchKernelGGL(k_nthcomp_bins, dim3(n_spec), dim3(NTH_THREADS), 0, nullptr, d_e.as<double>(), n_flux,
                     d_shift.as<double>(), d_x.as<double>(), d_s.as<double>(), d_n.as<int>(), d_out.as<double>());
  e |= (int)hipGetLastError();
  e |= (int)hipMemcpy(flux, d_out.p, sizeof(double) * (size_t)n_flux * n_spec, hipMemcpyDeviceToHost);
  if (e) {
    (void)hipGetLastError();
    err = "device error in the nthcomp kernels";
    return RX_ERR_DEVICE;
  }
  return RX_OK;
}

}  // namespace rx
