// engine.h -- host runtime of librelxill_gpu (internal).
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/relxill_gpu.h"
#include "rx_engine.h"
#include "rx_math.h"
#include "rx_tables.h"

namespace rx {

struct DevBuf {
  void *p = nullptr;
  size_t bytes = 0;
  ~DevBuf();
  int ensure(size_t n);  // grows (never shrinks); returns hipError_t
  template <class T>
  T *as() const { return reinterpret_cast<T *>(p); }
};

// Pinned host memory that kernels and copies on a stream read or write.
struct PinnedBuf {
  void *p = nullptr;
  size_t bytes = 0;
  ~PinnedBuf();
  bool ensure(size_t n);  // grows (never shrinks)
  template <class T>
  T *as() const { return reinterpret_cast<T *>(p); }
};

// Host mirror of get_rel_params + check_parameter_bounds
// (src/ModelDefinition.cpp:153-334) for one request.  Returns RX_OK or a status.
// prim: the primary continuum of the relxill models (PRIM_*)
int parse_request(int model, const double *par, bool phys_norm, ReqParams &p, std::string &err,
                  int prim = PRIM_CUTOFFPL);
// relxill requests: the xillver table corner and factors of the request's
// parameters (get_xilltab_indices_for_paramvals and interp_xill_table,
// src/xilltable.c:297-324, :1090-1125).
// ind / fac: the four inner axes.  The xillver models interpolate the
// inclination too (clamped into the table like the others): clamp_incl, and
// its bracket and factor in *inc_ind / *inc_fac.  A six-parameter table's
// first axis (interpolated outside the others) goes to *out_ind / *out_fac
// (0 and 0 for five parameters).
void xill_corner(const XillTableHost &t, double gam, double afe, double lxi, double ect, double dens, double ktbb,
                 double incl_deg, int *ind, double *fac, bool clamp_incl = false, int *inc_ind = nullptr,
                 double *inc_fac = nullptr, int *out_ind = nullptr, double *out_fac = nullptr);
int n_model_params(int model);
// Edges of the radial zones (RadialGrid::calculate_radial_grid, src/IonGradient.cpp:457-489).
void rzone_grid(double rmin, double rmax, int nzones, double h, double *rgrid);

// The work lists of a batch's kernels (device pointers and lengths).
struct WorkLists {
  const XillWork *xill, *conv, *zone, *nth;
  const int *prim, *ang, *rrc, *rrad;
  int n_xill1, n_xill, n_conv, n_zone, n_nth, n_prim, n_prim_rel, n_ang, n_rrc, n_rrad;
};

// Launch configuration of one run: every kernel argument and grid shape.  A
// run whose configuration equals the previous run's is captured into a
// hipGraph, which is replayed for as long as the configuration stays equal
// (the kernels read the batch's data through the same pointers).  Built with
// its padding zeroed, so configurations compare with memcmp.
struct RunKey {
  BatchDev bd;
  WorkLists wl;
  int n_blocks, prim_bins;
  int prof, cos_rows, finalize, angular, one_unit;
  // the request block fetched from pinned host memory at the start of the run
  // (n_fetch 16-byte words; 0: it is on the device) and the results delivered
  // there at its end (n_out output values; 0: statuses and counters only)
  const void *fetch_src;
  void *fetch_dst;
  int64_t n_fetch;
  void *res, *res_out;
  int64_t n_out;
};

// Request blocks up to STAGE_MAX go to the device through pinned memory in one
// piece; larger ones piece by piece from the batch's own arrays, a copy less.
constexpr size_t STAGE_MAX = 4u << 20;
// What a server slot's batch takes at least.  Growing frees memory, which waits for
// the other slots' batches, and allocates anew: 250 us for 2 MB and more, device or
// pinned, 1-60 us below that.  So its device allocation is SLOT_RESERVE at once (a
// slot's share of the server's budget at most: Batch::reserve), its other pieces are
// just below 2 MB, and its pinned request block is that or, for larger requests,
// STAGE_MAX.  Bursts of 8 / 32 / 64 / 128 requests at a new server, the first / second
// / third of them in ms: 0.7 0.3 0.3 / 1.0 0.7 0.7 / 1.5 1.2 1.2 / 3.8 2.3 2.0; with
// every piece grown to what the batch at hand takes 1.3 0.9 0.5 / 2.0 1.5 0.7 / 2.8 2.8
// 2.2 / 6.2 6.5 4.7.
constexpr size_t SLOT_RESERVE = 16u << 20, SLOT_SMALL = 1900u << 10;

struct Batch {
  int n_req = 0;
  int max_zones = 1;          // most zones of a request
  int seg_bins = 64;        // bins per work item
  int seg_forced = 0;       // 0: automatic / autotuned
  int waves_per_cu = 12;    // persistent integration wavefronts per CU
  int waves_forced = 0;
  std::vector<ReqParams> h_req;
  std::vector<int> h_status;  // host-side parse status
  std::vector<double> h_ener, h_flux_in;
  std::vector<int> h_prim;       // requests with a primary: n_prim_rel relxill ones, then the xillver models
  int n_prim_rel = 0;
  int prim_bins = 0;             // most caller bins of a request in h_prim
  std::vector<int> h_ang;        // requests with an emission-angle distribution (k_dist)
  std::vector<XillWork> h_conv;  // (request, zone) units of k_conv
  std::vector<XillWork> h_xill;  // k_xill units: one-zone requests first, then the others (all zones in one unit)
  int n_xill1 = 0;               // number of one-zone units at the front of h_xill
  std::vector<int> h_rrc;        // requests with returning-radiation corrections (k_before_rrad)
  std::vector<int> h_rrad;       // requests with returning radiation (k_rrad)
  std::vector<XillWork> h_zone;  // (request, zone) units of k_zone (relxill and xillver models)
  std::vector<XillWork> h_nth;   // nthcomp solves: (request, 0 source / 1 + zone)
  int n_nth_sol = 0;             // requests with the nthcomp primary (one source solution each)
  int64_t tot_ener = 0, tot_flux = 0, tot_pgrid = 0, tot_prof = 0, tot_xspec = 0, tot_dist = 0, tot_zone = 0;
  int64_t tot_rrc = 0;
  // One device allocation holds everything of the batch; it begins with the
  // request block (what the host writes: parameters, statuses, work lists, grids,
  // input spectra) and ends with k_integrate's work list as the batch was built.  A
  // work shape set later whose list is longer has it in an allocation of its own, so
  // that the last run's outputs, distributions, zones and statuses stay where they
  // are.
  DevBuf d_arena, d_items;
  int arena_items = 0;        // items that the first one's list takes
  size_t arena_items_at = 0;  // its offset
  bool ready = false;  // what the batch needs is there and laid out
  size_t reserve = 0;  // a server slot: least bytes of d_arena (SLOT_RESERVE)
  BatchDev dev;   // its pointers (dev_view adds the run's settings and the tables)
  WorkLists wl;
  size_t block_bytes = 0;
  struct BlockOffsets {
    size_t req, status, conv, xill, prim, zone, ang, rrc, rrad, nth, ener, flux;
  } off;
  bool staged = false;  // the block fits the pinned memory
  double *p_ener = nullptr, *p_flux = nullptr;  // grids and inputs on the host (pinned memory or h_ener, h_flux_in)
  // The request block in pinned memory (batches that are built again and again
  // keep their own, others use the library's while they are built), the run's
  // results (result_*).
  bool keep_stage = false;
  PinnedBuf h_stage, h_res;
  // an evaluation call: the run fetches the request block and delivers the
  // outputs itself (call_run: this one does)
  bool is_call = false, call_run = false;
  int64_t deliver_out = 0;  // output values that a run delivers to h_res
  // outputs read ahead by rx_batch_output: two pinned windows of the output
  // array, filled in turn
  struct OutWindow {
    int64_t lo = 0, hi = 0;  // values [lo, hi) of the output array
    bool pending = false;    // its copy is on the stream
    PinnedBuf buf;
  };
  OutWindow win[2];
  int win_cur = 0;
  int64_t win_next = -1, win_len = 0;  // end of the last read; length of the last window
  std::atomic<bool> synced{true};      // the stream was waited for since the last run
  std::mutex out_mu;                   // readers of one batch in several threads
  int item_cap = 0;
  // the work shape of the last evaluation call and what it was chosen for
  struct CallShape {
    int64_t windows, max_bins, window_bins;
    int seg_bins;
    int64_t item_cap;
  } call_shape = {};
  int n_blocks = 1;  // workgroups of k_integrate
  bool any_cosne = false, any_limb = false, any_angular = false;
  bool one_unit = false;  // every request has one unit of k_conv
  bool any_flux = false;  // some request has an input spectrum
  int fix_cap = 0;
  int last_mode = 1;
  bool fix_overflow = false;
  hipStream_t stream = nullptr;
  hipEvent_t ev[RX_N_TIMED + 1] = {};
  bool profiled = false;
  double kernel_ms[RX_N_TIMED] = {};
  int64_t counters[3] = {};  // items, FP64 re-checks, re-check overflow (last run)
  int shape_class = 0;
  uint64_t config_gen = 0;  // Global::config_gen at build time
  // graph of the launch sequence (captured on the second identical run)
  RunKey last_key, graph_key;
  bool last_valid = false, graph_failed = false;
  // one-shot batches (the server's slots: every run carries new requests)
  // never capture a launch graph, whose capture would cost more than it saves
  bool one_shot = false;
  hipGraph_t graph = nullptr;
  hipGraphExec_t gexec = nullptr;
  int64_t graph_replays = 0;
  ~Batch();
};

// Fills b (re-using device buffers when large enough) from the requests.
int batch_build(Batch &b, const rx_request *req, int n_req, std::string &err);
// Chooses the work-item segment length and the persistent wavefronts per CU
// (0: automatic / autotuned) and sizes the work list.
void batch_plan(Batch &b, int seg_bins, int waves_per_cu);
// Bins of an energy grid (n + 1 ascending edges) that the window of some radius of
// the resident table can reach; unit: the grid's energy of g = 1.
int reach_bins(const double *ener, int n, double unit);
// Default work shape of a batch: windows (radius chunk x zone, over all requests),
// the most bins of a profile grid, and the bins that the windows together can
// reach (reach_bins of a request times its windows).
struct WorkShape {
  int seg_bins, waves_per_cu;
};
WorkShape work_shape(int64_t windows, int max_bins, int64_t window_bins);
WorkShape batch_default_shape(const Batch &b);  // of a built batch
// Workgroups of k_integrate for a work list of that capacity: one an item for
// lists of up to ONE_ITEMS.
constexpr int ONE_ITEMS = 1 << 18;
int integrate_blocks(int item_cap, int64_t windows, int waves_per_cu);
int batch_upload(Batch &b);
// Sizes the work list for the batch's work shape (batch_plan).
int batch_place_items(Batch &b);
// Layout of a run's results in pinned host memory: the first RES_CTR counters,
// the statuses, the outputs.
inline int *result_ctr(const Batch &b) { return b.h_res.as<int>(); }
inline int *result_status(const Batch &b) { return b.h_res.as<int>() + RES_CTR; }
inline size_t result_out_offset(int n_req) { return (sizeof(int) * (RES_CTR + (size_t)n_req) + 255) & ~(size_t)255; }
inline double *result_out(const Batch &b) {
  return reinterpret_cast<double *>(b.h_res.as<char>() + result_out_offset(b.n_req));
}
// Copies n output values from off on (after the run's end) to host memory.
int batch_read(Batch &b, int64_t off, int64_t n, double *to);
int batch_run(Batch &b, int precision, std::string &err);
int batch_sync(Batch &b);
// Public status of a request from its device status.
int public_status(int dev_status);

// One resident xillver table: the host table, why a table named by
// RELXILL_TABLE_PATH could not be loaded (empty: loaded), its energy edges
// (elo, then the last ehi) and the device copies (renormalised spectra,
// edges, the Ecut / kTe axis, the axis ensure_ecut_within_boundarys reads, the
// inclinations).
struct XillSlot {
  XillTableHost t;
  bool loaded = false, dirty = true;
  std::string err;
  std::vector<double> ener;
  double rr_lo = 1e300, rr_hi = -1e300;  // DevXillTable's
  DevBuf spec, d_ener, ect, q, incl, lxi;
};

// global state
struct Global {
  std::recursive_mutex mu;
  bool device_ready = false;
  int device = 0;
  int n_cu = 256;
  RelTableHost rel;
  LpTableHost lp;
  bool rel_loaded = false, lp_loaded = false;
  // why a table named by RELXILL_TABLE_PATH could not be loaded (empty: loaded)
  std::string rel_err, lp_err, rrad_err;
  bool rel_dirty = true, lp_dirty = true;
  double rel_gmin_all = 0.0, rel_gmax_all = 1e30;  // g range reachable by any window
  DevBuf t_a, t_mu0, t_r, t_gmin, t_gmax, t_trff1, t_trff2, t_cosne1, t_cosne2;
  DevBuf l_a, l_h, l_rad, l_int, l_del, l_inc;
  // xillver tables, one per primary continuum (PRIM_*: xillver-a-Ec5.fits for
  // the cut-off power law, xillverCp_v3.4.fits for nthcomp, xillverNS-2.fits
  // for the blackbody, src/common.h:163-167;
  // loaded and uploaded on the first relxill request that needs one)
  XillSlot xill[N_PRIM];
  // returning-radiation table (loaded and uploaded on the first request with it)
  RradTableHost rrad;
  bool rrad_loaded = false, rrad_dirty = true;
  PinnedBuf stage;  // request block of the batch being built (under mu)
  DevBuf nth_grid;  // what all nthcomp solves share
  bool nth_grid_ready = false;
  DevBuf r_rlo, r_rhi, r_tf, r_gmin, r_gmax, r_fg;
  // convolution grid
  int conv_n = 4096;
  double conv_emin = 0.00035, conv_emax = 2000.0;
  std::vector<double> conv_ener, conv_cfac, conv_cfinv, conv_inv_emid, conv_tw, conv_twp_fwd, conv_twp_inv;
  int conv_i1kev = 0;
  int conv_band_lo = 0, conv_band_hi = 0;
  bool conv_dirty = true;
  std::vector<double> coarse_ener, coarse_ln, conv_ln_emid;
  DevBuf c_coarse, c_coarse_ln, c_ln_emid;
  DevBuf c_ener, c_cfac, c_cfinv, c_inv_emid, c_tw, c_twp_fwd, c_twp_inv;
  int nr_fine = 1000;
  // reflection sets
  std::vector<DevReflSet> refl_sets;
  std::vector<DevBuf *> refl_bufs;
  DevBuf d_refl_sets;
  bool refl_dirty = false;
  bool profile = false;
  bool use_graphs = true;  // replay repeated launch sequences as hipGraphs
  // bumped by every change that invalidates built batches (tables, conv grid,
  // fine-grid size, clearing reflection sets); a batch refuses to run on a
  // newer configuration than it was built for
  uint64_t config_gen = 1;
  float guard = ROMB_GUARD;
  // autotune cache: shape class -> (segment bins, waves per CU)
  struct Tuned {
    int shape, seg_bins, waves_per_cu;
  };
  std::vector<Tuned> tune;
};

Global &G();
void ensure_tables_host();
int ensure_device(std::string &err);  // device + uploads (tables, conv grid, refl sets)
// rx_nthcomp: n_spec nthcomp spectra on one caller grid (host arrays)
int nthcomp_spectra(const double *ener, int n_flux, int n_spec, const double *kte, const double *gam,
                    const double *ener_shift, double *flux, std::string &err);
void ensure_xilltable_host(int prim);
void ensure_rradtable_host();
int ensure_rradtable_device(std::string &err);
// the returning-radiation table zones of an LP request (select_spinIndexForTable
// and allocate_radial_grid, src/Relreturn_Table.cpp:343-404); a status != 0 if
// the table does not cover the disk
int rrad_zones(const RradTableHost &t, ReqParams &p, int nr_fine);
int ensure_xilltable_device(int prim, std::string &err);
void fill_dev_views(BatchDev &bd);
void set_last(int status, const std::string &msg);
// the same with a static message (no allocation)
void set_last_static(int status, const char *msg);
// Looks up the device address of the allocation-free entry point's scratch
// array on `device` (current) once (noalloc.hip).
int noalloc_setup(int device, std::string &err);
int last_status();
const char *last_error();
bool phys_norm_env();

}  // namespace rx
