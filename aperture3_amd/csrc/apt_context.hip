// apt_context.hip -- the C ABI (include/aperture_amd.h): context lifetime,
// device memory, host<->device transfers and the step sequencing of
// ptc_updater::update_particles (ptc_updater.cu:748-841) and
// field_solver::update_fields (field_solver.cu:334-358).  All work is
// enqueued on the context's stream; nothing inside a step reads a count
// back to the host.
#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/aperture_amd.h"
#include "apt_common.hpp"
#include "apt_kernels.hpp"
#include "apt_math.hpp"
#include "apt_sort.hpp"
#include "apt_tiles.hpp"

using namespace apt;

struct EventPair {
  hipEvent_t a, b;
};

struct apt_ctx {
  apt_grid grid;
  int device = 0;  // the device current at apt_create
  apt_params params;
  Mesh mesh;
  Species sp;
  hipStream_t stream = nullptr;
  int prec = APT_PREC_FP64;
  uint64_t ncell = 0;

  // fields (double* in the FP64 form, float* in the mixed form)
  void *E[3] = {}, *B[3] = {}, *Ebg[3] = {}, *Bbg[3] = {}, *J[3] = {};
  void *Rho[4] = {}, *divE = nullptr, *divB = nullptr, *jtmp = nullptr;
  void *ftmp[3] = {};  // with jtmp, a filter pass's other arrays (smoothed boxes)
  // Cartesian steps: the background fields hold what apt_create wrote (zeros),
  // and Rho holds zeros
  bool ebg_zero = true, bbg_zero = true, rho_zero = true;
  // sim_data::EdotB, photon_produced, pair_produced (sim_data.h:57-59)
  void *EdotB = nullptr, *ph_produced = nullptr, *pair_produced = nullptr;
  // collect_diagnostics moments, allocated on the first collection
  void *diag_num[4] = {}, *diag_gamma[4] = {}, *diag_ph = nullptr;
  long long *Jacc[3][2] = {};
  long long *Racc[4][2] = {};

  // particles (double buffered for the sort gather)
  uint64_t cap = 0, number = 0;
  PtcF64 p64{}, p64b{};
  PtcF32 p32{}, p32b{};
  bool have_b = false;
  unsigned long long *d_counters = nullptr;
  // Gauss-law residual: partial maxima (2 per block) and, once asked for,
  // the residual field in FP64
  double *divres_part = nullptr;
  double *divres_field = nullptr;
  SortWork sortw;

  double wmax = 1.0;  // max |q w| over particles, sets the fixed-point scale
  int H = 22;

  // mixed-form tiling
  uint32_t *tile_off = nullptr;
  TileInfo tiles{};
  bool tiling = false;       // shape set up for this mesh
  bool tiles_valid = false;  // particles are binned by tile
  uint32_t pushes_since_sort = 0;  // eager tiled pushes since the binning
  // 3D, shape not named by the caller: a small halo while the drift of light
  // since the binning, in cells, is small (see setup_tiles)
  bool tiles_by_drift = false;
  double drift = 0.0;
  TileSortWork tsort;

  // runs of cell-sorted slots by tile (Cartesian FP64 and untiled mixed, 2D
  // log-spherical): built by a sort, valid until the slots below runs.end are
  // replaced
  uint32_t *run_off = nullptr;
  CellRuns runs{};
  bool runs_valid = false;

  // log-spherical path
  bool logsph = false;
  // 1D GR gap (Grid_1dGR): coefficient arrays on the device and their host
  // copy, and the reference's float parameters a, omega, B0, track_percent
  bool gr1d = false;
  double *gr_dev[GR_NCOEF] = {};
  std::vector<double> gr_host[GR_NCOEF];
  float gr_a = 0.0f, gr_omega = 0.0f, gr_B0 = 0.0f, gr_track = 0.0f;
  // 1D pulsar gap (labs/1dgap): beta_phi(x) = x, the reference's float
  // B0, omega and track_percent
  bool gap1d = false;
  float gap_B0 = 0.0f, gap_omega = 0.0f, gap_track = 0.0f;
  LsParams lp{};
  LsCoef coef{};
  double *coef_mem[LS_NCOEF] = {};
  long long *surf = nullptr;  // 4 N1 int64: surface density e-, ion (2 limbs)
  uint32_t inject_epoch = 0;
  double wmaxw = 1.0;  // largest particle weight: surface-density scale

  // force-free / vacuum solver scratch (3D log-spherical contexts)
  void *ffe[12] = {};  // En[3], Bn[3], dE[3], dB[3]
  // 3D Cartesian force-free solver: the work fields m_Etmp[3], m_Btmp[3]
  // and a scalar work field, then a copy of E_in when E_out is E_in
  void *ffc[10] = {};

  // photons and pair creation
  RtParams rt{};
  RtWork rtw;
  uint32_t rt_epoch = 0;
  uint64_t ph_cap = 0, ph_number = 0;
  PhoF64 ph64{}, ph64b{};
  PhoF32 ph32{}, ph32b{};
  bool ph_have_b = false;
  uint64_t id_next = 0, ph_id_next = 0;

  // device-count mode (apt_set_device_counts, log-spherical contexts): the
  // exact counts, ids, epochs and event totals live in d_dc; number and
  // ph_number above are then upper bounds that size launches, and every
  // slot from a count up to the capacity is empty
  bool dcount = false;
  unsigned long long *d_dc = nullptr;
  // a step recorded by apt_graph_begin / apt_graph_end, replayed by
  // apt_graph_launch
  bool capturing = false;
  bool timing_saved = false;
  hipGraphExec_t gexec = nullptr;

  std::string err;
  bool timing = false;
  std::vector<EventPair> ev[APT_KERNEL_NUM];
  size_t ev_used[APT_KERNEL_NUM] = {};

  apt_status fail(apt_status code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    err = buf;
    return code;
  }
  size_t esize() const { return prec == APT_PREC_FP64 ? 8 : 4; }
};

#define HIPCHK(call)                                                    \
  do {                                                                  \
    hipError_t e_ = (call);                                             \
    if (e_ != hipSuccess)                                               \
      return ctx->fail(APT_ERR_HIP, "%s: %s", #call, hipGetErrorString(e_)); \
  } while (0)

static uint32_t *ptc_cells(apt_ctx *ctx) {
  return ctx->prec == APT_PREC_FP64 ? ctx->p64.cell : ctx->p32.cell;
}
static uint32_t *ph_cells(apt_ctx *ctx) {
  return ctx->prec == APT_PREC_FP64 ? ctx->ph64.cell : ctx->ph32.cell;
}

// Device-count mode: the exact counts, ids and epochs back on the host (a
// synchronisation); the host bounds become exact.
static apt_status exact_counts(apt_ctx *ctx) {
  if (!ctx->dcount) return APT_OK;
  if (ctx->capturing)
    return ctx->fail(APT_ERR_STATE, "the counts cannot be read while a step is recorded");
  unsigned long long h[DC_N];
  HIPCHK(hipMemcpyAsync(h, ctx->d_dc, sizeof(h), hipMemcpyDeviceToHost, ctx->stream));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  ctx->number = h[DC_NUM];
  ctx->ph_number = h[DC_PH];
  ctx->id_next = h[DC_ID];
  ctx->ph_id_next = h[DC_PH_ID];
  ctx->rt_epoch = (uint32_t)h[DC_RT_EPOCH];
  ctx->inject_epoch = (uint32_t)h[DC_INJ_EPOCH];
  return APT_OK;
}

// Device-count mode: counts the host has just set (uploads, restarts)
// written to the device, event totals kept.
static apt_status push_counts(apt_ctx *ctx) {
  if (!ctx->dcount) return APT_OK;
  unsigned long long h[DC_N];
  HIPCHK(hipMemcpyAsync(h, ctx->d_dc, sizeof(h), hipMemcpyDeviceToHost, ctx->stream));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  h[DC_NUM] = ctx->number;
  h[DC_PH] = ctx->ph_number;
  h[DC_ID] = ctx->id_next;
  h[DC_PH_ID] = ctx->ph_id_next;
  h[DC_RT_EPOCH] = ctx->rt_epoch;
  h[DC_INJ_EPOCH] = ctx->inject_epoch;
  HIPCHK(hipMemcpyAsync(ctx->d_dc, h, sizeof(h), hipMemcpyHostToDevice, ctx->stream));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  return APT_OK;
}

#define CHECK_CTX(ctx) \
  do {                 \
    if (!(ctx)) return APT_ERR_INVALID_ARG; \
  } while (0)

static int ceil_log2(double x) {
  int e = 0;
  double v = 1.0;
  while (v < x && e < 60) {
    v *= 2.0;
    e++;
  }
  while (v / 2.0 >= x && e > -60) {
    v /= 2.0;
    e--;
  }
  return e;
}

// fixed-point exponent for the current from the largest |q w|: FP64 keeps
// |J| < 2^41 wmax in the high limb; the mixed form rounds every
// contribution (|c| <= |q w|) to an int32 multiple of 2^-H, H = 30 - e,
// and sums in int64, so |J| < 2^33 wmax.
static void update_scale(apt_ctx *ctx) {
  int e = ceil_log2(ctx->wmax > 0 ? ctx->wmax : 1.0);
  ctx->H = (ctx->prec == APT_PREC_FP64) ? 22 - e : 30 - e;
}

// surface-density fixed point (injection gate): 2^-Hs with the largest
// particle weight below 2^(22-Hs)
static int surface_scale(const apt_ctx *ctx) {
  return 22 - ceil_log2(ctx->wmaxw > 1.0 ? ctx->wmaxw : 1.0);
}

static apt_status alloc_ptc(apt_ctx *ctx, bool second) {
  uint64_t n = ctx->cap;
  if (ctx->prec == APT_PREC_FP64) {
    PtcF64 &p = second ? ctx->p64b : ctx->p64;
    HIPCHK(hipMalloc(&p.cell, n * 4));
    HIPCHK(hipMalloc(&p.x1, n * 8));
    HIPCHK(hipMalloc(&p.x2, n * 8));
    HIPCHK(hipMalloc(&p.x3, n * 8));
    HIPCHK(hipMalloc(&p.p1, n * 8));
    HIPCHK(hipMalloc(&p.p2, n * 8));
    HIPCHK(hipMalloc(&p.p3, n * 8));
    HIPCHK(hipMalloc(&p.E, n * 8));
    HIPCHK(hipMalloc(&p.w, n * 8));
    HIPCHK(hipMalloc(&p.flag, n * 4));
    HIPCHK(hipMalloc(&p.id, n * 8));
    HIPCHK(launch_fill<uint32_t>(p.cell, MAX_CELL, n, ctx->stream));
  } else {
    PtcF32 &p = second ? ctx->p32b : ctx->p32;
    HIPCHK(hipMalloc(&p.cell, n * 4));
    HIPCHK(hipMalloc(&p.x1, n * 4));
    HIPCHK(hipMalloc(&p.x2, n * 4));
    HIPCHK(hipMalloc(&p.x3, n * 4));
    HIPCHK(hipMalloc(&p.u1, n * 4));
    HIPCHK(hipMalloc(&p.u2, n * 4));
    HIPCHK(hipMalloc(&p.u3, n * 4));
    HIPCHK(hipMalloc(&p.w, n * 4));
    HIPCHK(hipMalloc(&p.flag, n * 4));
    HIPCHK(launch_fill<uint32_t>(p.cell, MAX_CELL, n, ctx->stream));
  }
  return APT_OK;
}

static void drop_ftmp(apt_ctx *ctx) {
  for (void *&q : ctx->ftmp) {
    (void)hipFree(q);
    q = nullptr;
  }
  (void)hipGetLastError();  // of the allocation that did not fit
}

// Memory that the context can do without, given back for an allocation that did
// not fit: the sort's scratch, which may hold more room than is needed, and the
// smoothing's work arrays, unless a recorded step holds them.
static apt_status give_back(apt_ctx *ctx) {
  HIPCHK(hipStreamSynchronize(ctx->stream));
  ctx->sortw.release();
  if (!ctx->gexec && !ctx->capturing) drop_ftmp(ctx);
  return APT_OK;
}

static void free_ptc64(PtcF64 &p) {
  (void)hipFree(p.cell); (void)hipFree(p.x1); (void)hipFree(p.x2); (void)hipFree(p.x3);
  (void)hipFree(p.p1); (void)hipFree(p.p2); (void)hipFree(p.p3); (void)hipFree(p.E); (void)hipFree(p.w);
  (void)hipFree(p.flag); (void)hipFree(p.id);
  p = PtcF64{};
}
static void free_ptc32(PtcF32 &p) {
  (void)hipFree(p.cell); (void)hipFree(p.x1); (void)hipFree(p.x2); (void)hipFree(p.x3);
  (void)hipFree(p.u1); (void)hipFree(p.u2); (void)hipFree(p.u3); (void)hipFree(p.w);
  (void)hipFree(p.flag);
  p = PtcF32{};
}

static apt_status alloc_photons(apt_ctx *ctx, bool second) {
  uint64_t n = ctx->ph_cap;
  if (ctx->prec == APT_PREC_FP64) {
    PhoF64 &p = second ? ctx->ph64b : ctx->ph64;
    HIPCHK(hipMalloc(&p.cell, n * 4));
    double **d[] = {&p.x1, &p.x2, &p.x3, &p.p1, &p.p2, &p.p3, &p.E, &p.w, &p.path};
    for (double **q : d) HIPCHK(hipMalloc(q, n * 8));
    HIPCHK(hipMalloc(&p.flag, n * 4));
    HIPCHK(hipMalloc(&p.id, n * 8));
    HIPCHK(launch_fill<uint32_t>(p.cell, MAX_CELL, n, ctx->stream));
  } else {
    PhoF32 &p = second ? ctx->ph32b : ctx->ph32;
    HIPCHK(hipMalloc(&p.cell, n * 4));
    float **d[] = {&p.x1, &p.x2, &p.x3, &p.p1, &p.p2, &p.p3, &p.w, &p.path};
    for (float **q : d) HIPCHK(hipMalloc(q, n * 4));
    HIPCHK(hipMalloc(&p.flag, n * 4));
    HIPCHK(launch_fill<uint32_t>(p.cell, MAX_CELL, n, ctx->stream));
  }
  return APT_OK;
}

static void free_ph64(PhoF64 &p) {
  void *a[] = {p.cell, p.x1, p.x2, p.x3, p.p1, p.p2, p.p3, p.E, p.w, p.path, p.flag, p.id};
  for (void *q : a) (void)hipFree(q);
  p = PhoF64{};
}
static void free_ph32(PhoF32 &p) {
  void *a[] = {p.cell, p.x1, p.x2, p.x3, p.p1, p.p2, p.p3, p.w, p.path, p.flag};
  for (void *q : a) (void)hipFree(q);
  p = PhoF32{};
}

// no guard cells along an axis that the mesh does not have (the updates of such a
// mesh differ in the rows and planes beside it that they read)
static bool no_idle_guards(const Mesh &m) {
  for (int d = m.dim; d < 3; d++)
    if (m.dims[d] != 1) return false;
  return true;
}

// Tiling of the mixed form: every tiled dimension periodic; an axis whose N
// is not a multiple of the tile extent is split evenly over ceil(N / extent)
// tiles.  (Before, such a mesh took the untiled push with one HBM atomic per
// contribution: 1000 x 505 cells at 16 particles per cell 2433 us per push,
// tiled 125 us.)
//
// Shapes chosen here when the caller names none, from the mesh size.  The halo
// has to hold the drift of a sort interval, since particles past it are
// pushed one by one through HBM (16 x 16 + 6 against + 8: 12 M against 0.3 M
// such pushes per 140 steps of 1024 x 768 cells at 32 per cell).  Us per push,
// one thing changed at a time (256 threads with halo 8 leave one workgroup's
// worth of waves on a CU):
//   2D, cells, per cell      16x16+6/256  16x16+8/256  16x16+8/512  32x16+8/512
//       512 x 512,   8            50           83           43           49
//       1024 x 256, 32           138          298          131          130
//       1024 x 768,  2            63          106           57           56
//       1024 x 768,  8           136          246          126          121
//       1024 x 768, 32           405          881          395          395
//       2048^2,     0.5          221          429          214          205
//       2048^2,      4           461          862          390          371
// so 16 x 16 + 8 with 512 threads below 1024 tiles of 32 x 16, those above it.
// 3D, from 512 tiles of 8^3 on: halo 5, 1024 threads, one workgroup per CU; below
// that halo 4, 512 threads (32 x 46 x 32 at 6 per cell: 29 us, halo 5 with 1024
// threads 35).  The 3D window is large beside its tile, so while the halo of 3
// holds the particles (up to a drift of 2.5 cells for light), and on thin plasma
// always, the first of these is the faster one; us per push, sorted every 3, 5,
// 10, 20 steps of half a cell:
//   cells, per cell        8^3+3/256               8^3+5/1024
//   128^3, 0.25      136  140  168  223       198  192  201  229
//   128^3, 1         184  186  266  431       235  231  248  355
//   128^3, 8         671  668  896 1845       693  685  739 1003
//   256^3, 0.25     1081 1098 1356 1733      1548 1569 1660 1973
//   256^3, 1        1476 1566 2032 3233      1949 2001 2160 2847
//   256^3, 2        1919 2065 2742 4759      2386 2454 2671 4172
static apt_status setup_tiles(apt_ctx *ctx) {
  const Mesh &m = ctx->mesh;
  const apt_params &pr = ctx->params;
  ctx->tiling = false;
  if (m.dim < 2) return APT_OK;
  int T[3] = {1, 1, 1};
  int halo, threads = pr.tile_threads > 0 ? pr.tile_threads : 256;
  const bool named = pr.tile[0] > 0 || pr.tile[1] > 0 || pr.tile_halo > 0 || pr.tile_threads > 0;
  auto tiles_of = [](int N, int t) { return (uint64_t)((N + t - 1) / t); };
  if (m.dim == 2) {
    const bool wide = !named && tiles_of(m.N[0], 32) * tiles_of(m.N[1], 16) >= 1024;
    T[0] = pr.tile[0] > 0 ? pr.tile[0] : (wide ? 32 : 16);
    T[1] = pr.tile[1] > 0 ? pr.tile[1] : 16;
    halo = T[0] == 8 ? 4 : 6;
    if (!named) {
      halo = 8;
      threads = 512;
    }
  } else {
    T[0] = T[1] = T[2] = pr.tile[0] > 0 ? pr.tile[0] : 8;
    halo = 3;
    if (!named) {
      const bool many = tiles_of(m.N[0], 8) * tiles_of(m.N[1], 8) * tiles_of(m.N[2], 8) >= 512;
      halo = many ? 5 : 4;
      threads = many ? 1024 : 512;
      ctx->tiles_by_drift = many;
    }
  }
  if (ctx->params.tile_halo > 0) halo = ctx->params.tile_halo;
  if (!tile_shape_supported(m.dim, T, halo, threads)) return APT_OK;
  uint64_t ntiles = 1;
  for (int d = 0; d < m.dim; d++) {
    if (!m.periodic[d]) return APT_OK;
    if (m.N[d] % T[d] != 0 && !no_idle_guards(m)) return APT_OK;
    ctx->tiles.nt[d] = (m.N[d] + T[d] - 1) / T[d];
    ctx->tiles.ax[d] = make_tile_axis(m.N[d], ctx->tiles.nt[d]);
    ntiles *= (uint64_t)ctx->tiles.nt[d];
  }
  for (int d = m.dim; d < 3; d++) {
    ctx->tiles.nt[d] = 1;
    ctx->tiles.ax[d] = make_tile_axis(1, 1);
  }
  ctx->tiles.shifts = true;
  for (int d = 0; d < 3; d++) {
    const TileAxis &a = ctx->tiles.ax[d];
    ctx->tiles.T[d] = T[d];
    ctx->tiles.sh[d] = a.dw.shift();
    ctx->tiles.shifts = ctx->tiles.shifts && a.r == 0 && (a.w & (a.w - 1)) == 0;
  }
  ctx->tiles.halo = halo;
  ctx->tiles.threads = threads;
  ctx->tiles.ntiles = (uint32_t)ntiles;
  HIPCHK(hipMalloc(&ctx->tile_off, (ntiles + 1) * 4));
  ctx->tiles.tile_off = ctx->tile_off;
  ctx->tiles.tiled_end = 0;
  ctx->tiling = true;
  return APT_OK;
}

static PtcF64 slots_from(const PtcF64 &p, uint64_t first) {
  return PtcF64{p.cell + first, p.x1 + first, p.x2 + first, p.x3 + first, p.p1 + first,
                p.p2 + first,   p.p3 + first, p.E + first,  p.w + first,  p.flag + first,
                p.id + first};
}

// ---- timing helpers ----------------------------------------------------
static void time_begin(apt_ctx *ctx, int k) {
  if (!ctx->timing) return;
  auto &v = ctx->ev[k];
  if (ctx->ev_used[k] == v.size()) {
    EventPair p;
    (void)hipEventCreate(&p.a);
    (void)hipEventCreate(&p.b);
    v.push_back(p);
  }
  (void)hipEventRecord(v[ctx->ev_used[k]].a, ctx->stream);
}
static void time_end(apt_ctx *ctx, int k) {
  if (!ctx->timing) return;
  (void)hipEventRecord(ctx->ev[k][ctx->ev_used[k]].b, ctx->stream);
  ctx->ev_used[k]++;
}

static apt_status relayout_tiles(apt_ctx *ctx);

// ------------------------------------------------------------------------
// Entry points: C linkage comes from the declarations in aperture_amd.h.

// apt_create has no context to hold its error message when it fails; the
// message of the last failed creation on this thread is kept here and
// returned by apt_last_error(NULL).
static thread_local std::string g_create_err = "no error";

// ---- the device histogram of apt_energy_histogram_noalloc --------------
// One copy of this array per GPU, held until the process ends.  In host
// code its name is only a handle: every host use goes through the device
// address resolved by resolve_scratch() for the device in question, never
// through `scratch` itself.
static __device__ __align__(256) uint32_t scratch[APT_NOALLOC_HIST_MAX_BINS];

constexpr int SCRATCH_MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static uint32_t *g_scratch_ptr[SCRATCH_MAX_DEVICES];

// Resolves the array's address on `dev`, which must be the current device;
// once per device (later calls return the kept pointer).
static hipError_t resolve_scratch(int dev) {
  if (dev < 0 || dev >= SCRATCH_MAX_DEVICES) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev]) return hipSuccess;
  void *ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess) return e;
  if (!ptr) return hipErrorInvalidSymbol;
  g_scratch_ptr[dev] = (uint32_t *)ptr;
  return hipSuccess;
}

static uint32_t *scratch_of(int dev) {
  if (dev < 0 || dev >= SCRATCH_MAX_DEVICES) return nullptr;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  return g_scratch_ptr[dev];
}

static apt_status create_fail(apt_status code, const char *msg) {
  g_create_err = msg;
  return code;
}

apt_status apt_create(const apt_grid *grid, const apt_params *params,
                      apt_ctx **out) {
  if (!grid || !params || !out)
    return create_fail(APT_ERR_INVALID_ARG, "create: null argument");
  *out = nullptr;
  // sorts and event scans count slots with 32-bit signed integers
  if (params->max_ptc_number > APT_MAX_SLOTS)
    return create_fail(APT_ERR_INVALID_ARG,
                       "create: max_ptc_number above 2^31 - 1 slots");
  if (params->max_photon_number > APT_MAX_SLOTS)
    return create_fail(APT_ERR_INVALID_ARG,
                       "create: max_photon_number above 2^31 - 1 slots");
  int devs = 0;
  if (hipGetDeviceCount(&devs) != hipSuccess || devs < 1)
    return APT_ERR_HIP;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return APT_ERR_HIP;
  if (resolve_scratch(dev) != hipSuccess)
    return create_fail(APT_ERR_HIP, "create: the no-allocation scratch array has no address");
  apt_ctx *ctx = new apt_ctx();
  ctx->device = dev;
  ctx->grid = *grid;
  ctx->params = *params;
  ctx->prec = params->precision;
  if (ctx->prec != APT_PREC_FP64 && ctx->prec != APT_PREC_MIXED) {
    delete ctx;
    return APT_ERR_INVALID_ARG;
  }
  Mesh &m = ctx->mesh;
  m.dim = 0;
  for (int d = 0; d < 3; d++) {
    if (grid->N[d] < 1 || grid->guard[d] < 0) {
      delete ctx;
      return APT_ERR_INVALID_ARG;
    }
    m.N[d] = grid->N[d];
    m.guard[d] = grid->guard[d];
    m.dims[d] = grid->N[d] + 2 * grid->guard[d];
    m.periodic[d] = grid->periodic[d] ? 1 : 0;
    m.lower[d] = grid->lower[d];
    m.delta[d] = grid->size[d] / grid->N[d];
    m.inv_delta[d] = 1.0 / m.delta[d];
    if (grid->N[d] > 1) m.dim = d + 1;
  }
  if (m.dim == 0) m.dim = 1;
  m.div0 = make_fastdiv((uint32_t)m.dims[0]);
  m.div01 = make_fastdiv((uint32_t)m.dims[0] * (uint32_t)m.dims[1]);
  for (int d = 0; d < m.dim; d++)
    if (m.guard[d] < 2) {
      delete ctx;
      return APT_ERR_INVALID_ARG;  // CIC + one-cell moves need guard >= 2
    }
  ctx->ncell = m.size();
  if (ctx->ncell >= 0xffffffffull) {
    delete ctx;
    return APT_ERR_INVALID_ARG;
  }
  // charges and masses (sim_environment_impl.hpp:87-98)
  for (int i = 0; i < 8; i++) {
    ctx->sp.q[i] = params->q_e;
    ctx->sp.m[i] = params->q_e;
  }
  ctx->sp.q[0] = -params->q_e;
  ctx->sp.m[2] = params->q_e * params->ion_mass;
  ctx->wmax = fabs(params->q_e);
  update_scale(ctx);

  if (hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking) !=
      hipSuccess) {
    delete ctx;
    return APT_ERR_HIP;
  }
  apt_status st = APT_OK;
  const size_t es = ctx->esize();
  const uint64_t nc = ctx->ncell;
  auto alloc_field = [&](void **p) -> bool {
    if (hipMalloc(p, nc * es) != hipSuccess) return false;
    if (ctx->prec == APT_PREC_FP64)
      return launch_fill<double>((double *)*p, 0.0, nc, ctx->stream) ==
             hipSuccess;
    return launch_fill<float>((float *)*p, 0.0f, nc, ctx->stream) ==
           hipSuccess;
  };
  bool ok = true;
  for (int c = 0; c < 3 && ok; c++)
    ok = alloc_field(&ctx->E[c]) && alloc_field(&ctx->B[c]) &&
         alloc_field(&ctx->Ebg[c]) && alloc_field(&ctx->Bbg[c]) &&
         alloc_field(&ctx->J[c]);
  int ns = params->num_species < 1 ? 1 : params->num_species;
  if (ns > 4) ns = 4;
  ctx->params.num_species = ns;
  // charge arrays for all four species slots: injected ions and pair
  // secondaries never index a missing array, whatever num_species says
  for (int s = 0; s < 4 && ok; s++) ok = alloc_field(&ctx->Rho[s]);
  ok = ok && alloc_field(&ctx->divE) && alloc_field(&ctx->divB) &&
       alloc_field(&ctx->jtmp) && alloc_field(&ctx->EdotB) &&
       alloc_field(&ctx->ph_produced) && alloc_field(&ctx->pair_produced);
  int limbs = ctx->prec == APT_PREC_FP64 ? 2 : 1;
  for (int c = 0; c < 3 && ok; c++)
    for (int l = 0; l < limbs && ok; l++)
      ok = hipMalloc(&ctx->Jacc[c][l], nc * 8) == hipSuccess &&
           launch_fill<long long>(ctx->Jacc[c][l], 0, nc, ctx->stream) ==
               hipSuccess;
  for (int s = 0; s < 4 && ok; s++)
    for (int l = 0; l < limbs && ok; l++)
      ok = hipMalloc(&ctx->Racc[s][l], nc * 8) == hipSuccess &&
           launch_fill<long long>(ctx->Racc[s][l], 0, nc, ctx->stream) ==
               hipSuccess;
  ok = ok && hipMalloc(&ctx->divres_part, 2 * DIVRES_MAX_BLOCKS * 8) == hipSuccess;
  ok = ok && hipMalloc(&ctx->d_counters, CTR_NUM * 8) == hipSuccess &&
       hipMemsetAsync(ctx->d_counters, 0, CTR_NUM * 8, ctx->stream) ==
           hipSuccess;
  if (!ok) {
    apt_destroy(ctx);
    return APT_ERR_HIP;
  }
  ctx->cap = params->max_ptc_number;
  if (ctx->cap > 0xffffffffull) {
    apt_destroy(ctx);
    return APT_ERR_INVALID_ARG;
  }
  if (ctx->cap > 0) st = alloc_ptc(ctx, false);
  if (st != APT_OK) {
    apt_destroy(ctx);
    return st;
  }
  ctx->logsph = params->coord == APT_COORD_LOGSPH;
  // a log-spherical step without charge output writes 0 / dV, a signed zero
  // (or no number) in guard cells
  if (ctx->logsph) ctx->rho_zero = false;
  ctx->gr1d = params->coord == APT_COORD_1DGR;
  ctx->gap1d = params->coord == APT_COORD_1DGAP;
  if (params->coord != APT_COORD_CARTESIAN && !ctx->logsph && !ctx->gr1d && !ctx->gap1d) {
    apt_destroy(ctx);
    return APT_ERR_INVALID_ARG;
  }
  if (ctx->gap1d) {
    // one line, FP64 form; the deposit reaches two cells below the
    // particle's cell (ptc_updater_1dgap.cu:139-141)
    if (m.dim != 1 || m.guard[0] < 2 || ctx->prec != APT_PREC_FP64) {
      apt_destroy(ctx);
      return create_fail(APT_ERR_INVALID_ARG,
                         "create: a 1D gap context is 1D, FP64, guard >= 2");
    }
    ctx->gap_B0 = (float)params->B0;
    ctx->gap_omega = (float)params->omega;
    ctx->gap_track = (float)params->track_percent;
  }
  if (ctx->gr1d) {
    // one field line, FP64 form; the stencils reach two cells past the
    // particle's cell (ptc_updater_1dgr.cu:172-175, 261-262)
    if (m.dim != 1 || m.guard[0] < 3 || ctx->prec != APT_PREC_FP64) {
      apt_destroy(ctx);
      return APT_ERR_INVALID_ARG;
    }
    ctx->gr_a = (float)params->spin_a;
    ctx->gr_omega = (float)params->omega;
    ctx->gr_B0 = (float)params->B0;
    ctx->gr_track = (float)params->track_percent;
    bool okc = true;
    for (int k = 0; k < GR_NCOEF && okc; k++) {
      ctx->gr_host[k].assign(m.dims[0], 0.0);
      okc = hipMalloc(&ctx->gr_dev[k], (size_t)m.dims[0] * 8) == hipSuccess &&
            hipMemcpy(ctx->gr_dev[k], ctx->gr_host[k].data(), (size_t)m.dims[0] * 8,
                      hipMemcpyHostToDevice) == hipSuccess;
    }
    if (!okc) {
      apt_destroy(ctx);
      return APT_ERR_HIP;
    }
  }
  if (ctx->logsph) {
    // 2D: the particle path and Yee solver (field_solver_logsph.cu:357-358);
    // 3D: the force-free / vacuum solver, which updates two guard layers
    // (ffe_solver_logsph.cu:18) and needs guard >= 3
    bool ok2 = m.dim == 2 && m.guard[0] >= 2 && m.guard[1] >= 2;
    bool ok3 = m.dim == 3 && m.guard[0] >= 3 && m.guard[1] >= 3 && m.guard[2] >= 3;
    if (!(ok2 || ok3) || params->damping_length < 0 ||
        params->damping_length > m.dims[0]) {
      apt_destroy(ctx);
      return APT_ERR_INVALID_ARG;
    }
    LsParams &lp = ctx->lp;
    lp.compactness = params->compactness;
    lp.omega = params->omega;
    lp.gravity = params->gravity_on ? params->gravity : 0.0;
    lp.rad_cooling_on = params->rad_cooling_on;
    lp.rad_cooling_coef = params->rad_cooling_coef;
    lp.B0 = params->B0;
    lp.damping_length = params->damping_length;
    lp.damping_coef = params->damping_coef;
    lp.inject_ions = params->inject_ions;
    lp.track_percent = params->track_percent;
    std::vector<double> c[LS_NCOEF];
    logsph_coef_host(m, c);
    bool okc = true;
    const uint64_t n2 = (uint64_t)m.dims[0] * m.dims[1];  // 2D arrays
    for (int k = 0; k < LS_NCOEF && okc; k++) {
      okc = hipMalloc(&ctx->coef_mem[k], n2 * 8) == hipSuccess &&
            hipMemcpy(ctx->coef_mem[k], c[k].data(), n2 * 8,
                      hipMemcpyHostToDevice) == hipSuccess;
      ctx->coef.a[k] = ctx->coef_mem[k];
    }
    const uint64_t N1 = (uint64_t)m.N[1];
    okc = okc && hipMalloc(&ctx->surf, 4 * N1 * 8) == hipSuccess;
    if (!okc) {
      apt_destroy(ctx);
      return APT_ERR_HIP;
    }
  }
  RtParams &rt = ctx->rt;
  rt.model = params->rt_model;
  rt.gamma_thr = params->gamma_thr;
  rt.photon_path = params->photon_path;
  rt.E_secondary = params->E_secondary;
  rt.r_cutoff = params->r_cutoff;
  rt.e_frac = params->e_frac;
  rt.max_ptc = ctx->cap;
  rt.max_photon = params->max_photon_number;
  ctx->ph_cap = params->max_photon_number;
  if (ctx->ph_cap > 0xffffffffull) {
    apt_destroy(ctx);
    return APT_ERR_INVALID_ARG;
  }
  ctx->sortw.most = ctx->rtw.most = ctx->cap > ctx->ph_cap ? ctx->cap : ctx->ph_cap;
  if (ctx->ph_cap > 0 && (st = alloc_photons(ctx, false)) != APT_OK) {
    apt_destroy(ctx);
    return st;
  }
  if (ctx->prec == APT_PREC_MIXED && !ctx->logsph) {
    st = setup_tiles(ctx);
    if (st != APT_OK) {
      apt_destroy(ctx);
      return st;
    }
  }
  // a smoothed box's work arrays last: where they do not fit, each component is
  // filtered through jtmp in turn
  if (params->coord == APT_COORD_CARTESIAN && params->current_smoothing > 0 &&
      guard_images_ok(m)) {
    bool room = true;
    for (int q = 0; q < 3 && room; q++) room = alloc_field(&ctx->ftmp[q]);
    if (!room) drop_ftmp(ctx);
  }
  if (hipStreamSynchronize(ctx->stream) != hipSuccess) {
    apt_destroy(ctx);
    return APT_ERR_HIP;
  }
  *out = ctx;
  return APT_OK;
}

apt_status apt_destroy(apt_ctx *ctx) {
  CHECK_CTX(ctx);
  if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
  for (int k = 0; k < GR_NCOEF; k++) (void)hipFree(ctx->gr_dev[k]);
  for (int c = 0; c < 3; c++) {
    (void)hipFree(ctx->E[c]); (void)hipFree(ctx->B[c]); (void)hipFree(ctx->Ebg[c]);
    (void)hipFree(ctx->Bbg[c]); (void)hipFree(ctx->J[c]);
    (void)hipFree(ctx->Jacc[c][0]); (void)hipFree(ctx->Jacc[c][1]);
  }
  for (int s = 0; s < 4; s++) {
    (void)hipFree(ctx->Rho[s]);
    (void)hipFree(ctx->Racc[s][0]);
    (void)hipFree(ctx->Racc[s][1]);
  }
  (void)hipFree(ctx->divE); (void)hipFree(ctx->divB); (void)hipFree(ctx->jtmp);
  for (void *q : ctx->ftmp) (void)hipFree(q);
  (void)hipFree(ctx->divres_part); (void)hipFree(ctx->divres_field);
  (void)hipFree(ctx->EdotB); (void)hipFree(ctx->ph_produced);
  (void)hipFree(ctx->pair_produced); (void)hipFree(ctx->diag_ph);
  for (int s = 0; s < 4; s++) {
    (void)hipFree(ctx->diag_num[s]);
    (void)hipFree(ctx->diag_gamma[s]);
  }
  (void)hipFree(ctx->d_counters);
  (void)hipFree(ctx->d_dc);
  if (ctx->gexec) (void)hipGraphExecDestroy(ctx->gexec);
  for (int k = 0; k < LS_NCOEF; k++) (void)hipFree(ctx->coef_mem[k]);
  for (int k = 0; k < 12; k++) (void)hipFree(ctx->ffe[k]);
  for (int k = 0; k < 10; k++) (void)hipFree(ctx->ffc[k]);
  (void)hipFree(ctx->surf);
  free_ph64(ctx->ph64); free_ph64(ctx->ph64b);
  free_ph32(ctx->ph32); free_ph32(ctx->ph32b);
  ctx->rtw.release();
  (void)hipFree(ctx->tile_off);
  (void)hipFree(ctx->run_off);
  ctx->tsort.release();
  free_ptc64(ctx->p64); free_ptc64(ctx->p64b);
  free_ptc32(ctx->p32); free_ptc32(ctx->p32b);
  ctx->sortw.release();
  for (int k = 0; k < APT_KERNEL_NUM; k++)
    for (auto &p : ctx->ev[k]) {
      (void)hipEventDestroy(p.a);
      (void)hipEventDestroy(p.b);
    }
  if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
  delete ctx;
  return APT_OK;
}

const char *apt_last_error(const apt_ctx *ctx) {
  return ctx ? ctx->err.c_str() : g_create_err.c_str();
}

apt_status apt_get_jexp(const apt_ctx *ctx, int *H) {
  CHECK_CTX(ctx);
  if (!H) return APT_ERR_INVALID_ARG;
  *H = ctx->H;
  return APT_OK;
}

apt_status apt_get_mesh(const apt_ctx *ctx, int dims[3], double delta[3]) {
  CHECK_CTX(ctx);
  for (int d = 0; d < 3; d++) {
    if (dims) dims[d] = ctx->mesh.dims[d];
    if (delta) delta[d] = ctx->mesh.delta[d];
  }
  return APT_OK;
}

apt_status apt_get_info(const apt_ctx *cctx, apt_info *out) {
  apt_ctx *ctx = const_cast<apt_ctx *>(cctx);
  CHECK_CTX(ctx);
  if (!out) return APT_ERR_INVALID_ARG;
  apt_status st = exact_counts(ctx);
  if (st != APT_OK) return st;
  out->number = ctx->number;
  out->ph_number = ctx->ph_number;
  out->H = ctx->H;
  out->Hs = surface_scale(ctx);
  out->id_next = ctx->id_next;
  out->ph_id_next = ctx->ph_id_next;
  out->rt_epoch = ctx->rt_epoch;
  out->inject_epoch = ctx->inject_epoch;
  return APT_OK;
}

// restores the id counters, random-stream epochs and fixed-point exponents
// (a snapshot reload); counts come from the restored arrays.  Only the
// exponents of the weight scales matter, so they are restored as powers of
// two that give the same H and Hs.
apt_status apt_set_counters(apt_ctx *ctx, const apt_info *in) {
  CHECK_CTX(ctx);
  if (!in) return APT_ERR_INVALID_ARG;
  const int e = (ctx->prec == APT_PREC_FP64 ? 22 : 30) - in->H;
  const int es = 22 - in->Hs;
  if (e < -60 || e > 60 || es < 0 || es > 60)
    return ctx->fail(APT_ERR_INVALID_ARG, "set_counters: exponents out of range");
  ctx->id_next = in->id_next;
  ctx->ph_id_next = in->ph_id_next;
  ctx->rt_epoch = in->rt_epoch;
  ctx->inject_epoch = in->inject_epoch;
  ctx->wmax = ldexp(1.0, e);
  update_scale(ctx);
  ctx->wmaxw = ldexp(1.0, es);
  return push_counts(ctx);
}

apt_status apt_get_coef(apt_ctx *ctx, int which, double *dst, uint64_t count) {
  CHECK_CTX(ctx);
  if (ctx->gr1d) {
    if (which < 0 || which >= GR_NCOEF || !dst || count != (uint64_t)ctx->mesh.dims[0])
      return ctx->fail(APT_ERR_INVALID_ARG, "get_coef: bad coefficient/size");
    std::copy(ctx->gr_host[which].begin(), ctx->gr_host[which].end(), dst);
    return APT_OK;
  }
  if (!ctx->logsph)
    return ctx->fail(APT_ERR_UNSUPPORTED, "get_coef: not a log-spherical context");
  const uint64_t n2 = (uint64_t)ctx->mesh.dims[0] * ctx->mesh.dims[1];
  if (which < 0 || which >= LS_NCOEF || !dst || count != n2)
    return ctx->fail(APT_ERR_INVALID_ARG, "get_coef: bad coefficient/size");
  HIPCHK(hipStreamSynchronize(ctx->stream));
  HIPCHK(hipMemcpy(dst, ctx->coef_mem[which], count * 8, hipMemcpyDeviceToHost));
  return APT_OK;
}

static void **field_slot(apt_ctx *ctx, int which, int comp) {
  if (comp < 0) return nullptr;
  switch (which) {
    case APT_FIELD_E: return comp < 3 ? &ctx->E[comp] : nullptr;
    case APT_FIELD_B: return comp < 3 ? &ctx->B[comp] : nullptr;
    case APT_FIELD_EBG: return comp < 3 ? &ctx->Ebg[comp] : nullptr;
    case APT_FIELD_BBG: return comp < 3 ? &ctx->Bbg[comp] : nullptr;
    case APT_FIELD_J: return comp < 3 ? &ctx->J[comp] : nullptr;
    case APT_FIELD_RHO:
      return comp < ctx->params.num_species ? &ctx->Rho[comp] : nullptr;
    case APT_FIELD_DIVE: return comp == 0 ? &ctx->divE : nullptr;
    case APT_FIELD_DIVB: return comp == 0 ? &ctx->divB : nullptr;
    case APT_FIELD_EDOTB: return comp == 0 ? &ctx->EdotB : nullptr;
    case APT_FIELD_PHOTON_PRODUCED: return comp == 0 ? &ctx->ph_produced : nullptr;
    case APT_FIELD_PAIR_PRODUCED: return comp == 0 ? &ctx->pair_produced : nullptr;
    case APT_FIELD_PTC_NUM:
      return comp < ctx->params.num_species ? &ctx->diag_num[comp] : nullptr;
    case APT_FIELD_GAMMA:
      return comp < ctx->params.num_species ? &ctx->diag_gamma[comp] : nullptr;
    case APT_FIELD_PHOTON_NUM: return comp == 0 ? &ctx->diag_ph : nullptr;
    case APT_FIELD_FFE_E: return comp < 3 ? &ctx->ffc[comp] : nullptr;
    case APT_FIELD_FFE_B: return comp < 3 ? &ctx->ffc[3 + comp] : nullptr;
    case APT_FIELD_FFE_F: return comp == 0 ? &ctx->ffc[6] : nullptr;
  }
  return nullptr;
}

// a field was written other than through a step's own kernels
static void field_written(apt_ctx *ctx, int which) {
  if (which == APT_FIELD_EBG) ctx->ebg_zero = false;
  if (which == APT_FIELD_BBG) ctx->bbg_zero = false;
  if (which == APT_FIELD_RHO) ctx->rho_zero = false;
}

// the Cartesian force-free work fields, zeroed, on first use
static hipError_t ensure_ffe_cart(apt_ctx *ctx, int n = 7) {
  const size_t es = ctx->prec == APT_PREC_FP64 ? 8 : 4;
  for (int k = 0; k < n; k++) {
    if (ctx->ffc[k]) continue;
    hipError_t e = hipMalloc(&ctx->ffc[k], ctx->ncell * es);
    if (e == hipSuccess)
      e = ctx->prec == APT_PREC_FP64
              ? launch_fill<double>((double *)ctx->ffc[k], 0.0, ctx->ncell, ctx->stream)
              : launch_fill<float>((float *)ctx->ffc[k], 0.0f, ctx->ncell, ctx->stream);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

static bool is_ffe_work(int which) {
  return which == APT_FIELD_FFE_E || which == APT_FIELD_FFE_B || which == APT_FIELD_FFE_F;
}

apt_status apt_field_set(apt_ctx *ctx, int which, int comp,
                         const double *src, uint64_t count) {
  CHECK_CTX(ctx);
  if (is_ffe_work(which)) HIPCHK(ensure_ffe_cart(ctx));
  void **slot = field_slot(ctx, which, comp);
  if (!slot || !src || count != ctx->ncell)
    return ctx->fail(APT_ERR_INVALID_ARG, "field_set: bad field/size");
  if (!*slot)
    return ctx->fail(APT_ERR_STATE, "field_set: moments not collected yet");
  field_written(ctx, which);
  HIPCHK(hipStreamSynchronize(ctx->stream));
  if (ctx->prec == APT_PREC_FP64) {
    HIPCHK(hipMemcpy(*slot, src, count * 8, hipMemcpyHostToDevice));
  } else {
    std::vector<float> tmp(count);
    for (uint64_t i = 0; i < count; i++) tmp[i] = (float)src[i];
    HIPCHK(hipMemcpy(*slot, tmp.data(), count * 4, hipMemcpyHostToDevice));
  }
  return APT_OK;
}

apt_status apt_field_get(apt_ctx *ctx, int which, int comp, double *dst,
                         uint64_t count) {
  CHECK_CTX(ctx);
  if (is_ffe_work(which)) HIPCHK(ensure_ffe_cart(ctx));
  void **slot = field_slot(ctx, which, comp);
  if (!slot || !dst || count != ctx->ncell)
    return ctx->fail(APT_ERR_INVALID_ARG, "field_get: bad field/size");
  if (!*slot)
    return ctx->fail(APT_ERR_STATE, "field_get: moments not collected yet");
  HIPCHK(hipStreamSynchronize(ctx->stream));
  if (ctx->prec == APT_PREC_FP64) {
    HIPCHK(hipMemcpy(dst, *slot, count * 8, hipMemcpyDeviceToHost));
  } else {
    std::vector<float> tmp(count);
    HIPCHK(hipMemcpy(tmp.data(), *slot, count * 4, hipMemcpyDeviceToHost));
    for (uint64_t i = 0; i < count; i++) dst[i] = tmp[i];
  }
  return APT_OK;
}

apt_status apt_ptc_set(apt_ctx *ctx, const apt_particles *src, uint64_t n) {
  CHECK_CTX(ctx);
  if (!src || !src->cell || !src->x1 || !src->x2 || !src->x3 || !src->p1 ||
      !src->p2 || !src->p3 || !src->weight || !src->flag)
    return ctx->fail(APT_ERR_INVALID_ARG, "ptc_set: missing arrays");
  if (n > ctx->cap)
    return ctx->fail(APT_ERR_CAPACITY, "ptc_set: %llu > capacity %llu",
                     (unsigned long long)n, (unsigned long long)ctx->cap);
  HIPCHK(hipStreamSynchronize(ctx->stream));
  double wmax = fabs(ctx->params.q_e), wmaxw = 1.0;
  for (uint64_t i = 0; i < n; i++) {
    int s = (int)(src->flag[i] >> 29);
    if (s > 3)
      return ctx->fail(APT_ERR_INVALID_ARG, "ptc_set: species %d > 3 at %llu", s,
                       (unsigned long long)i);
    double qw = fabs(ctx->sp.q[s] * src->weight[i]);
    if (qw > wmax) wmax = qw;
    if (fabs(src->weight[i]) > wmaxw) wmaxw = fabs(src->weight[i]);
  }
  ctx->wmax = wmax;
  ctx->wmaxw = wmaxw;
  update_scale(ctx);
  ctx->id_next = n;
  if (src->id)
    for (uint64_t i = 0; i < n; i++)
      if (src->id[i] + 1 > ctx->id_next) ctx->id_next = src->id[i] + 1;
  if (ctx->prec == APT_PREC_FP64) {
    PtcF64 &p = ctx->p64;
    HIPCHK(hipMemcpy(p.cell, src->cell, n * 4, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(p.x1, src->x1, n * 8, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(p.x2, src->x2, n * 8, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(p.x3, src->x3, n * 8, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(p.p1, src->p1, n * 8, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(p.p2, src->p2, n * 8, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(p.p3, src->p3, n * 8, hipMemcpyHostToDevice));
    if (src->E) {
      HIPCHK(hipMemcpy(p.E, src->E, n * 8, hipMemcpyHostToDevice));
    } else {
      std::vector<double> g(n);
      for (uint64_t i = 0; i < n; i++)
        g[i] = sqrt(1.0 + src->p1[i] * src->p1[i] + src->p2[i] * src->p2[i] +
                    src->p3[i] * src->p3[i]);
      HIPCHK(hipMemcpy(p.E, g.data(), n * 8, hipMemcpyHostToDevice));
    }
    HIPCHK(hipMemcpy(p.w, src->weight, n * 8, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(p.flag, src->flag, n * 4, hipMemcpyHostToDevice));
    if (src->id) {
      HIPCHK(hipMemcpy(p.id, src->id, n * 8, hipMemcpyHostToDevice));
    } else {
      std::vector<uint64_t> ids(n);
      for (uint64_t i = 0; i < n; i++) ids[i] = i;
      HIPCHK(hipMemcpy(p.id, ids.data(), n * 8, hipMemcpyHostToDevice));
    }
  } else {
    PtcF32 &p = ctx->p32;
    std::vector<float> f(n);
    auto put = [&](float *d, const double *s) -> hipError_t {
      for (uint64_t i = 0; i < n; i++) f[i] = (float)s[i];
      return hipMemcpy(d, f.data(), n * 4, hipMemcpyHostToDevice);
    };
    auto put_off = [&](float *d, const double *s) -> hipError_t {
      for (uint64_t i = 0; i < n; i++) {
        float v = (float)s[i];
        f[i] = v >= 1.0f ? 0x1.fffffep-1f : v;
      }
      return hipMemcpy(d, f.data(), n * 4, hipMemcpyHostToDevice);
    };
    HIPCHK(hipMemcpy(p.cell, src->cell, n * 4, hipMemcpyHostToDevice));
    HIPCHK(put_off(p.x1, src->x1));
    HIPCHK(ctx->mesh.dim > 1 ? put_off(p.x2, src->x2) : put(p.x2, src->x2));
    HIPCHK(ctx->mesh.dim > 2 ? put_off(p.x3, src->x3) : put(p.x3, src->x3));
    HIPCHK(put(p.u1, src->p1));
    HIPCHK(put(p.u2, src->p2));
    HIPCHK(put(p.u3, src->p3));
    HIPCHK(put(p.w, src->weight));
    // bit 27 is the tiled push's scratch mark: a particle uploaded with it
    // set would be pushed twice when its tile's queue overflows
    std::vector<uint32_t> fl(src->flag, src->flag + n);
    for (auto &v : fl) v &= ~(uint32_t)APT_FLAG_RESERVED;
    HIPCHK(hipMemcpy(p.flag, fl.data(), n * 4, hipMemcpyHostToDevice));
  }
  // slots past n are empty
  if (n < ctx->number)
    HIPCHK(launch_fill<uint32_t>(
        (ctx->prec == APT_PREC_FP64 ? ctx->p64.cell : ctx->p32.cell) + n,
        MAX_CELL, ctx->number - n, ctx->stream));
  ctx->number = n;
  ctx->tiles_valid = false;
  ctx->runs_valid = false;
  HIPCHK(hipStreamSynchronize(ctx->stream));
  return push_counts(ctx);
}

apt_status apt_ptc_get(apt_ctx *ctx, apt_particles *dst, uint64_t cap,
                       uint64_t *n) {
  CHECK_CTX(ctx);
  if (!dst) return APT_ERR_INVALID_ARG;
  {
    apt_status st = exact_counts(ctx);
    if (st != APT_OK) return st;
  }
  HIPCHK(hipStreamSynchronize(ctx->stream));
  uint64_t num = ctx->number;
  if (n) *n = num;
  if (num > cap)
    return ctx->fail(APT_ERR_CAPACITY, "ptc_get: %llu particles > cap %llu",
                     (unsigned long long)num, (unsigned long long)cap);
  if (ctx->prec == APT_PREC_FP64) {
    PtcF64 &p = ctx->p64;
    if (dst->cell) HIPCHK(hipMemcpy(dst->cell, p.cell, num * 4, hipMemcpyDeviceToHost));
    if (dst->x1) HIPCHK(hipMemcpy(dst->x1, p.x1, num * 8, hipMemcpyDeviceToHost));
    if (dst->x2) HIPCHK(hipMemcpy(dst->x2, p.x2, num * 8, hipMemcpyDeviceToHost));
    if (dst->x3) HIPCHK(hipMemcpy(dst->x3, p.x3, num * 8, hipMemcpyDeviceToHost));
    if (dst->p1) HIPCHK(hipMemcpy(dst->p1, p.p1, num * 8, hipMemcpyDeviceToHost));
    if (dst->p2) HIPCHK(hipMemcpy(dst->p2, p.p2, num * 8, hipMemcpyDeviceToHost));
    if (dst->p3) HIPCHK(hipMemcpy(dst->p3, p.p3, num * 8, hipMemcpyDeviceToHost));
    if (dst->E) HIPCHK(hipMemcpy(dst->E, p.E, num * 8, hipMemcpyDeviceToHost));
    if (dst->weight) HIPCHK(hipMemcpy(dst->weight, p.w, num * 8, hipMemcpyDeviceToHost));
    if (dst->flag) HIPCHK(hipMemcpy(dst->flag, p.flag, num * 4, hipMemcpyDeviceToHost));
    if (dst->id) HIPCHK(hipMemcpy(dst->id, p.id, num * 8, hipMemcpyDeviceToHost));
  } else {
    PtcF32 &p = ctx->p32;
    std::vector<float> f(num), u1(num), u2(num), u3(num);
    auto get = [&](double *d, const float *s) -> hipError_t {
      hipError_t e = hipMemcpy(f.data(), s, num * 4, hipMemcpyDeviceToHost);
      if (e == hipSuccess && d)
        for (uint64_t i = 0; i < num; i++) d[i] = f[i];
      return e;
    };
    if (dst->cell) HIPCHK(hipMemcpy(dst->cell, p.cell, num * 4, hipMemcpyDeviceToHost));
    if (dst->x1) HIPCHK(get(dst->x1, p.x1));
    if (dst->x2) HIPCHK(get(dst->x2, p.x2));
    if (dst->x3) HIPCHK(get(dst->x3, p.x3));
    HIPCHK(hipMemcpy(u1.data(), p.u1, num * 4, hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(u2.data(), p.u2, num * 4, hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(u3.data(), p.u3, num * 4, hipMemcpyDeviceToHost));
    for (uint64_t i = 0; i < num; i++) {
      if (dst->p1) dst->p1[i] = u1[i];
      if (dst->p2) dst->p2[i] = u2[i];
      if (dst->p3) dst->p3[i] = u3[i];
      if (dst->E)
        dst->E[i] = sqrt(1.0 + (double)u1[i] * u1[i] + (double)u2[i] * u2[i] +
                         (double)u3[i] * u3[i]);
      if (dst->id) dst->id[i] = i;
    }
    if (dst->weight) HIPCHK(get(dst->weight, p.w));
    if (dst->flag) HIPCHK(hipMemcpy(dst->flag, p.flag, num * 4, hipMemcpyDeviceToHost));
  }
  return APT_OK;
}

apt_status apt_ptc_number(apt_ctx *ctx, uint64_t *n) {
  CHECK_CTX(ctx);
  if (!n) return APT_ERR_INVALID_ARG;
  apt_status st = exact_counts(ctx);
  if (st != APT_OK) return st;
  *n = ctx->number;
  return APT_OK;
}

apt_status apt_ph_set(apt_ctx *ctx, const apt_photons *src, uint64_t n) {
  CHECK_CTX(ctx);
  if (!src || !src->cell || !src->x1 || !src->x2 || !src->x3 || !src->p1 ||
      !src->p2 || !src->p3 || !src->weight || !src->path_left)
    return ctx->fail(APT_ERR_INVALID_ARG, "ph_set: missing arrays");
  if (n > ctx->ph_cap)
    return ctx->fail(APT_ERR_CAPACITY, "ph_set: %llu > photon capacity %llu",
                     (unsigned long long)n, (unsigned long long)ctx->ph_cap);
  HIPCHK(hipStreamSynchronize(ctx->stream));
  std::vector<uint32_t> fl(n, 0u);
  if (src->flag) fl.assign(src->flag, src->flag + n);
  if (ctx->prec == APT_PREC_FP64) {
    PhoF64 &p = ctx->ph64;
    HIPCHK(hipMemcpy(p.cell, src->cell, n * 4, hipMemcpyHostToDevice));
    const double *hs[] = {src->x1, src->x2, src->x3, src->p1, src->p2,
                          src->p3, src->weight, src->path_left};
    double *ds[] = {p.x1, p.x2, p.x3, p.p1, p.p2, p.p3, p.w, p.path};
    for (int k = 0; k < 8; k++)
      HIPCHK(hipMemcpy(ds[k], hs[k], n * 8, hipMemcpyHostToDevice));
    std::vector<double> e(n);
    for (uint64_t i = 0; i < n; i++)
      e[i] = src->E ? src->E[i]
                    : sqrt(src->p1[i] * src->p1[i] + src->p2[i] * src->p2[i] +
                           src->p3[i] * src->p3[i]);
    HIPCHK(hipMemcpy(p.E, e.data(), n * 8, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(p.flag, fl.data(), n * 4, hipMemcpyHostToDevice));
    std::vector<uint64_t> ids(n);
    for (uint64_t i = 0; i < n; i++) ids[i] = src->id ? src->id[i] : i;
    HIPCHK(hipMemcpy(p.id, ids.data(), n * 8, hipMemcpyHostToDevice));
  } else {
    PhoF32 &p = ctx->ph32;
    HIPCHK(hipMemcpy(p.cell, src->cell, n * 4, hipMemcpyHostToDevice));
    const double *hs[] = {src->x1, src->x2, src->x3, src->p1, src->p2,
                          src->p3, src->weight, src->path_left};
    float *ds[] = {p.x1, p.x2, p.x3, p.p1, p.p2, p.p3, p.w, p.path};
    std::vector<float> f(n);
    for (int k = 0; k < 8; k++) {
      for (uint64_t i = 0; i < n; i++) f[i] = (float)hs[k][i];
      HIPCHK(hipMemcpy(ds[k], f.data(), n * 4, hipMemcpyHostToDevice));
    }
    HIPCHK(hipMemcpy(p.flag, fl.data(), n * 4, hipMemcpyHostToDevice));
  }
  uint32_t *cell = ctx->prec == APT_PREC_FP64 ? ctx->ph64.cell : ctx->ph32.cell;
  if (n < ctx->ph_number)
    HIPCHK(launch_fill<uint32_t>(cell + n, MAX_CELL, ctx->ph_number - n,
                                 ctx->stream));
  ctx->ph_number = n;
  ctx->ph_id_next = n;
  if (src->id)
    for (uint64_t i = 0; i < n; i++)
      if (src->id[i] + 1 > ctx->ph_id_next) ctx->ph_id_next = src->id[i] + 1;
  HIPCHK(hipStreamSynchronize(ctx->stream));
  return push_counts(ctx);
}

apt_status apt_ph_get(apt_ctx *ctx, apt_photons *dst, uint64_t cap,
                      uint64_t *n) {
  CHECK_CTX(ctx);
  {
    apt_status st = exact_counts(ctx);
    if (st != APT_OK) return st;
  }
  if (!dst) return APT_ERR_INVALID_ARG;
  HIPCHK(hipStreamSynchronize(ctx->stream));
  const uint64_t num = ctx->ph_number;
  if (n) *n = num;
  if (num > cap)
    return ctx->fail(APT_ERR_CAPACITY, "ph_get: %llu photons > cap %llu",
                     (unsigned long long)num, (unsigned long long)cap);
  if (num == 0) return APT_OK;
  if (ctx->prec == APT_PREC_FP64) {
    PhoF64 &p = ctx->ph64;
    double *hs[] = {dst->x1, dst->x2, dst->x3, dst->p1, dst->p2, dst->p3,
                    dst->E, dst->weight, dst->path_left};
    double *ds[] = {p.x1, p.x2, p.x3, p.p1, p.p2, p.p3, p.E, p.w, p.path};
    for (int k = 0; k < 9; k++)
      if (hs[k]) HIPCHK(hipMemcpy(hs[k], ds[k], num * 8, hipMemcpyDeviceToHost));
    if (dst->id) HIPCHK(hipMemcpy(dst->id, p.id, num * 8, hipMemcpyDeviceToHost));
    if (dst->cell) HIPCHK(hipMemcpy(dst->cell, p.cell, num * 4, hipMemcpyDeviceToHost));
    if (dst->flag) HIPCHK(hipMemcpy(dst->flag, p.flag, num * 4, hipMemcpyDeviceToHost));
  } else {
    PhoF32 &p = ctx->ph32;
    double *hs[] = {dst->x1, dst->x2, dst->x3, dst->p1, dst->p2, dst->p3,
                    dst->weight, dst->path_left};
    float *ds[] = {p.x1, p.x2, p.x3, p.p1, p.p2, p.p3, p.w, p.path};
    std::vector<float> f(num), pp[3];
    for (int k = 0; k < 8; k++) {
      HIPCHK(hipMemcpy(f.data(), ds[k], num * 4, hipMemcpyDeviceToHost));
      if (k >= 3 && k < 6) pp[k - 3] = f;
      if (hs[k])
        for (uint64_t i = 0; i < num; i++) hs[k][i] = f[i];
    }
    if (dst->E)
      for (uint64_t i = 0; i < num; i++)
        dst->E[i] = sqrt((double)pp[0][i] * pp[0][i] + (double)pp[1][i] * pp[1][i] +
                         (double)pp[2][i] * pp[2][i]);
    if (dst->id)
      for (uint64_t i = 0; i < num; i++) dst->id[i] = i;
    if (dst->cell) HIPCHK(hipMemcpy(dst->cell, p.cell, num * 4, hipMemcpyDeviceToHost));
    if (dst->flag) HIPCHK(hipMemcpy(dst->flag, p.flag, num * 4, hipMemcpyDeviceToHost));
  }
  return APT_OK;
}

apt_status apt_ptc_load_uniform(apt_ctx *ctx, int ppc_pairs,
                                const double theta[2], const double drift[2],
                                double weight) {
  CHECK_CTX(ctx);
  if (ppc_pairs < 1 || !theta || !drift)
    return ctx->fail(APT_ERR_INVALID_ARG, "load_uniform: bad arguments");
  const Mesh &m = ctx->mesh;
  uint64_t bulk = (uint64_t)m.N[0] * m.N[1] * m.N[2];
  uint64_t add = bulk * (uint64_t)ppc_pairs * 2;
  uint64_t base = ctx->number + (ctx->number & 1);
  if (base + add > ctx->cap)
    return ctx->fail(APT_ERR_CAPACITY, "load_uniform: %llu particles > cap",
                     (unsigned long long)(base + add));
  LoadParams lp;
  lp.ppc = ppc_pairs;
  lp.theta[0] = theta[0];
  lp.theta[1] = theta[1];
  lp.drift[0] = drift[0];
  lp.drift[1] = drift[1];
  lp.weight = weight;
  lp.seed = ctx->params.random_seed;
  lp.base = base;
  double qw = fabs(ctx->params.q_e * weight);
  if (ctx->number == 0 || qw > ctx->wmax) ctx->wmax = qw;
  update_scale(ctx);
  // the tile-major loader writes tiles of one extent
  bool tiled_load = ctx->prec == APT_PREC_MIXED && ctx->tiling && base == 0 &&
                    ctx->tiles.ax[0].r == 0 && ctx->tiles.ax[1].r == 0 &&
                    ctx->tiles.ax[2].r == 0;
  if (ctx->prec == APT_PREC_FP64)
    HIPCHK(launch_load_uniform_f64(m, lp, ctx->p64, ctx->d_counters,
                                   ctx->stream));
  else if (tiled_load)
    HIPCHK(launch_load_tiled_f32(m, lp, ctx->tiles, ctx->p32, ctx->d_counters,
                                 ctx->stream));
  else
    HIPCHK(launch_load_uniform_f32(m, lp, ctx->p32, ctx->d_counters,
                                   ctx->stream));
  ctx->number = base + add;
  if (ctx->id_next < ctx->number) ctx->id_next = ctx->number;
  if (fabs(weight) > ctx->wmaxw) ctx->wmaxw = fabs(weight);
  ctx->tiles_valid = false;
  ctx->runs_valid = false;
  if (tiled_load) {
    const uint64_t per = (uint64_t)ctx->tiles.ax[0].w * ctx->tiles.ax[1].w *
                         ctx->tiles.ax[2].w * 2 * (uint64_t)ppc_pairs;
    std::vector<uint32_t> off(ctx->tiles.ntiles + 1);
    for (uint64_t t = 0; t <= ctx->tiles.ntiles; t++) off[t] = (uint32_t)(t * per);
    HIPCHK(hipMemcpyAsync(ctx->tile_off, off.data(), off.size() * 4,
                          hipMemcpyHostToDevice, ctx->stream));
    ctx->tiles.tiled_end = add;
    ctx->drift = 0.0;
    ctx->tiles_valid = true;
    ctx->pushes_since_sort = 0;
  }
  HIPCHK(hipStreamSynchronize(ctx->stream));
  return APT_OK;
}

// ---- the particle step --------------------------------------------------
static apt_status filter_pass(apt_ctx *ctx, void *arr) {
  if (ctx->prec == APT_PREC_FP64)
    HIPCHK(launch_filter<double>(ctx->mesh, (double *)arr,
                                 (double *)ctx->jtmp,
                                 ctx->params.fix_3d_filter, ctx->stream));
  else
    HIPCHK(launch_filter<float>(ctx->mesh, (float *)arr, (float *)ctx->jtmp,
                                ctx->params.fix_3d_filter, ctx->stream));
  return APT_OK;
}

template <typename T>
static apt_status logsph_smooth(apt_ctx *ctx, int rho) {
  const double *A[3] = {ctx->coef.a[LS_A1E], ctx->coef.a[LS_A2E],
                        ctx->coef.a[LS_A3E]};
  for (int pass = 0; pass < ctx->params.current_smoothing; pass++) {
    for (int c = 0; c < 3; c++)
      HIPCHK(launch_logsph_filter<T>(ctx->mesh, (T *)ctx->J[c], (T *)ctx->jtmp,
                                     A[c], ctx->stream));
    if (rho)
      for (int s = 0; s < ctx->params.num_species; s++)
        HIPCHK(launch_logsph_filter<T>(ctx->mesh, (T *)ctx->Rho[s],
                                       (T *)ctx->jtmp, ctx->coef.a[LS_DV],
                                       ctx->stream));
  }
  return APT_OK;
}

static apt_status smooth(apt_ctx *ctx, int rho) {
  if (ctx->logsph)
    return ctx->prec == APT_PREC_FP64 ? logsph_smooth<double>(ctx, rho)
                                      : logsph_smooth<float>(ctx, rho);
  for (int pass = 0; pass < ctx->params.current_smoothing; pass++) {
    for (int c = 0; c < 3; c++) {
      apt_status st = filter_pass(ctx, ctx->J[c]);
      if (st != APT_OK) return st;
    }
    if (rho)
      for (int s = 0; s < ctx->params.num_species; s++) {
        apt_status st = filter_pass(ctx, ctx->Rho[s]);
        if (st != APT_OK) return st;
      }
  }
  return APT_OK;
}

// The accumulators of a Cartesian step into J (and, on deposit steps, Rho; Rho
// is cleared on the others, unless it is clear) and current_smoothing filter
// passes over them.  Where the filter can write guard images itself the passes
// alternate between the field and a work array, and the finalization starts
// with whichever makes the last pass end in the field.
template <typename T>
static apt_status finalize_smooth(apt_ctx *ctx, int rho) {
  const int passes = ctx->params.current_smoothing, ns = ctx->params.num_species;
  const bool fused = passes > 0 && ctx->ftmp[2] && guard_images_ok(ctx->mesh);
  T *tmp[4] = {(T *)ctx->jtmp, (T *)ctx->ftmp[0], (T *)ctx->ftmp[1], (T *)ctx->ftmp[2]};
  const bool odd = fused && (passes & 1);
  auto run = [&](void *const *field, int n) -> apt_status {
    for (int k = 0; k < passes; k++) {
      const bool from_tmp = ((passes - k) & 1) != 0;  // the last pass writes the field
      T *const *fld = (T *const *)field;
      HIPCHK(launch_filter_set<T>(ctx->mesh, from_tmp ? tmp : fld, from_tmp ? fld : tmp, n,
                                  ctx->params.fix_3d_filter, ctx->stream));
    }
    return APT_OK;
  };
  FinalizeSet<T> fs;
  for (int c = 0; c < 3; c++) {
    fs.hi[c] = ctx->Jacc[c][0];
    fs.lo[c] = ctx->Jacc[c][1];
    fs.out[c] = odd ? tmp[c] : (T *)ctx->J[c];
  }
  fs.n = 3;
  if (!rho && (!ctx->rho_zero || ctx->capturing)) {
    for (int s = 0; s < 4; s++) fs.zero[s] = (T *)ctx->Rho[s];
    fs.nzero = 4;
  }
  HIPCHK(launch_finalize_set<T>(fs, ctx->ncell, ctx->H, ctx->stream));
  if (!ctx->capturing) ctx->rho_zero = !rho;
  if (fused) {
    apt_status st = run(ctx->J, 3);
    if (st != APT_OK) return st;
  }
  if (rho) {
    // every allocated charge slot (see apt_create); the filter covers the
    // species in use
    for (int s = 0; s < 4; s++) {
      fs.hi[s] = ctx->Racc[s][0];
      fs.lo[s] = ctx->Racc[s][1];
      fs.out[s] = odd && s < ns ? tmp[s] : (T *)ctx->Rho[s];
    }
    fs.n = 4;
    fs.nzero = 0;
    HIPCHK(launch_finalize_set<T>(fs, ctx->ncell, ctx->H, ctx->stream));
    if (fused) {
      apt_status st = run(ctx->Rho, ns);
      if (st != APT_OK) return st;
    }
  }
  return fused ? APT_OK : smooth(ctx, rho);
}

apt_status apt_smooth_current(apt_ctx *ctx, uint32_t step) {
  CHECK_CTX(ctx);
  const int di = ctx->params.data_interval > 0 ? ctx->params.data_interval : 1;
  return smooth(ctx, ((step + 1) % (uint32_t)di) == 0);
}

// device-count mode: the device-resident particle / photon counts that
// bound the slots a kernel processes (the host counts are upper bounds)
static const unsigned long long *dn_ptc(const apt_ctx *ctx) {
  return ctx->dcount ? ctx->d_dc + DC_NUM : nullptr;
}
static const unsigned long long *dn_ph(const apt_ctx *ctx) {
  return ctx->dcount ? ctx->d_dc + DC_PH : nullptr;
}

static apt_status move_photons(apt_ctx *ctx, double dt) {
  if (ctx->ph_number == 0) return APT_OK;
  const int ls = ctx->logsph ? 1 : 0;
  if (ctx->prec == APT_PREC_FP64)
    HIPCHK(rt_move_photons<double>(ctx->mesh, ls, ctx->rt.r_cutoff,
                                   view_of(ctx->ph64), ctx->ph_number, dt,
                                   ctx->stream, dn_ph(ctx)));
  else
    HIPCHK(rt_move_photons<float>(ctx->mesh, ls, ctx->rt.r_cutoff,
                                  view_of(ctx->ph32), ctx->ph_number, dt,
                                  ctx->stream, dn_ph(ctx)));
  if (ctx->logsph) {
    uint32_t *cell = ctx->prec == APT_PREC_FP64 ? ctx->ph64.cell : ctx->ph32.cell;
    HIPCHK(launch_erase_guard(ctx->mesh, cell, ctx->ph_number, ctx->stream, dn_ph(ctx)));
  }
  return APT_OK;
}

// ptc_updater_logsph::update_particles + apply_boundary
// (ptc_updater_logsph.cu:681-846): push + move + deposit (with the guard erase
// and the outflow flag), process_j, smoothing, axis J3, photon move.
static apt_status logsph_ptc_update(apt_ctx *ctx, double dt, int rho) {
  const int ns = 4;  // every allocated charge slot (see apt_create)
  if (ctx->dcount) HIPCHK(launch_dc_accum(ctx->d_dc, DC_PUSHED, DC_NUM, ctx->stream));
  time_begin(ctx, APT_KERNEL_PUSH_DEPOSIT);
  const CellRuns *runs = ctx->runs_valid && ctx->runs.end > 0 ? &ctx->runs : nullptr;
  if (ctx->prec == APT_PREC_FP64) {
    FieldsF64 f;
    AccF64 a;
    for (int c = 0; c < 3; c++) {
      f.E[c] = (const double *)ctx->E[c];
      f.B[c] = (const double *)ctx->B[c];
      a.J[c][0] = ctx->Jacc[c][0];
      a.J[c][1] = ctx->Jacc[c][1];
    }
    for (int s = 0; s < 4; s++) {
      a.R[s][0] = ctx->Racc[s][0];
      a.R[s][1] = ctx->Racc[s][1];
    }
    HIPCHK(launch_logsph_push_f64(ctx->mesh, ctx->sp, ctx->lp, dt, ctx->H, rho,
                                  ctx->p64, f, a, ctx->d_counters, ctx->number,
                                  ctx->stream, dn_ptc(ctx), runs));
  } else {
    FieldsF32 f;
    AccMixed a;
    for (int c = 0; c < 3; c++) {
      f.E[c] = (const float *)ctx->E[c];
      f.B[c] = (const float *)ctx->B[c];
      a.J[c] = ctx->Jacc[c][0];
    }
    for (int s = 0; s < 4; s++) a.R[s] = ctx->Racc[s][0];
    a.rho = rho;
    HIPCHK(launch_logsph_push_f32(ctx->mesh, ctx->sp, ctx->lp, (float)dt,
                                  ctx->H, ctx->p32, f, a, ctx->d_counters,
                                  ctx->number, ctx->stream, dn_ptc(ctx), runs));
  }
  time_end(ctx, APT_KERNEL_PUSH_DEPOSIT);
  const int limbs = ctx->prec == APT_PREC_FP64 ? 2 : 1;
  // Rho holds what a step without charge output writes: nothing to do for it
  const int nr = rho || !ctx->rho_zero || ctx->capturing ? ns : 0;
  const int smoothed = ctx->params.current_smoothing > 0;
  if (ctx->prec == APT_PREC_FP64)
    HIPCHK(launch_logsph_process_j<double>(ctx->mesh, ctx->coef, dt, ctx->H, limbs,
                                           ctx->Jacc, ctx->Racc, nr,
                                           (double *const *)ctx->J,
                                           (double *const *)ctx->Rho, !smoothed, ctx->stream));
  else
    HIPCHK(launch_logsph_process_j<float>(ctx->mesh, ctx->coef, dt, ctx->H, limbs,
                                          ctx->Jacc, ctx->Racc, nr,
                                          (float *const *)ctx->J,
                                          (float *const *)ctx->Rho, !smoothed, ctx->stream));
  if (!ctx->capturing) ctx->rho_zero = !rho;
  if (smoothed) {
    apt_status st = smooth(ctx, rho);
    if (st != APT_OK) return st;
    if (ctx->prec == APT_PREC_FP64)
      HIPCHK(launch_logsph_axis_j3<double>(ctx->mesh, (double *)ctx->J[2], ctx->stream));
    else
      HIPCHK(launch_logsph_axis_j3<float>(ctx->mesh, (float *)ctx->J[2], ctx->stream));
  }
  return move_photons(ctx, dt);
}

// ---- 1D GR gap -------------------------------------------------------
// Grid_1dGR::compute_coef (grid_1dgr.cpp:21-175) on the host: the profile
// arrays are taken as float, as the reference reads coef.h5
// (grid_1dgr.cpp:60-66); the build's own exp/sin/cos keep the result
// identical to the CPU restatement.
static double gr_sq(double x) { return x * x; }

static bool gr1d_coef_host(const Mesh &m, const float *vr, const float *vB1,
                           const float *vB3, const float *vrho, const float *vjr,
                           const float *vth, const float *vdpsi, uint64_t nprof,
                           double a, double omega, double B0, std::vector<double> *coef) {
  const int n_size = m.dims[0];
  for (int k = 0; k < GR_NCOEF; k++) coef[k].assign(n_size, 0.0);
  auto r_of_xi = [&](double xi) {
    const double rp = 1.0 + sqrt(1.0 - a * a), rm = 1.0 - sqrt(1.0 - a * a);
    const double e = apt_exp(xi * (rp - rm));
    return (rp - rm * e) / (1.0 - e);
  };
  uint64_t n_data = 0, n_mid = 0;
  for (int n = 0; n < n_size; n++) {
    const double xi = m.lower[0] + (double)(n - m.guard[0] + 1) * m.delta[0];
    const double r = r_of_xi(xi);
    while (n_data + 1 < nprof && vr[n_data + 1] < r) n_data += 1;
    if (n_data + 1 >= nprof) return false;
    const double x = (r - vr[n_data]) / (vr[n_data + 1] - vr[n_data]);
    const double B1 = vB1[n_data] * (1.0 - x) + vB1[n_data + 1] * x;
    const double B3 = vB3[n_data] * (1.0 - x) + vB3[n_data + 1] * x;
    const double theta = vth[n_data] * (1.0 - x) + vth[n_data + 1] * x;
    const double b31 = B3 / B1;
    coef[GR_B3B1][n] = b31;
    coef[GR_RHO0][n] = B0 * (vrho[n_data] * (1.0 - x) + vrho[n_data + 1] * x);
    double st, ct;
    apt_sincos(theta, st, ct);
    double Sigma = r * r + a * a * gr_sq(ct);
    double Delta = r * r - 2.0 * r + a * a;
    double A = gr_sq(r * r + a * a) - Delta * a * a * gr_sq(st);
    const double w = 2.0 * a * r / A;
    double g11 = Sigma / Delta;
    double g22 = Sigma;
    double g33 = A * gr_sq(st) / Sigma;
    double sqrt_gamma = sqrt(g11 * g22 * g33);
    coef[GR_K1][n] = Delta * sqrt_gamma / (vdpsi[n_data] * (1.0 - x) + vdpsi[n_data + 1] * x);
    coef[GR_D1][n] = (b31 * g33 * (omega - w)) * Delta;
    coef[GR_D2][n] = (g11 + b31 * b31 * g33) * Delta * Delta;
    coef[GR_D3][n] = g33 * gr_sq(omega - w);
    coef[GR_ALPHA][n] = sqrt(Delta * Sigma / A);
    coef[GR_GRR][n] = 1.0 / g11;
    coef[GR_GFF][n] = 1.0 / g33;
    coef[GR_BETA][n] = -2.0 * a * r / A;

    const double xi_mid = m.lower[0] + ((double)(n - m.guard[0]) + 0.5) * m.delta[0];
    const double r_mid = r_of_xi(xi_mid);
    while (n_mid + 1 < nprof && vr[n_mid + 1] < r_mid) n_mid += 1;
    if (n_mid + 1 >= nprof) return false;
    // the mid-point quantities are interpolated with the node r, as in
    // the reference (grid_1dgr.cpp:146)
    const double y = (r - vr[n_mid]) / (vr[n_mid + 1] - vr[n_mid]);
    coef[GR_J0][n] = B0 * (vjr[n_mid] * (1.0 - y) + vjr[n_mid + 1] * y) / Delta;
    const double theta_mid = vth[n_mid] * (1.0 - y) + vth[n_mid + 1] * y;
    apt_sincos(theta_mid, st, ct);
    Sigma = r_mid * r_mid + a * a * gr_sq(ct);
    Delta = r_mid * r_mid - 2.0 * r_mid + a * a;
    A = gr_sq(r_mid * r_mid + a * a) - Delta * a * a * gr_sq(st);
    g11 = Sigma / Delta;
    g22 = Sigma;
    g33 = A * gr_sq(st) / Sigma;
    sqrt_gamma = sqrt(g11 * g22 * g33);
    coef[GR_K1J][n] = Delta * sqrt_gamma / (vdpsi[n_mid] * (1.0 - y) + vdpsi[n_mid + 1] * y);
    coef[GR_AGRR][n] = Delta * Delta * sqrt(Delta * Sigma / A) * g11;
  }
  return true;
}

apt_status apt_1dgr_set_profile(apt_ctx *ctx, const double *r, const double *B1,
                                const double *B3, const double *rho, const double *jr,
                                const double *theta, const double *dpsidth, uint64_t n) {
  CHECK_CTX(ctx);
  if (!ctx->gr1d) return ctx->fail(APT_ERR_UNSUPPORTED, "1dgr_set_profile: not a 1D GR context");
  if (!r || !B1 || !B3 || !rho || !jr || !theta || !dpsidth || n < 2)
    return ctx->fail(APT_ERR_INVALID_ARG, "1dgr_set_profile: missing arrays");
  const double *src[7] = {r, B1, B3, rho, jr, theta, dpsidth};
  std::vector<float> f[7];
  for (int k = 0; k < 7; k++) {
    f[k].resize(n);
    for (uint64_t i = 0; i < n; i++) f[k][i] = (float)src[k][i];
  }
  std::vector<double> c[GR_NCOEF];
  if (!gr1d_coef_host(ctx->mesh, f[0].data(), f[1].data(), f[2].data(), f[3].data(),
                      f[4].data(), f[5].data(), f[6].data(), n, ctx->gr_a, ctx->gr_omega,
                      ctx->gr_B0, c))
    return ctx->fail(APT_ERR_INVALID_ARG,
                     "1dgr_set_profile: the grid reaches past the profile's last r");
  HIPCHK(hipStreamSynchronize(ctx->stream));
  for (int k = 0; k < GR_NCOEF; k++) {
    ctx->gr_host[k] = c[k];
    HIPCHK(hipMemcpy(ctx->gr_dev[k], c[k].data(), c[k].size() * 8, hipMemcpyHostToDevice));
  }
  return APT_OK;
}

apt_status apt_1dgr_initial_condition(apt_ctx *ctx, int multiplicity) {
  CHECK_CTX(ctx);
  if (!ctx->gr1d)
    return ctx->fail(APT_ERR_UNSUPPORTED, "1dgr_initial_condition: not a 1D GR context");
  const Mesh &m = ctx->mesh;
  if (multiplicity < 1)
    return ctx->fail(APT_ERR_INVALID_ARG, "1dgr_initial_condition: multiplicity < 1");
  const uint64_t number = (uint64_t)(m.dims[0] - 2 * m.guard[0]) * 2 * (uint64_t)multiplicity;
  if (number > ctx->cap)
    return ctx->fail(APT_ERR_CAPACITY, "1dgr_initial_condition: %llu > capacity %llu",
                     (unsigned long long)number, (unsigned long long)ctx->cap);
  // prepare_initial_condition (ptc_updater_1dgr.cu:16-72): slot
  // cell * 2 mult + 2 n (+1), so the first guard * 2 mult slots stay empty
  // and the last guard cells' pairs fall past number, as in the reference
  std::vector<uint32_t> cell(number, MAX_CELL), flag(number, 0);
  std::vector<double> x1(number, 0.0), zero(number, 0.0), E(number, 0.0), w(number, 0.0);
  std::vector<uint64_t> id(number);
  const double B0 = ctx->gr_B0, track = ctx->gr_track;
  const std::vector<double> *c = ctx->gr_host;
  for (int ci = m.guard[0]; ci < m.dims[0] - m.guard[0]; ci++)
    for (int n = 0; n < multiplicity; n++) {
      const uint64_t idx = (uint64_t)ci * (uint64_t)multiplicity * 2 + (uint64_t)n * 2;
      if (idx + 1 >= number) continue;
      const double D1 = c[GR_D1][ci], D2 = c[GR_D2][ci], D3 = c[GR_D3][ci];
      const double alpha = c[GR_ALPHA][ci], K1 = c[GR_K1][ci], rho0 = c[GR_RHO0][ci];
      const double u0 = sqrt(D2 / (D2 * (alpha * alpha - D3) + D1 * D1));
      const double rk = rho0 * K1;
      double u[2];
      uniform2(ctx->params.random_seed, idx, 0, 8, u[0], u[1]);
      for (int s = 0; s < 2; s++) {
        const uint64_t k = idx + (uint64_t)s;
        x1[k] = 1.0;
        E[k] = u0;
        cell[k] = (uint32_t)ci;
        w[k] = s == 0 ? 1.0 * B0 / multiplicity + fabs(fmin(rk, 0.0)) / multiplicity
                      : 1.0 * B0 / multiplicity + fmax(rk, 0.0) / multiplicity;
        flag[k] = ((uint32_t)s << 29) | (u[s] < track ? FLAG_TRACKED : 0u);
      }
    }
  for (uint64_t k = 0; k < number; k++) id[k] = k;
  apt_particles v{cell.data(), x1.data(), zero.data(), zero.data(), zero.data(),
                  zero.data(),  zero.data(), E.data(), w.data(), flag.data(), id.data()};
  return apt_ptc_set(ctx, &v, number);
}

// ptc_updater_1dgap::prepare_initial_condition (ptc_updater_1dgap.cu:21-72,
// 236-248), built on the host: slot cell * 2 mult + 2 n (+1), so the first
// guard * 2 mult slots stay empty and the last guard cells' pairs fall past
// number, as in the reference.  The offset and the two tracking draws come
// from the Philox stream (seed, slot, 0/1, purpose 14); the offset is
// rounded to float (curand_uniform, Pos_t).
apt_status apt_1dgap_initial_condition(apt_ctx *ctx, int multiplicity) {
  CHECK_CTX(ctx);
  if (!ctx->gap1d)
    return ctx->fail(APT_ERR_UNSUPPORTED, "1dgap_initial_condition: not a 1D gap context");
  const Mesh &m = ctx->mesh;
  if (multiplicity < 1)
    return ctx->fail(APT_ERR_INVALID_ARG, "1dgap_initial_condition: multiplicity < 1");
  const uint64_t number = (uint64_t)(m.dims[0] - 2 * m.guard[0]) * 2 * (uint64_t)multiplicity;
  if (number > ctx->cap)
    return ctx->fail(APT_ERR_CAPACITY, "1dgap_initial_condition: %llu > capacity %llu",
                     (unsigned long long)number, (unsigned long long)ctx->cap);
  std::vector<uint32_t> cell(number, MAX_CELL), flag(number, 0);
  std::vector<double> x1(number, 0.0), zero(number, 0.0), E(number, 0.0), w(number, 0.0);
  std::vector<uint64_t> id(number);
  const float B0 = ctx->gap_B0;
  const double rho0 = (double)(B0 * ctx->gap_omega);
  const double wbase = (double)(2.0f * B0 / (float)multiplicity);
  const double track = ctx->gap_track;
  for (int ci = m.guard[0]; ci < m.dims[0] - m.guard[0]; ci++)
    for (int n = 0; n < multiplicity; n++) {
      const uint64_t idx = (uint64_t)ci * (uint64_t)multiplicity * 2 + (uint64_t)n * 2;
      if (idx + 1 >= number) continue;
      double u[2], v[2];
      uniform2(ctx->params.random_seed, idx, 0, 14, u[0], u[1]);
      uniform2(ctx->params.random_seed, idx, 1, 14, v[0], v[1]);
      const double xo = (double)(float)u[0];
      const double x_pos = m.lower[0] + m.delta[0] * ((double)(ci - m.guard[0]) + xo);
      const double rho = rho0 * atan(2.0 * x_pos);
      const double tu[2] = {u[1], v[0]};
      for (int s = 0; s < 2; s++) {
        const uint64_t k = idx + (uint64_t)s;
        x1[k] = xo;
        E[k] = sqrt(1.0 + x_pos * x_pos);
        cell[k] = (uint32_t)ci;
        w[k] = s == 0 ? wbase + fabs(fmin(rho, 0.0)) / multiplicity
                      : wbase + fmax(rho, 0.0) / multiplicity;
        flag[k] = ((uint32_t)s << 29) | (tu[s] < track ? FLAG_TRACKED : 0u);
      }
    }
  for (uint64_t k = 0; k < number; k++) id[k] = k;
  apt_particles pv{cell.data(), x1.data(), zero.data(), zero.data(), zero.data(),
                   zero.data(),  zero.data(), E.data(), w.data(), flag.data(), id.data()};
  return apt_ptc_set(ctx, &pv, number);
}

// ptc_updater_1dgap::update_particles (ptc_updater_1dgap.cu:196-234): the
// filtered copy of E1 in E[2] (E[1] as the filter's scratch), the push with
// the current and charge deposit (Rho on every step), the smoothing of J1
// and Rho, then the photons.  The filter's open-boundary rows apply on a
// non-periodic line (sim_environment::is_boundary on one rank).
static apt_status gap_ptc_update(apt_ctx *ctx, double dt, uint32_t step) {
  (void)step;
  const Mesh &m = ctx->mesh;
  const uint64_t nc = ctx->ncell;
  const int bnd = m.periodic[0] ? 0 : 1;
  if (ctx->number > 0) {
    double *E0 = (double *)ctx->E[0], *E1 = (double *)ctx->E[1], *E2 = (double *)ctx->E[2];
    HIPCHK(hipMemcpyAsync(E2, E0, nc * 8, hipMemcpyDeviceToDevice, ctx->stream));
    for (int pass = 0; pass < ctx->params.current_smoothing; pass++) {
      HIPCHK(launch_gap_filter(m, E2, E1, bnd, bnd, ctx->stream));
      HIPCHK(hipMemcpyAsync(E2, E1, nc * 8, hipMemcpyDeviceToDevice, ctx->stream));
    }
    AccF64 acc;
    for (int c = 0; c < 3; c++) {
      acc.J[c][0] = ctx->Jacc[c][0];
      acc.J[c][1] = ctx->Jacc[c][1];
    }
    for (int s = 0; s < 4; s++) {
      acc.R[s][0] = ctx->Racc[s][0];
      acc.R[s][1] = ctx->Racc[s][1];
    }
    time_begin(ctx, APT_KERNEL_PUSH_DEPOSIT);
    HIPCHK(launch_gap_push(m, ctx->sp, ctx->p64, E2, acc, dt, ctx->H, ctx->number,
                           ctx->d_counters, ctx->stream));
    time_end(ctx, APT_KERNEL_PUSH_DEPOSIT);
    for (int c = 0; c < 3; c++)
      HIPCHK(launch_finalize_f64(ctx->Jacc[c][0], ctx->Jacc[c][1], (double *)ctx->J[c], nc,
                                 ctx->H, ctx->stream));
    for (int s = 0; s < 4; s++)
      HIPCHK(launch_finalize_f64(ctx->Racc[s][0], ctx->Racc[s][1], (double *)ctx->Rho[s], nc,
                                 ctx->H, ctx->stream));
    double *tmp = (double *)ctx->jtmp;
    for (int pass = 0; pass < ctx->params.current_smoothing; pass++) {
      HIPCHK(launch_gap_filter(m, (double *)ctx->J[0], tmp, bnd, bnd, ctx->stream));
      HIPCHK(hipMemcpyAsync(ctx->J[0], tmp, nc * 8, hipMemcpyDeviceToDevice, ctx->stream));
      for (int s = 0; s < ctx->params.num_species; s++) {
        HIPCHK(launch_gap_filter(m, (double *)ctx->Rho[s], tmp, bnd, bnd, ctx->stream));
        HIPCHK(hipMemcpyAsync(ctx->Rho[s], tmp, nc * 8, hipMemcpyDeviceToDevice, ctx->stream));
      }
    }
  }
  if (ctx->ph_number > 0)
    HIPCHK(launch_gap_photons(m, ctx->ph64, dt, ctx->ph_number, ctx->stream));
  return APT_OK;
}

static Gr1dCoef gr1d_coef(const apt_ctx *ctx) {
  Gr1dCoef cf;
  for (int k = 0; k < GR_NCOEF; k++) cf.a[k] = ctx->gr_dev[k];
  return cf;
}

// ptc_updater_1dgr::update_particles (ptc_updater_1dgr.cu:443-501): the
// filtered E in E[2] (E[1] as the filter's scratch), the push with the
// current and charge deposit, the K-weighted smoothing of J1 and Rho, then
// the photons
static apt_status gr1d_ptc_update(apt_ctx *ctx, double dt, uint32_t step) {
  const Mesh &m = ctx->mesh;
  const Gr1dCoef cf = gr1d_coef(ctx);
  const uint64_t nc = ctx->ncell;
  const int di = ctx->params.data_interval;
  if (ctx->number > 0) {
    double *E0 = (double *)ctx->E[0], *E1 = (double *)ctx->E[1], *E2 = (double *)ctx->E[2];
    HIPCHK(hipMemcpyAsync(E2, E0, nc * 8, hipMemcpyDeviceToDevice, ctx->stream));
    for (int pass = 0; pass < ctx->params.current_smoothing; pass++) {
      HIPCHK(launch_1dgr_filter(m, E2, E1, cf.a[GR_K1J], ctx->stream));
      HIPCHK(hipMemcpyAsync(E2, E1, nc * 8, hipMemcpyDeviceToDevice, ctx->stream));
    }
    AccF64 acc;
    for (int c = 0; c < 3; c++) {
      acc.J[c][0] = ctx->Jacc[c][0];
      acc.J[c][1] = ctx->Jacc[c][1];
    }
    for (int s = 0; s < 4; s++) {
      acc.R[s][0] = ctx->Racc[s][0];
      acc.R[s][1] = ctx->Racc[s][1];
    }
    time_begin(ctx, APT_KERNEL_PUSH_DEPOSIT);
    HIPCHK(launch_1dgr_push(m, cf, ctx->sp, ctx->p64, E2, acc, dt, step, di, ctx->gr_a,
                            ctx->gr_omega, ctx->H, ctx->number, ctx->stream));
    time_end(ctx, APT_KERNEL_PUSH_DEPOSIT);
    for (int c = 0; c < 3; c++)
      HIPCHK(launch_finalize_f64(ctx->Jacc[c][0], ctx->Jacc[c][1], (double *)ctx->J[c], nc,
                                 ctx->H, ctx->stream));
    for (int s = 0; s < 4; s++)
      HIPCHK(launch_finalize_f64(ctx->Racc[s][0], ctx->Racc[s][1], (double *)ctx->Rho[s], nc,
                                 ctx->H, ctx->stream));
    double *tmp = (double *)ctx->jtmp;
    for (int pass = 0; pass < ctx->params.current_smoothing; pass++) {
      HIPCHK(launch_1dgr_filter(m, (double *)ctx->J[0], tmp, cf.a[GR_K1J], ctx->stream));
      HIPCHK(hipMemcpyAsync(ctx->J[0], tmp, nc * 8, hipMemcpyDeviceToDevice, ctx->stream));
      for (int s = 0; s < ctx->params.num_species; s++) {
        HIPCHK(launch_1dgr_filter(m, (double *)ctx->Rho[s], tmp, cf.a[GR_K1], ctx->stream));
        HIPCHK(hipMemcpyAsync(ctx->Rho[s], tmp, nc * 8, hipMemcpyDeviceToDevice, ctx->stream));
      }
    }
  }
  if (ctx->ph_number > 0)
    HIPCHK(launch_1dgr_photons(m, cf, ctx->ph64, dt, step, di, ctx->ph_number, ctx->stream));
  return APT_OK;
}

apt_status apt_ptc_update(apt_ctx *ctx, double dt, uint32_t step) {
  CHECK_CTX(ctx);
  if (ctx->gr1d) {
    if (!(dt > 0.0)) return ctx->fail(APT_ERR_INVALID_ARG, "ptc_update: dt must be > 0");
    return gr1d_ptc_update(ctx, dt, step);
  }
  if (ctx->gap1d) {
    if (!(dt > 0.0)) return ctx->fail(APT_ERR_INVALID_ARG, "ptc_update: dt must be > 0");
    return gap_ptc_update(ctx, dt, step);
  }
  const int di = ctx->params.data_interval > 0 ? ctx->params.data_interval : 1;
  const int rho = ((step + 1) % (uint32_t)di) == 0;
  if (ctx->logsph) {
    if (ctx->mesh.dim != 2)
      return ctx->fail(APT_ERR_UNSUPPORTED, "ptc_update: 3D log-spherical contexts "
                                            "carry the force-free solver only");
    if (!(dt > 0.0))
      return ctx->fail(APT_ERR_INVALID_ARG, "ptc_update: dt must be > 0");
    return logsph_ptc_update(ctx, dt, rho);
  }
  if (ctx->prec == APT_PREC_FP64) {
    FieldsF64 f;
    for (int c = 0; c < 3; c++) {
      f.E[c] = (const double *)ctx->E[c];
      f.B[c] = (const double *)ctx->B[c];
    }
    AccF64 a;
    for (int c = 0; c < 3; c++) {
      a.J[c][0] = ctx->Jacc[c][0];
      a.J[c][1] = ctx->Jacc[c][1];
    }
    for (int s = 0; s < 4; s++) {
      a.R[s][0] = ctx->Racc[s][0];
      a.R[s][1] = ctx->Racc[s][1];
    }
    time_begin(ctx, APT_KERNEL_PUSH_DEPOSIT);
    // slots sorted by cell by tile, those appended since (or all of them,
    // before the first sort) in chunks of consecutive slots
    const uint64_t sorted = ctx->runs_valid ? ctx->runs.end : 0;
    if (sorted > 0)
      HIPCHK(launch_push_deposit_f64_runs(ctx->mesh, ctx->sp, dt, ctx->H, rho, ctx->p64, f, a,
                                          ctx->runs, ctx->d_counters, ctx->stream));
    HIPCHK(launch_push_deposit_f64(ctx->mesh, ctx->sp, dt, ctx->H, rho, ctx->params.num_species,
                                   slots_from(ctx->p64, sorted), f, a, ctx->d_counters,
                                   ctx->number - sorted, ctx->stream));
    time_end(ctx, APT_KERNEL_PUSH_DEPOSIT);
    apt_status st = finalize_smooth<double>(ctx, rho);
    if (st != APT_OK) return st;
  } else {
    FieldsF32 f;
    for (int c = 0; c < 3; c++) {
      f.E[c] = (const float *)ctx->E[c];
      f.B[c] = (const float *)ctx->B[c];
    }
    if (ctx->mesh.dim == 3 && ctx->tiles_valid && !ctx->capturing) {
      const int iv = ctx->params.cell_order_interval == 0 ? 5 : ctx->params.cell_order_interval;
      // a re-layout drops a recorded step; where an axis is no multiple of the
      // tile extent it waits for the recording to go instead
      bool ragged = false;
      for (int d = 0; d < 3; d++) ragged = ragged || ctx->mesh.N[d] % ctx->tiles.T[d] != 0;
      if (iv > 0 && ctx->pushes_since_sort > 0 && ctx->pushes_since_sort % (uint32_t)iv == 0 &&
          tile_cellsort_supported(ctx->tiles) && !(ragged && ctx->gexec)) {
        apt_status st = relayout_tiles(ctx);
        if (st != APT_OK) return st;
      }
      ctx->pushes_since_sort++;
    }
    TileInfo ti = ctx->tiles;
    if (ctx->tiles_by_drift) {
      // a recorded step takes the large halo: it may be replayed at any drift
      double step_cells = 0.0;
      for (int d = 0; d < 3; d++) step_cells = fmax(step_cells, fabs(dt) * ctx->mesh.inv_delta[d]);
      if (!ctx->capturing) ctx->drift += step_cells;
      if ((!ctx->capturing && ctx->drift <= 2.5) || ti.tiled_end < 192ull * ti.ntiles) {
        ti.halo = 3;
        ti.threads = 256;
      }
    }
    if (!ctx->tiles_valid) {
      ti.tile_off = nullptr;
      ti.ntiles = 0;
      ti.tiled_end = 0;
    }
    AccMixed a;
    for (int c = 0; c < 3; c++) a.J[c] = ctx->Jacc[c][0];
    for (int s = 0; s < 4; s++) a.R[s] = ctx->Racc[s][0];
    a.rho = rho;
    time_begin(ctx, APT_KERNEL_PUSH_DEPOSIT);
    const uint64_t sorted = ctx->runs_valid ? ctx->runs.end : 0;  // untiled, sorted by cell
    if (sorted > 0)
      HIPCHK(launch_push_deposit_mixed_runs(ctx->mesh, ctx->sp, (float)dt, ctx->H, ctx->p32, f, a,
                                            ctx->runs, ctx->d_counters, ctx->stream));
    HIPCHK(launch_push_deposit_mixed(ctx->mesh, ctx->sp, (float)dt, ctx->H,
                                     ctx->p32, f, a, ti, ctx->d_counters,
                                     ctx->number, ctx->stream, sorted));
    time_end(ctx, APT_KERNEL_PUSH_DEPOSIT);
    apt_status st = finalize_smooth<float>(ctx, rho);
    if (st != APT_OK) return st;
  }
  return move_photons(ctx, dt);
}

// ---- fields --------------------------------------------------------------
template <typename T>
static FieldSet<T> field_set(apt_ctx *ctx) {
  FieldSet<T> f;
  for (int c = 0; c < 3; c++) {
    f.E[c] = (T *)ctx->E[c];
    f.B[c] = (T *)ctx->B[c];
    f.Ebg[c] = (const T *)ctx->Ebg[c];
    f.Bbg[c] = (const T *)ctx->Bbg[c];
    f.J[c] = (const T *)ctx->J[c];
  }
  f.divE = (T *)ctx->divE;
  f.divB = (T *)ctx->divB;
  f.EdotB = (T *)ctx->EdotB;
  // a recorded step reads them: they may be set before a replay
  f.has_ebg = !ctx->ebg_zero || ctx->capturing;
  f.has_bbg = !ctx->bbg_zero || ctx->capturing;
  return f;
}

template <typename T>
static apt_status update_e_t(apt_ctx *ctx, double dt) {
  HIPCHK(launch_update_e<T>(ctx->mesh, field_set<T>(ctx), dt, ctx->stream));
  return APT_OK;
}
template <typename T>
static apt_status update_b_t(apt_ctx *ctx, double dt) {
  HIPCHK(launch_update_b<T>(ctx->mesh, field_set<T>(ctx), dt, ctx->stream,
                            ctx->params.reference_3d_b_stencil));
  return APT_OK;
}
template <typename T>
static apt_status divs_t(apt_ctx *ctx) {
  HIPCHK(launch_divs<T>(ctx->mesh, field_set<T>(ctx), ctx->stream));
  return APT_OK;
}

template <typename T>
static apt_status field_update_t(apt_ctx *ctx, double dt, uint32_t step) {
  apt_status st;
  time_begin(ctx, APT_KERNEL_FIELD);
  if (step == 0 && (st = update_e_t<T>(ctx, 0.5 * dt)) != APT_OK) return st;
  if ((st = update_b_t<T>(ctx, dt)) != APT_OK) return st;
  if ((st = update_e_t<T>(ctx, dt)) != APT_OK) return st;
  if ((st = divs_t<T>(ctx)) != APT_OK) return st;
  time_end(ctx, APT_KERNEL_FIELD);
  return APT_OK;
}

template <typename T>
static apt_status logsph_field_update_t(apt_ctx *ctx, double dt) {
  time_begin(ctx, APT_KERNEL_FIELD);
  // compute_edotb's delta is the float 1.0f / data_interval
  // (cuda/sim_data.cu:60)
  const int di = ctx->params.data_interval > 0 ? ctx->params.data_interval : 1;
  const double delta = (double)(1.0f / (float)di);
  HIPCHK(launch_logsph_field_update<T>(ctx->mesh, ctx->coef, ctx->lp,
                                       field_set<T>(ctx), dt, delta, ctx->stream));
  time_end(ctx, APT_KERNEL_FIELD);
  return APT_OK;
}

apt_status apt_field_update(apt_ctx *ctx, double dt, uint32_t step) {
  CHECK_CTX(ctx);
  if (ctx->gap1d) {  // field_solver_1dgap::update_fields (field_solver_1dgap.cu:31-39)
    time_begin(ctx, APT_KERNEL_FIELD);
    HIPCHK(launch_gap_update_e(ctx->mesh, (double *)ctx->E[0], (const double *)ctx->J[0],
                               (double)ctx->gap_B0 * 1.6, dt, ctx->stream));
    time_end(ctx, APT_KERNEL_FIELD);
    return APT_OK;
  }
  if (ctx->gr1d) {  // field_solver_1dgr::update_fields (field_solver_1dgr.cu:46-58)
    time_begin(ctx, APT_KERNEL_FIELD);
    HIPCHK(launch_1dgr_update_e(ctx->mesh, gr1d_coef(ctx), (double *)ctx->E[0],
                                (const double *)ctx->J[0], dt, ctx->stream));
    time_end(ctx, APT_KERNEL_FIELD);
    return APT_OK;
  }
  if (ctx->logsph && ctx->mesh.dim != 2)
    return ctx->fail(APT_ERR_UNSUPPORTED, "field_update: use apt_ffe_update in 3D");
  if (ctx->logsph)
    return ctx->prec == APT_PREC_FP64 ? logsph_field_update_t<double>(ctx, dt)
                                      : logsph_field_update_t<float>(ctx, dt);
  return ctx->prec == APT_PREC_FP64 ? field_update_t<double>(ctx, dt, step)
                                    : field_update_t<float>(ctx, dt, step);
}

apt_status apt_field_boundary(apt_ctx *ctx, double omega, double time) {
  CHECK_CTX(ctx);
  (void)time;
  if (!ctx->logsph) return APT_OK;
  if (ctx->mesh.dim != 2)
    return ctx->fail(APT_ERR_UNSUPPORTED, "field_boundary: use apt_ffe_boundary in 3D");
  if (ctx->prec == APT_PREC_FP64)
    HIPCHK(launch_logsph_field_boundary<double>(ctx->mesh, ctx->lp,
                                                field_set<double>(ctx), omega,
                                                ctx->stream));
  else
    HIPCHK(launch_logsph_field_boundary<float>(ctx->mesh, ctx->lp,
                                               field_set<float>(ctx), omega,
                                               ctx->stream));
  return APT_OK;
}

static apt_status inject_common(apt_ctx *ctx, int r_cells, int inj_per_cell, double p1,
                                double theta, double w);

apt_status apt_inject_ptc(apt_ctx *ctx, int inj_per_cell, double p1,
                          double p2, double p3, double w, double omega) {
  CHECK_CTX(ctx);
  (void)p2;
  (void)p3;
  (void)omega;
  return inject_common(ctx, 0, inj_per_cell, p1, 0.0, w);
}

apt_status apt_inject_ptc_thermal(apt_ctx *ctx, int r_cells, int inj_per_cell, double theta,
                                  double w, double omega) {
  CHECK_CTX(ctx);
  (void)omega;
  if (r_cells < 1 || r_cells > 16 || !(theta > 0.0))
    return ctx->fail(APT_ERR_INVALID_ARG, "inject_ptc_thermal: 1 <= r_cells <= 16, theta > 0");
  if (ctx->logsph && ctx->mesh.dim == 2 && 2 + r_cells > ctx->mesh.N[0])
    return ctx->fail(APT_ERR_INVALID_ARG, "inject_ptc_thermal: %d radial cells past the grid",
                     r_cells);
  return inject_common(ctx, r_cells, inj_per_cell, 0.0, theta, w);
}

// r_cells = 0: inject_ptc's single cell and fixed momentum
static apt_status inject_common(apt_ctx *ctx, int r_cells, int inj_per_cell, double p1,
                                double theta, double w) {
  if (!ctx->logsph || ctx->mesh.dim != 2)
    return ctx->fail(APT_ERR_UNSUPPORTED, "inject_ptc: 2D log-spherical contexts only");
  if (inj_per_cell < 1)
    return ctx->fail(APT_ERR_INVALID_ARG, "inject_ptc: inj_per_cell < 1");
  if (ctx->capturing && !ctx->dcount)
    return ctx->fail(APT_ERR_STATE, "inject_ptc: a recorded step changes counts only with "
                                    "device counts on (apt_set_device_counts)");
  const uint64_t rows = (uint64_t)ctx->mesh.N[1] - 2;
  const uint64_t add = rows * (uint64_t)(r_cells > 0 ? r_cells : 1) * inj_per_cell * 2;
  if (add / 2 >= (1ull << 31))
    return ctx->fail(APT_ERR_INVALID_ARG, "inject_ptc: %llu pairs in one call",
                     (unsigned long long)(add / 2));
  // device-count mode: pairs past the capacity are dropped on the device
  // and counted as overflow (the exact count is not known here)
  if (!ctx->dcount && ctx->number + add > ctx->cap)
    return ctx->fail(APT_ERR_CAPACITY, "inject_ptc: %llu particles > capacity",
                     (unsigned long long)(ctx->number + add));
  if (fabs(w) > ctx->wmaxw) ctx->wmaxw = fabs(w);
  double qw = fabs(ctx->params.q_e * w);
  if (qw > ctx->wmax) {
    ctx->wmax = qw;
    update_scale(ctx);
  }
  const int Hs = surface_scale(ctx);
  if (ctx->prec == APT_PREC_FP64)
    HIPCHK(launch_logsph_inject<double>(ctx->mesh, ctx->lp, view_of(ctx->p64),
                                        ctx->number, inj_per_cell, p1, w,
                                        ctx->params.q_e, ctx->params.random_seed,
                                        ctx->inject_epoch, Hs, ctx->id_next,
                                        ctx->surf, ctx->stream, r_cells, theta,
                                        ctx->dcount ? ctx->d_dc : nullptr, ctx->cap,
                                        ctx->d_counters));
  else
    HIPCHK(launch_logsph_inject<float>(ctx->mesh, ctx->lp, view_of(ctx->p32),
                                       ctx->number, inj_per_cell, p1, w,
                                       ctx->params.q_e, ctx->params.random_seed,
                                       ctx->inject_epoch, Hs, ctx->id_next,
                                       ctx->surf, ctx->stream, r_cells, theta,
                                       ctx->dcount ? ctx->d_dc : nullptr, ctx->cap,
                                       ctx->d_counters));
  ctx->inject_epoch++;
  ctx->number = ctx->number + add < ctx->cap ? ctx->number + add : ctx->cap;
  ctx->id_next += add;
  return APT_OK;
}

// ---- force-free / vacuum solver (3D log-spherical) ---------------------
template <typename T>
static apt_status ffe_buffers(apt_ctx *ctx, FfeBuf<T> &b) {
  for (int k = 0; k < 12; k++) {
    if (!ctx->ffe[k]) {
      HIPCHK(hipMalloc(&ctx->ffe[k], ctx->ncell * sizeof(T)));
      HIPCHK(launch_fill<T>((T *)ctx->ffe[k], (T)0, ctx->ncell, ctx->stream));
    }
  }
  for (int q = 0; q < 3; q++) {
    b.En[q] = (T *)ctx->ffe[q];
    b.Bn[q] = (T *)ctx->ffe[3 + q];
    b.dE[q] = (T *)ctx->ffe[6 + q];
    b.dB[q] = (T *)ctx->ffe[9 + q];
  }
  return APT_OK;
}

static apt_status ffe_check(apt_ctx *ctx, const char *what) {
  if (!ctx->logsph || ctx->mesh.dim != 3)
    return ctx->fail(APT_ERR_UNSUPPORTED, "%s: 3D log-spherical contexts only", what);
  return APT_OK;
}

template <typename T>
static apt_status ffe_update_t(apt_ctx *ctx, double dt, double omega,
                               double time) {
  FfeBuf<T> b;
  apt_status st = ffe_buffers<T>(ctx, b);
  if (st != APT_OK) return st;
  time_begin(ctx, APT_KERNEL_FIELD);
  HIPCHK(launch_ffe_update<T>(ctx->mesh, ctx->coef, ctx->lp.damping_length,
                              ctx->lp.damping_coef, field_set<T>(ctx), b, dt,
                              omega, time, ctx->stream));
  time_end(ctx, APT_KERNEL_FIELD);
  return APT_OK;
}

apt_status apt_ffe_update(apt_ctx *ctx, double dt, double omega, double time) {
  CHECK_CTX(ctx);
  apt_status st = ffe_check(ctx, "ffe_update");
  if (st != APT_OK) return st;
  return ctx->prec == APT_PREC_FP64 ? ffe_update_t<double>(ctx, dt, omega, time)
                                    : ffe_update_t<float>(ctx, dt, omega, time);
}

apt_status apt_ffe_boundary(apt_ctx *ctx, double omega, double time) {
  CHECK_CTX(ctx);
  (void)time;
  apt_status st = ffe_check(ctx, "ffe_boundary");
  if (st != APT_OK) return st;
  if (ctx->prec == APT_PREC_FP64)
    HIPCHK(launch_ffe_boundary<double>(ctx->mesh, ctx->lp.damping_length,
                                       ctx->lp.damping_coef,
                                       field_set<double>(ctx), omega, ctx->stream));
  else
    HIPCHK(launch_ffe_boundary<float>(ctx->mesh, ctx->lp.damping_length,
                                      ctx->lp.damping_coef,
                                      field_set<float>(ctx), omega, ctx->stream));
  return APT_OK;
}

template <typename T>
static apt_status ffe_clean_t(apt_ctx *ctx, int mode) {
  FfeBuf<T> b;
  apt_status st = ffe_buffers<T>(ctx, b);
  if (st != APT_OK) return st;
  HIPCHK(launch_ffe_clean<T>(ctx->mesh, field_set<T>(ctx), b, mode, ctx->stream));
  return APT_OK;
}

apt_status apt_ffe_clean_epar(apt_ctx *ctx) {
  CHECK_CTX(ctx);
  apt_status st = ffe_check(ctx, "ffe_clean_epar");
  if (st != APT_OK) return st;
  return ctx->prec == APT_PREC_FP64 ? ffe_clean_t<double>(ctx, 0)
                                    : ffe_clean_t<float>(ctx, 0);
}

apt_status apt_ffe_check_egtb(apt_ctx *ctx) {
  CHECK_CTX(ctx);
  apt_status st = ffe_check(ctx, "ffe_check_egtb");
  if (st != APT_OK) return st;
  return ctx->prec == APT_PREC_FP64 ? ffe_clean_t<double>(ctx, 1)
                                    : ffe_clean_t<float>(ctx, 1);
}

apt_status apt_emit_photons(apt_ctx *ctx, uint64_t *emitted) {
  CHECK_CTX(ctx);
  if (ctx->ph_cap == 0)
    return ctx->fail(APT_ERR_STATE, "emit_photons: max_photon_number is 0");
  if (ctx->capturing && !ctx->dcount)
    return ctx->fail(APT_ERR_STATE, "emit_photons: a recorded step changes counts only with "
                                    "device counts on (apt_set_device_counts)");
  if (ctx->dcount && emitted && ctx->capturing)
    return ctx->fail(APT_ERR_STATE, "emit_photons: no event count while a step is recorded");
  uint64_t k = 0;
  const uint64_t seed = ctx->params.random_seed;
  unsigned long long *dc = ctx->dcount ? ctx->d_dc : nullptr;
  if (ctx->prec == APT_PREC_FP64)
    HIPCHK(rt_emit<double>(ctx->mesh, ctx->rt, view_of(ctx->p64), ctx->number,
                           view_of(ctx->ph64), ctx->ph_number, seed,
                           ctx->rt_epoch, ctx->ph_id_next, ctx->rtw,
                           ctx->d_counters, ctx->stream, (double *)ctx->ph_produced, &k, dc));
  else
    HIPCHK(rt_emit<float>(ctx->mesh, ctx->rt, view_of(ctx->p32), ctx->number,
                          view_of(ctx->ph32), ctx->ph_number, seed,
                          ctx->rt_epoch, ctx->ph_id_next, ctx->rtw,
                          ctx->d_counters, ctx->stream, (float *)ctx->ph_produced, &k, dc));
  ctx->rt_epoch++;
  if (ctx->dcount) {
    // at most one photon per particle slot below the particle bound
    const uint64_t b = ctx->ph_number + ctx->number;
    ctx->ph_number = b < ctx->ph_cap ? b : ctx->ph_cap;
    if (emitted) {
      unsigned long long h = 0;
      HIPCHK(hipMemcpyAsync(&h, ctx->d_dc + DC_LAST, 8, hipMemcpyDeviceToHost, ctx->stream));
      HIPCHK(hipStreamSynchronize(ctx->stream));
      *emitted = h;
    }
    return APT_OK;
  }
  ctx->ph_number += k;
  ctx->ph_id_next += k;
  if (emitted) *emitted = k;
  return APT_OK;
}

apt_status apt_produce_pairs(apt_ctx *ctx, uint64_t *pairs) {
  CHECK_CTX(ctx);
  if (ctx->ph_cap == 0)
    return ctx->fail(APT_ERR_STATE, "produce_pairs: max_photon_number is 0");
  if (ctx->capturing && !ctx->dcount)
    return ctx->fail(APT_ERR_STATE, "produce_pairs: a recorded step changes counts only with "
                                    "device counts on (apt_set_device_counts)");
  if (ctx->dcount && pairs && ctx->capturing)
    return ctx->fail(APT_ERR_STATE, "produce_pairs: no event count while a step is recorded");
  uint64_t k = 0;
  unsigned long long *dc = ctx->dcount ? ctx->d_dc : nullptr;
  if (ctx->prec == APT_PREC_FP64)
    HIPCHK(rt_pairs<double>(ctx->mesh, ctx->rt, view_of(ctx->p64), ctx->number,
                            view_of(ctx->ph64), ctx->ph_number, ctx->id_next,
                            ctx->rtw, ctx->d_counters, ctx->stream,
                            (double *)ctx->pair_produced, &k, dc));
  else
    HIPCHK(rt_pairs<float>(ctx->mesh, ctx->rt, view_of(ctx->p32), ctx->number,
                           view_of(ctx->ph32), ctx->ph_number, ctx->id_next,
                           ctx->rtw, ctx->d_counters, ctx->stream,
                           (float *)ctx->pair_produced, &k, dc));
  if (ctx->dcount) {
    // at most one pair per photon slot below the photon bound
    const uint64_t b = ctx->number + 2 * ctx->ph_number;
    ctx->number = b < ctx->cap ? b : ctx->cap;
    if (pairs) {
      unsigned long long h = 0;
      HIPCHK(hipMemcpyAsync(&h, ctx->d_dc + DC_LAST, 8, hipMemcpyDeviceToHost, ctx->stream));
      HIPCHK(hipStreamSynchronize(ctx->stream));
      *pairs = h;
    }
    return APT_OK;
  }
  if (k > 0) {
    // secondaries carry weights from the photons (<= any parent weight),
    // so the fixed-point scale stays valid
    ctx->number += 2 * k;
    ctx->id_next += 2 * k;
  }
  if (pairs) *pairs = k;
  return APT_OK;
}
apt_status apt_field_update_e(apt_ctx *ctx, double dt) {
  CHECK_CTX(ctx);
  return ctx->prec == APT_PREC_FP64 ? update_e_t<double>(ctx, dt)
                                    : update_e_t<float>(ctx, dt);
}
apt_status apt_field_update_b(apt_ctx *ctx, double dt) {
  CHECK_CTX(ctx);
  return ctx->prec == APT_PREC_FP64 ? update_b_t<double>(ctx, dt)
                                    : update_b_t<float>(ctx, dt);
}
apt_status apt_field_compute_divs(apt_ctx *ctx) {
  CHECK_CTX(ctx);
  return ctx->prec == APT_PREC_FP64 ? divs_t<double>(ctx)
                                    : divs_t<float>(ctx);
}

// ---- sort -------------------------------------------------------------
static apt_status ensure_second_buffer(apt_ctx *ctx) {
  if (ctx->have_b) return APT_OK;
  apt_status st = alloc_ptc(ctx, true);
  if (st != APT_OK) {
    free_ptc64(ctx->p64b);
    free_ptc32(ctx->p32b);
    st = give_back(ctx);
    if (st == APT_OK) st = alloc_ptc(ctx, true);
  }
  if (st != APT_OK) return st;
  ctx->have_b = true;
  return APT_OK;
}

static apt_status gather_all32(apt_ctx *ctx, uint64_t n) {
  PtcF32 &a = ctx->p32, &b = ctx->p32b;
  GatherSet g;
  g.add(a.cell, b.cell);
  g.add(a.x1, b.x1);
  g.add(a.x2, b.x2);
  g.add(a.x3, b.x3);
  g.add(a.u1, b.u1);
  g.add(a.u2, b.u2);
  g.add(a.u3, b.u3);
  g.add(a.w, b.w);
  g.add(a.flag, b.flag);
  HIPCHK(gather_set(ctx->sortw, g, n, ctx->stream));
  std::swap(ctx->p32, ctx->p32b);
  return APT_OK;
}

// 3D tiled mixed form between sorts: each tile's particles laid out cell by
// cell again (the slots appended since the sort are copied over as they
// are).  A recorded step holds the buffers of the old layout, so it is
// dropped.
static apt_status relayout_tiles(apt_ctx *ctx) {
  const TileInfo &ti = ctx->tiles;
  const uint64_t n = ctx->number, te = ti.tiled_end;
  time_begin(ctx, APT_KERNEL_SORT);
  HIPCHK(tile_sort_by_cell(ctx->mesh, ti, ctx->tile_off, ctx->p32, ctx->p32b, ctx->stream));
  if (n > te) {
    const PtcF32 &a = ctx->p32, &b = ctx->p32b;
    void *dst[9] = {b.cell + te, b.x1 + te, b.x2 + te, b.x3 + te, b.u1 + te,
                    b.u2 + te, b.u3 + te, b.w + te, b.flag + te};
    const void *src[9] = {a.cell + te, a.x1 + te, a.x2 + te, a.x3 + te, a.u1 + te,
                          a.u2 + te, a.u3 + te, a.w + te, a.flag + te};
    for (int k = 0; k < 9; k++)
      HIPCHK(hipMemcpyAsync(dst[k], src[k], (n - te) * 4, hipMemcpyDeviceToDevice,
                            ctx->stream));
  }
  std::swap(ctx->p32, ctx->p32b);
  time_end(ctx, APT_KERNEL_SORT);
  if (ctx->gexec) {
    (void)hipGraphExecDestroy(ctx->gexec);
    ctx->gexec = nullptr;
  }
  return APT_OK;
}

// Mixed form with tiling: the deterministic tile-binning sort; when a
// particle moved further than one tile (or slots were appended past the
// tiled range) a stable radix sort by tile key instead.  Both leave the
// particles binned by tile with the tile offsets on the device.
static apt_status sort_tiles(apt_ctx *ctx) {
  const uint64_t n = ctx->number;
  TileInfo &ti = ctx->tiles;
  time_begin(ctx, APT_KERNEL_SORT);
  unsigned long long far = 1;
  if (ctx->tiles_valid) {
    HIPCHK(tile_sort_count(ctx->mesh, ti, ctx->p32.cell, n, ctx->tsort,
                           ctx->stream));
    HIPCHK(hipMemcpyAsync(&far, ctx->tsort.far, 8, hipMemcpyDeviceToHost,
                          ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
  }
  if (far == 0) {
    HIPCHK(tile_sort_offsets(ctx->mesh, ti, ctx->tsort, ctx->stream));
    HIPCHK(tile_sort_scatter(ctx->mesh, ti, ctx->p32, ctx->p32b, n,
                             ctx->tsort, ctx->stream));
    if (ctx->mesh.dim == 3 && tile_cellsort_supported(ti)) {
      // 3D: each tile's particles cell by cell, back into the first buffer
      // (the 3D push reads its field taps through L1, which a wave whose
      // lanes share cells serves from the same lines)
      HIPCHK(tile_sort_by_cell(ctx->mesh, ti, ctx->tsort.newoff, ctx->p32b, ctx->p32,
                               ctx->stream));
    } else {
      std::swap(ctx->p32, ctx->p32b);
    }
    HIPCHK(hipMemcpyAsync(ctx->tile_off, ctx->tsort.newoff,
                          (ti.ntiles + 1) * 4ull, hipMemcpyDeviceToDevice,
                          ctx->stream));
  } else {
    HIPCHK(ctx->sortw.ensure(n));
    HIPCHK(tile_keys(ctx->mesh, ti, ctx->p32.cell, n, ctx->sortw.keys_in,
                     ctx->sortw.perm_in, ctx->stream));
    HIPCHK(hipcub_sort_pairs(ctx->sortw, n, key_bits(ti.ntiles), ctx->stream));
    apt_status st = gather_all32(ctx, n);
    if (st != APT_OK) return st;
    HIPCHK(tile_offsets_from_sorted(ctx->sortw.keys_out, n, ti.ntiles,
                                    ctx->tile_off, ctx->stream));
  }
  time_end(ctx, APT_KERNEL_SORT);
  uint32_t kept = 0;
  HIPCHK(hipMemcpyAsync(&kept, ctx->tile_off + ti.ntiles, 4,
                        hipMemcpyDeviceToHost, ctx->stream));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  if (kept < n)
    HIPCHK(launch_fill<uint32_t>(ctx->p32.cell + kept, MAX_CELL, n - kept,
                                 ctx->stream));
  ctx->number = kept;
  ti.tiled_end = kept;
  ctx->tiles_valid = true;
  ctx->pushes_since_sort = 0;
  ctx->drift = 0.0;
  return APT_OK;
}

// photons.sort_by_cell (sim_data_impl.hpp:80): stable sort by cell,
// empty slots dropped
static apt_status sort_photons(apt_ctx *ctx) {
  const uint64_t n = ctx->ph_number;
  if (n == 0) return APT_OK;
  if (ctx->capturing) return ctx->fail(APT_ERR_STATE, "sort: not while a step is recorded");
  if (!ctx->ph_have_b) {
    apt_status st = alloc_photons(ctx, true);
    if (st != APT_OK) {
      free_ph64(ctx->ph64b);
      free_ph32(ctx->ph32b);
      st = give_back(ctx);
      if (st == APT_OK) st = alloc_photons(ctx, true);
    }
    if (st != APT_OK) return st;
    ctx->ph_have_b = true;
  }
  const uint32_t empty_key = (uint32_t)ctx->ncell;
  SortWork &w = ctx->sortw;
  if (ctx->prec == APT_PREC_FP64) {
    PhoF64 &a = ctx->ph64, &b = ctx->ph64b;
    HIPCHK(sort_keys(w, a.cell, n, empty_key, nullptr, ctx->stream));
    GatherSet g;
    g.add(a.cell, b.cell);
    g.add(a.flag, b.flag);
    double *sa[] = {a.x1, a.x2, a.x3, a.p1, a.p2, a.p3, a.E, a.w, a.path};
    double *sb[] = {b.x1, b.x2, b.x3, b.p1, b.p2, b.p3, b.E, b.w, b.path};
    for (int k = 0; k < 9; k++) g.add(sa[k], sb[k]);
    g.add(a.id, b.id);
    HIPCHK(gather_set(w, g, n, ctx->stream));
    std::swap(ctx->ph64, ctx->ph64b);
  } else {
    PhoF32 &a = ctx->ph32, &b = ctx->ph32b;
    HIPCHK(sort_keys(w, a.cell, n, empty_key, nullptr, ctx->stream));
    GatherSet g;
    g.add(a.cell, b.cell);
    g.add(a.flag, b.flag);
    float *sa[] = {a.x1, a.x2, a.x3, a.p1, a.p2, a.p3, a.w, a.path};
    float *sb[] = {b.x1, b.x2, b.x3, b.p1, b.p2, b.p3, b.w, b.path};
    for (int k = 0; k < 8; k++) g.add(sa[k], sb[k]);
    HIPCHK(gather_set(w, g, n, ctx->stream));
    std::swap(ctx->ph32, ctx->ph32b);
  }
  if (ctx->dcount) {
    // the kept count stays on the device: slots from it up to the bound,
    // and past the bound (old data of this buffer), become empty
    uint32_t *cell = ph_cells(ctx);
    HIPCHK(launch_fill_tail(cell, w.count, n, ctx->stream));
    if (ctx->ph_cap > n)
      HIPCHK(launch_fill<uint32_t>(cell + n, MAX_CELL, ctx->ph_cap - n, ctx->stream));
    HIPCHK(launch_dc_set(ctx->d_dc, DC_PH, w.count, ctx->stream));
    return APT_OK;
  }
  unsigned long long kept = 0;
  HIPCHK(hipMemcpyAsync(&kept, w.count, 8, hipMemcpyDeviceToHost, ctx->stream));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  uint32_t *cell = ctx->prec == APT_PREC_FP64 ? ctx->ph64.cell : ctx->ph32.cell;
  if (kept < n)
    HIPCHK(launch_fill<uint32_t>(cell + kept, MAX_CELL, n - kept, ctx->stream));
  ctx->ph_number = kept;
  return APT_OK;
}

static apt_status sort_particles_only(apt_ctx *ctx);

apt_status apt_sort_particles(apt_ctx *ctx) {
  CHECK_CTX(ctx);
  // device-count mode: the sort runs over the exact counts (read back
  // once per sort), not over bounds that may have grown to the capacity
  apt_status st = exact_counts(ctx);
  if (st != APT_OK) return st;
  st = sort_particles_only(ctx);
  if (st != APT_OK) return st;
  return sort_photons(ctx);
}

// The run table, at the first sort; false where it does not fit: the updates then
// take consecutive slots.
static bool make_run_table(apt_ctx *ctx) {
  int T[3];
  if (ctx->prec == APT_PREC_FP64)
    f64_runs_tile(ctx->mesh.dim, T);
  else
    mixed_runs_tile(ctx->mesh.dim, T);
  // a log-spherical tile is shared later: its particles cluster, and each share
  // flushes a window (a cloud on half of the tiles: 78 us a push with 512, 70 with
  // 2048; FP64 152, 140)
  cell_runs_shape(ctx->mesh, T, ctx->logsph ? 2048 : 512, ctx->runs);
  const uint64_t entries = cell_runs_size(ctx->mesh, ctx->runs);
  if (hipMalloc(&ctx->run_off, (entries + 2 + 2 * (uint64_t)ctx->runs.items) * 4) != hipSuccess) {
    (void)hipGetLastError();
    ctx->run_off = nullptr;
    return false;
  }
  ctx->runs.off = ctx->run_off;
  ctx->runs.work = ctx->run_off + entries;
  return true;
}

static apt_status sort_particles_only(apt_ctx *ctx) {
  uint64_t n = ctx->number;
  if (n == 0) return APT_OK;
  if (ctx->capturing) return ctx->fail(APT_ERR_STATE, "sort: not while a step is recorded");
  apt_status st = ensure_second_buffer(ctx);
  if (st != APT_OK) return st;
  const uint32_t empty_key = (uint32_t)ctx->ncell;
  if (ctx->prec == APT_PREC_MIXED && ctx->tiling) return sort_tiles(ctx);
  // the updates that walk runs of sorted slots (the log-spherical one is 2D)
  bool by_runs = no_idle_guards(ctx->mesh) &&
                 (ctx->logsph ? ctx->mesh.dim == 2 : !ctx->gr1d && !ctx->gap1d);
  if (by_runs && !ctx->run_off) by_runs = make_run_table(ctx);
  time_begin(ctx, APT_KERNEL_SORT);
  if (ctx->prec == APT_PREC_FP64) {
    PtcF64 &a = ctx->p64, &b = ctx->p64b;
    HIPCHK(sort_keys(ctx->sortw, a.cell, n, empty_key, nullptr, ctx->stream));
    GatherSet g;
    g.add(a.cell, b.cell);
    g.add(a.flag, b.flag);
    double *sa[] = {a.x1, a.x2, a.x3, a.p1, a.p2, a.p3, a.E, a.w};
    double *sb[] = {b.x1, b.x2, b.x3, b.p1, b.p2, b.p3, b.E, b.w};
    for (int k = 0; k < 8; k++) g.add(sa[k], sb[k]);
    g.add(a.id, b.id);
    HIPCHK(gather_set(ctx->sortw, g, n, ctx->stream));
    std::swap(ctx->p64, ctx->p64b);
  } else {
    HIPCHK(sort_keys(ctx->sortw, ctx->p32.cell, n, empty_key, nullptr, ctx->stream));
    st = gather_all32(ctx, n);
    if (st != APT_OK) return st;
  }
  ctx->runs_valid = false;
  if (by_runs) {
    HIPCHK(build_cell_runs(ctx->mesh, ctx->runs, ctx->sortw.keys_out, n, ctx->run_off,
                           ctx->stream));
  }
  time_end(ctx, APT_KERNEL_SORT);
  if (ctx->dcount) {
    // the kept count stays on the device: slots from it up to the bound,
    // and past the bound (old data of this buffer), become empty
    uint32_t *cell = ptc_cells(ctx);
    HIPCHK(launch_fill_tail(cell, ctx->sortw.count, n, ctx->stream));
    if (ctx->cap > n)
      HIPCHK(launch_fill<uint32_t>(cell + n, MAX_CELL, ctx->cap - n, ctx->stream));
    HIPCHK(launch_dc_set(ctx->d_dc, DC_NUM, ctx->sortw.count, ctx->stream));
    if (by_runs) {  // the table holds the kept count, the host its bound
      ctx->runs.end = n;
      ctx->runs_valid = true;
    }
    return APT_OK;
  }
  uint64_t kept = 0;
  bool pay = true;
  if (by_runs) {  // the table's last entry, then the items and the slots in tiles
    uint32_t h[3];
    HIPCHK(hipMemcpyAsync(h, ctx->runs.work - 1, sizeof(h), hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    kept = h[0];
    ctx->runs.guard_slots = kept - h[2];
    if (!ctx->logsph)
      pay = ctx->prec == APT_PREC_FP64 ? f64_runs_pay(ctx->mesh.dim, kept, h[1])
                                       : mixed_runs_pay(ctx->mesh.dim, kept, h[1]);
  } else {
    HIPCHK(hipMemcpyAsync(&kept, ctx->sortw.count, 8, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
  }
  // the slots freed by the compaction become empty
  if (kept < n) {
    uint32_t *cell = ctx->prec == APT_PREC_FP64 ? ctx->p64.cell : ctx->p32.cell;
    HIPCHK(launch_fill<uint32_t>(cell + kept, MAX_CELL, n - kept, ctx->stream));
  }
  ctx->number = kept;
  if (by_runs && pay) {
    ctx->runs.end = kept;
    ctx->runs_valid = true;
  }
  return APT_OK;
}

template <typename R, typename P, typename H>
static apt_status diagnostics_t(apt_ctx *ctx, const P &p, const H &ph) {
  DiagArrays<R> d;
  for (int s = 0; s < 4; s++) {
    d.num[s] = (R *)ctx->diag_num[s];
    d.gamma[s] = (R *)ctx->diag_gamma[s];
  }
  d.photon_num = (R *)ctx->diag_ph;
  HIPCHK(launch_diagnostics<R>(view_of(p), ctx->number, view_of(ph),
                               ctx->ph_cap ? ctx->ph_number : 0, d,
                               ctx->params.num_species, ctx->ncell, ctx->stream));
  return APT_OK;
}

apt_status apt_collect_diagnostics(apt_ctx *ctx) {
  CHECK_CTX(ctx);
  {
    apt_status st = exact_counts(ctx);
    if (st != APT_OK) return st;
  }
  const size_t bytes = ctx->ncell * (ctx->prec == APT_PREC_FP64 ? 8 : 4);
  if (!ctx->diag_ph) {
    HIPCHK(hipMalloc(&ctx->diag_ph, bytes));
    for (int s = 0; s < 4; s++) {
      HIPCHK(hipMalloc(&ctx->diag_num[s], bytes));
      HIPCHK(hipMalloc(&ctx->diag_gamma[s], bytes));
    }
  }
  if (ctx->prec == APT_PREC_FP64) return diagnostics_t<double>(ctx, ctx->p64, ctx->ph64);
  return diagnostics_t<float>(ctx, ctx->p32, ctx->ph32);
}

apt_status apt_clear_guard_cells(apt_ctx *ctx) {
  CHECK_CTX(ctx);
  uint32_t *cell = ctx->prec == APT_PREC_FP64 ? ctx->p64.cell : ctx->p32.cell;
  HIPCHK(launch_erase_guard(ctx->mesh, cell, ctx->number, ctx->stream));
  return APT_OK;
}

apt_status apt_energy_histogram(apt_ctx *ctx, uint32_t *hist, int nbins,
                                double E_max, int flag_bit) {
  CHECK_CTX(ctx);
  {
    apt_status st = exact_counts(ctx);
    if (st != APT_OK) return st;
  }
  if (!hist || nbins < 1 || nbins > 8192 || !(E_max > 1.0))
    return ctx->fail(APT_ERR_INVALID_ARG, "energy_histogram: bad arguments");
  uint32_t *d = nullptr;
  HIPCHK(hipMalloc(&d, nbins * 4));
  hipError_t e = hipMemsetAsync(d, 0, nbins * 4, ctx->stream);
  if (e == hipSuccess)
    e = ctx->prec == APT_PREC_FP64
            ? launch_energy_histogram_f64(ctx->p64.E, ctx->p64.flag,
                                          ctx->number, d, nbins, E_max,
                                          flag_bit, ctx->stream)
            : launch_energy_histogram_mixed(ctx->p32.u1, ctx->p32.u2,
                                            ctx->p32.u3, ctx->p32.flag,
                                            ctx->number, d, nbins, E_max,
                                            flag_bit, ctx->stream);
  if (e == hipSuccess)
    e = hipMemcpyAsync(hist, d, nbins * 4, hipMemcpyDeviceToHost,
                       ctx->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
  (void)hipFree(d);
  HIPCHK(e);
  return APT_OK;
}

apt_status apt_energy_histogram_noalloc(apt_ctx *ctx, uint32_t *hist, int nbins,
                                        double E_max, int flag_bit) {
  CHECK_CTX(ctx);
  {
    apt_status st = exact_counts(ctx);
    if (st != APT_OK) return st;
  }
  if (!hist || nbins < 1 || !(E_max > 1.0))
    return ctx->fail(APT_ERR_INVALID_ARG, "energy_histogram_noalloc: bad arguments");
  if (nbins > APT_NOALLOC_HIST_MAX_BINS)
    return ctx->fail(APT_ERR_INVALID_ARG,
                     "energy_histogram_noalloc: %d bins > the maximum of %d", nbins,
                     APT_NOALLOC_HIST_MAX_BINS);
  uint32_t *d = scratch_of(ctx->device);
  if (!d)
    return ctx->fail(APT_ERR_HIP, "energy_histogram_noalloc: no scratch on device %d",
                     ctx->device);
  // the array keeps the last call's counts: cleared by a fill kernel
  HIPCHK(launch_fill<uint32_t>(d, 0u, (uint64_t)nbins, ctx->stream));
  HIPCHK(ctx->prec == APT_PREC_FP64
             ? launch_energy_histogram_f64(ctx->p64.E, ctx->p64.flag, ctx->number, d, nbins,
                                           E_max, flag_bit, ctx->stream)
             : launch_energy_histogram_mixed(ctx->p32.u1, ctx->p32.u2, ctx->p32.u3,
                                             ctx->p32.flag, ctx->number, d, nbins, E_max,
                                             flag_bit, ctx->stream));
  HIPCHK(hipMemcpyAsync(hist, d, (size_t)nbins * 4, hipMemcpyDeviceToHost, ctx->stream));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  return APT_OK;
}

// ---- field_solver_ffe (3D Cartesian) ----------------------------------

static bool ffe_cart_ok(apt_ctx *ctx, const char *what) {
  if (ctx->logsph || ctx->gr1d || ctx->gap1d || ctx->mesh.dim != 3) {
    ctx->fail(APT_ERR_UNSUPPORTED, "%s: a 3D Cartesian context only", what);
    return false;
  }
  return true;
}

static bool is_vec_field(int w) {
  return w == APT_FIELD_E || w == APT_FIELD_B || w == APT_FIELD_EBG || w == APT_FIELD_BBG ||
         w == APT_FIELD_J || w == APT_FIELD_FFE_E || w == APT_FIELD_FFE_B;
}
static bool is_scalar_field(apt_ctx *ctx, int w, int comp) {
  if (w == APT_FIELD_RHO) return comp >= 0 && comp < ctx->params.num_species;
  return comp == 0 && (w == APT_FIELD_DIVE || w == APT_FIELD_DIVB || w == APT_FIELD_EDOTB ||
                       w == APT_FIELD_FFE_F);
}

template <typename T>
static apt_status ffe_cart_substep_t(apt_ctx *ctx, int eo, int bo, int jo, int ei, int bi,
                                     double dt) {
  T *vEo[3], *vBo[3], *vJo[3];
  const T *vEi[3], *vBi[3];
  for (int c = 0; c < 3; c++) {
    vEo[c] = (T *)*field_slot(ctx, eo, c);
    vBo[c] = (T *)*field_slot(ctx, bo, c);
    vJo[c] = (T *)*field_slot(ctx, jo, c);
    vEi[c] = (const T *)*field_slot(ctx, ei, c);
    vBi[c] = (const T *)*field_slot(ctx, bi, c);
  }
  if (eo == ei) {  // read E_in from a copy: the update reads the neighbours it writes
    HIPCHK(ensure_ffe_cart(ctx, 10));
    for (int c = 0; c < 3; c++) {
      HIPCHK(hipMemcpyAsync(ctx->ffc[7 + c], vEi[c], ctx->ncell * sizeof(T),
                            hipMemcpyDeviceToDevice, ctx->stream));
      vEi[c] = (const T *)ctx->ffc[7 + c];
    }
  }
  time_begin(ctx, APT_KERNEL_FIELD);
  HIPCHK(launch_ffe_cart_curl_add<T>(ctx->mesh, vBo, vEi, (T)dt, ctx->stream));
  HIPCHK(launch_ffe_cart_de<T>(ctx->mesh, vEo, vJo, vEi, vBi, (T)dt, ctx->stream));
  time_end(ctx, APT_KERNEL_FIELD);
  return APT_OK;
}

apt_status apt_ffe_cart_substep(apt_ctx *ctx, int e_out, int b_out, int j_out, int e_in,
                                int b_in, double dt) {
  CHECK_CTX(ctx);
  if (!ffe_cart_ok(ctx, "ffe_cart_substep")) return APT_ERR_UNSUPPORTED;
  const int ids[5] = {e_out, b_out, j_out, e_in, b_in};
  for (int w : ids)
    if (!is_vec_field(w))
      return ctx->fail(APT_ERR_INVALID_ARG, "ffe_cart_substep: %d is not a vector field", w);
  // B_out and E_in, and J_out and every other argument, must differ: each
  // kernel reads the neighbours of the cells it writes.  B_in may be B_out
  // (read after its update) and E_out may be E_in (read from a copy).
  if (b_out == e_in || e_out == b_in || e_out == b_out || j_out == e_out ||
      j_out == b_out || j_out == e_in || j_out == b_in)
    return ctx->fail(APT_ERR_INVALID_ARG, "ffe_cart_substep: overlapping fields");
  for (int w : {e_out, b_out, j_out}) field_written(ctx, w);
  HIPCHK(ensure_ffe_cart(ctx));
  return ctx->prec == APT_PREC_FP64
             ? ffe_cart_substep_t<double>(ctx, e_out, b_out, j_out, e_in, b_in, dt)
             : ffe_cart_substep_t<float>(ctx, e_out, b_out, j_out, e_in, b_in, dt);
}

template <typename T>
static void vec_of(apt_ctx *ctx, int w, const T *v[3]) {
  for (int c = 0; c < 3; c++) v[c] = (const T *)*field_slot(ctx, w, c);
}

apt_status apt_ffe_cart_edotb(apt_ctx *ctx, int out, int out_comp, int e, int b, double q) {
  CHECK_CTX(ctx);
  if (!ffe_cart_ok(ctx, "ffe_cart_edotb")) return APT_ERR_UNSUPPORTED;
  if (!is_scalar_field(ctx, out, out_comp) || !is_vec_field(e) || !is_vec_field(b))
    return ctx->fail(APT_ERR_INVALID_ARG, "ffe_cart_edotb: bad fields");
  field_written(ctx, out);
  HIPCHK(ensure_ffe_cart(ctx));
  if (ctx->prec == APT_PREC_FP64) {
    const double *ve[3], *vb[3];
    vec_of(ctx, e, ve);
    vec_of(ctx, b, vb);
    HIPCHK(launch_ffe_cart_edotb<double>(ctx->mesh, (double *)*field_slot(ctx, out, out_comp),
                                         ve, vb, q, ctx->stream));
  } else {
    const float *ve[3], *vb[3];
    vec_of(ctx, e, ve);
    vec_of(ctx, b, vb);
    HIPCHK(launch_ffe_cart_edotb<float>(ctx->mesh, (float *)*field_slot(ctx, out, out_comp),
                                        ve, vb, (float)q, ctx->stream));
  }
  return APT_OK;
}

apt_status apt_ffe_cart_j(apt_ctx *ctx, int j_out, int f, int f_comp, int e, int b,
                          double q) {
  CHECK_CTX(ctx);
  if (!ffe_cart_ok(ctx, "ffe_cart_j")) return APT_ERR_UNSUPPORTED;
  if (!is_vec_field(j_out) || !is_scalar_field(ctx, f, f_comp) || !is_vec_field(e) ||
      !is_vec_field(b) || j_out == e || j_out == b)
    return ctx->fail(APT_ERR_INVALID_ARG, "ffe_cart_j: bad fields");
  field_written(ctx, j_out);
  HIPCHK(ensure_ffe_cart(ctx));
  if (ctx->prec == APT_PREC_FP64) {
    const double *ve[3], *vb[3];
    double *vj[3];
    vec_of(ctx, e, ve);
    vec_of(ctx, b, vb);
    for (int c = 0; c < 3; c++) vj[c] = (double *)*field_slot(ctx, j_out, c);
    HIPCHK(launch_ffe_cart_j<double>(ctx->mesh, vj, (const double *)*field_slot(ctx, f, f_comp),
                                     ve, vb, q, ctx->stream));
  } else {
    const float *ve[3], *vb[3];
    float *vj[3];
    vec_of(ctx, e, ve);
    vec_of(ctx, b, vb);
    for (int c = 0; c < 3; c++) vj[c] = (float *)*field_slot(ctx, j_out, c);
    HIPCHK(launch_ffe_cart_j<float>(ctx->mesh, vj, (const float *)*field_slot(ctx, f, f_comp),
                                    ve, vb, (float)q, ctx->stream));
  }
  return APT_OK;
}

// The Gauss-law check: max over the bulk of |div E - kappa sum_s Rho_s| and
// of |div E|, reduced in FP64 on the device; the residual field on request.
apt_status apt_div_residual(apt_ctx *ctx, double kappa, double *max_abs, double *scale,
                            double *residual, uint64_t count) {
  CHECK_CTX(ctx);
  if (!max_abs || !scale)
    return ctx->fail(APT_ERR_INVALID_ARG, "div_residual: null output");
  if (residual && count != ctx->ncell)
    return ctx->fail(APT_ERR_INVALID_ARG, "div_residual: residual needs %llu values",
                     (unsigned long long)ctx->ncell);
  if (residual && !ctx->divres_field) {
    HIPCHK(hipMalloc(&ctx->divres_field, ctx->ncell * 8));
  }
  double *out = residual ? ctx->divres_field : nullptr;
  if (out) HIPCHK(launch_fill<double>(out, 0.0, ctx->ncell, ctx->stream));
  const int ns = ctx->params.num_species < 4 ? ctx->params.num_species : 4;
  int nb = 0;
  if (ctx->prec == APT_PREC_FP64) {
    RhoSet<double> r{{(const double *)ctx->Rho[0], (const double *)ctx->Rho[1],
                      (const double *)ctx->Rho[2], (const double *)ctx->Rho[3]}};
    HIPCHK(launch_div_residual<double>(ctx->mesh, (const double *)ctx->divE, r, ns, kappa,
                                       out, ctx->divres_part, DIVRES_MAX_BLOCKS, &nb,
                                       ctx->stream));
  } else {
    RhoSet<float> r{{(const float *)ctx->Rho[0], (const float *)ctx->Rho[1],
                     (const float *)ctx->Rho[2], (const float *)ctx->Rho[3]}};
    HIPCHK(launch_div_residual<float>(ctx->mesh, (const float *)ctx->divE, r, ns, kappa, out,
                                      ctx->divres_part, DIVRES_MAX_BLOCKS, &nb, ctx->stream));
  }
  std::vector<double> part(2 * (size_t)nb);
  HIPCHK(hipMemcpyAsync(part.data(), ctx->divres_part, part.size() * 8,
                        hipMemcpyDeviceToHost, ctx->stream));
  if (out)
    HIPCHK(hipMemcpyAsync(residual, out, ctx->ncell * 8, hipMemcpyDeviceToHost, ctx->stream));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  double mr = 0.0, md = 0.0;
  for (int b = 0; b < nb; b++) {
    mr = fmax(mr, part[2 * b]);
    md = fmax(md, part[2 * b + 1]);
  }
  *max_abs = mr;
  *scale = md;
  return APT_OK;
}

apt_status apt_tile_offsets(apt_ctx *ctx, uint32_t *off, uint64_t cap,
                            uint32_t *ntiles, int tile_extent[3]) {
  CHECK_CTX(ctx);
  if (!ntiles) return APT_ERR_INVALID_ARG;
  *ntiles = 0;
  if (tile_extent)
    for (int d = 0; d < 3; d++) tile_extent[d] = ctx->tiles.T[d];
  if (!ctx->tiling || !ctx->tiles_valid) return APT_OK;
  *ntiles = ctx->tiles.ntiles;
  if (!off) return APT_OK;
  if (cap < (uint64_t)ctx->tiles.ntiles + 1)
    return ctx->fail(APT_ERR_CAPACITY, "tile_offsets: need %u entries",
                     ctx->tiles.ntiles + 1);
  HIPCHK(hipMemcpyAsync(off, ctx->tile_off, (ctx->tiles.ntiles + 1) * 4ull,
                        hipMemcpyDeviceToHost, ctx->stream));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  return APT_OK;
}

apt_status apt_stream_probe(apt_ctx *ctx, uint64_t n, int reps, double *ms) {
  CHECK_CTX(ctx);
  if (!ms || reps < 1 || ctx->prec != APT_PREC_MIXED || n > ctx->cap)
    return ctx->fail(APT_ERR_INVALID_ARG, "stream_probe: mixed form, n <= cap");
  hipEvent_t a, b;
  HIPCHK(hipEventCreate(&a));
  HIPCHK(hipEventCreate(&b));
  HIPCHK(launch_stream_probe(ctx->p32, n, ctx->stream));  // warm-up
  HIPCHK(hipEventRecord(a, ctx->stream));
  for (int r = 0; r < reps; r++)
    HIPCHK(launch_stream_probe(ctx->p32, n, ctx->stream));
  HIPCHK(hipEventRecord(b, ctx->stream));
  HIPCHK(hipEventSynchronize(b));
  float t = 0.0f;
  HIPCHK(hipEventElapsedTime(&t, a, b));
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  *ms = t / reps;
  return APT_OK;
}

// ---- device-resident counts and the recorded step ---------------------
apt_status apt_set_device_counts(apt_ctx *ctx, int on) {
  CHECK_CTX(ctx);
  if (ctx->capturing) return ctx->fail(APT_ERR_STATE, "set_device_counts: a step is recorded");
  if (!on) {
    apt_status st = exact_counts(ctx);
    if (st != APT_OK) return st;
    if (ctx->dcount) ctx->runs_valid = false;  // runs.end may be a bound
    ctx->dcount = false;
    return APT_OK;
  }
  if (!ctx->logsph || ctx->mesh.dim != 2)
    return ctx->fail(APT_ERR_UNSUPPORTED, "set_device_counts: 2D log-spherical contexts only");
  if (ctx->dcount) return APT_OK;
  if (!ctx->d_dc) HIPCHK(hipMalloc(&ctx->d_dc, DC_N * sizeof(unsigned long long)));
  // every slot past a count is empty from here on
  if (ctx->cap > ctx->number)
    HIPCHK(launch_fill<uint32_t>(ptc_cells(ctx) + ctx->number, MAX_CELL,
                                 ctx->cap - ctx->number, ctx->stream));
  if (ctx->ph_cap > ctx->ph_number)
    HIPCHK(launch_fill<uint32_t>(ph_cells(ctx) + ctx->ph_number, MAX_CELL,
                                 ctx->ph_cap - ctx->ph_number, ctx->stream));
  unsigned long long h[DC_N] = {};
  h[DC_NUM] = ctx->number;
  h[DC_PH] = ctx->ph_number;
  h[DC_ID] = ctx->id_next;
  h[DC_PH_ID] = ctx->ph_id_next;
  h[DC_RT_EPOCH] = ctx->rt_epoch;
  h[DC_INJ_EPOCH] = ctx->inject_epoch;
  HIPCHK(hipMemcpyAsync(ctx->d_dc, h, sizeof(h), hipMemcpyHostToDevice, ctx->stream));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  ctx->dcount = true;
  return APT_OK;
}

apt_status apt_get_events(apt_ctx *ctx, uint64_t *emitted, uint64_t *converted,
                          uint64_t *pushed) {
  CHECK_CTX(ctx);
  if (!emitted || !converted) return APT_ERR_INVALID_ARG;
  if (!ctx->dcount) return ctx->fail(APT_ERR_STATE, "get_events: device counts are off");
  if (ctx->capturing) return ctx->fail(APT_ERR_STATE, "get_events: a step is recorded");
  unsigned long long h[DC_N];
  HIPCHK(hipMemcpyAsync(h, ctx->d_dc, sizeof(h), hipMemcpyDeviceToHost, ctx->stream));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  *emitted = h[DC_EMITTED];
  *converted = h[DC_CONVERTED];
  if (pushed) *pushed = h[DC_PUSHED];
  return APT_OK;
}

apt_status apt_graph_begin(apt_ctx *ctx) {
  CHECK_CTX(ctx);
  if (ctx->capturing) return ctx->fail(APT_ERR_STATE, "graph_begin: already recording");
  if (ctx->dcount) {
    // the recorded launches cover every slot (kernels stop at the device
    // counts), so a replay stays valid however the counts grow; scan
    // scratch sized for it
    HIPCHK(ctx->rtw.ensure(ctx->cap > ctx->ph_cap ? ctx->cap : ctx->ph_cap));
    ctx->number = ctx->cap;
    ctx->ph_number = ctx->ph_cap;
  }
  // with host counts a recording holds calls that change no count (push,
  // fields, boundaries, filters): the launches keep the current counts
  HIPCHK(hipStreamSynchronize(ctx->stream));
  ctx->timing_saved = ctx->timing;
  ctx->timing = false;
  HIPCHK(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
  ctx->capturing = true;
  return APT_OK;
}

apt_status apt_graph_end(apt_ctx *ctx) {
  CHECK_CTX(ctx);
  if (!ctx->capturing) return ctx->fail(APT_ERR_STATE, "graph_end: not recording");
  ctx->capturing = false;
  ctx->timing = ctx->timing_saved;
  hipGraph_t g = nullptr;
  HIPCHK(hipStreamEndCapture(ctx->stream, &g));
  if (ctx->gexec) {
    (void)hipGraphExecDestroy(ctx->gexec);
    ctx->gexec = nullptr;
  }
  hipError_t e = hipGraphInstantiate(&ctx->gexec, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  HIPCHK(e);
  return APT_OK;
}

apt_status apt_graph_launch(apt_ctx *ctx, int times) {
  CHECK_CTX(ctx);
  if (!ctx->gexec) return ctx->fail(APT_ERR_STATE, "graph_launch: no recorded step");
  if (ctx->capturing) return ctx->fail(APT_ERR_STATE, "graph_launch: a step is recorded");
  ctx->rho_zero = false;  // a recorded deposit step writes Rho
  ctx->drift = 1e30;      // and moves the particles on
  for (int k = 0; k < times; k++) HIPCHK(hipGraphLaunch(ctx->gexec, ctx->stream));
  return APT_OK;
}

// ---- control ------------------------------------------------------------
apt_status apt_sync(apt_ctx *ctx) {
  CHECK_CTX(ctx);
  HIPCHK(hipStreamSynchronize(ctx->stream));
  return APT_OK;
}

apt_status apt_get_counters(apt_ctx *ctx, apt_counters *out) {
  CHECK_CTX(ctx);
  if (!out) return APT_ERR_INVALID_ARG;
  unsigned long long h[CTR_NUM];
  HIPCHK(hipMemcpyAsync(h, ctx->d_counters, sizeof(h), hipMemcpyDeviceToHost,
                        ctx->stream));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  out->nan_momenta = h[CTR_NAN];
  out->multi_cell_moves = h[CTR_MULTICELL];
  out->capacity_overflow = h[CTR_OVERFLOW];
  out->outside_tile = h[CTR_OUTSIDE];
  out->global_deposits = h[CTR_GLOBAL_DEP];
  return APT_OK;
}

apt_status apt_reset_counters(apt_ctx *ctx) {
  CHECK_CTX(ctx);
  HIPCHK(launch_fill<long long>((long long *)ctx->d_counters, 0, CTR_NUM,
                                ctx->stream));
  return APT_OK;
}

apt_status apt_timing_enable(apt_ctx *ctx, int on) {
  CHECK_CTX(ctx);
  HIPCHK(hipStreamSynchronize(ctx->stream));
  ctx->timing = on != 0;
  for (int k = 0; k < APT_KERNEL_NUM; k++) ctx->ev_used[k] = 0;
  return APT_OK;
}

apt_status apt_timing_get(apt_ctx *ctx, int kernel, double *total_ms,
                          uint64_t *launches) {
  CHECK_CTX(ctx);
  if (kernel < 0 || kernel >= APT_KERNEL_NUM)
    return ctx->fail(APT_ERR_INVALID_ARG, "timing_get: bad kernel id");
  HIPCHK(hipStreamSynchronize(ctx->stream));
  double tot = 0.0;
  for (size_t i = 0; i < ctx->ev_used[kernel]; i++) {
    float ms = 0.0f;
    HIPCHK(hipEventElapsedTime(&ms, ctx->ev[kernel][i].a,
                               ctx->ev[kernel][i].b));
    tot += ms;
  }
  if (total_ms) *total_ms = tot;
  if (launches) *launches = ctx->ev_used[kernel];
  return APT_OK;
}

