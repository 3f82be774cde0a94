// apt_kernels.hpp -- device pointer bundles and host launchers of every
// kernel in the library (the role data_ptrs plays in the reference,
// cuda/data_ptrs.h:11-29, but passed per launch and split by precision).
#pragma once
#include <vector>

#include "apt_common.hpp"

namespace apt {

enum CounterIdx {
  CTR_NAN = 0,        // NaN momentum seen by the push
  CTR_MULTICELL = 1,  // a particle moved more than one cell in a step
  CTR_OVERFLOW = 2,   // a particle could not be stored (capacity)
  CTR_OUTSIDE = 3,    // a particle left the deposit window of its tile
  CTR_GLOBAL_DEP = 4, // an FP64 particle whose chunk was too spread for an LDS window
  CTR_NUM = 8
};

// ---- plain FP64 form ------------------------------------------------
struct PtcF64 {
  uint32_t *cell;
  double *x1, *x2, *x3;
  double *p1, *p2, *p3;
  double *E;
  double *w;
  uint32_t *flag;
  uint64_t *id;
};

struct FieldsF64 {
  const double *E[3];
  const double *B[3];
};

struct AccF64 {
  long long *J[3][2];
  long long *R[4][2];
};

// One axis of the tiling: its N cells split evenly over nt tiles, the first r
// of w + 1 cells, the others of w (an even split instead of full tiles and a
// narrow last one: no tile is so thin that particles cross it whole between
// sorts, and every tile carries the same load).
struct TileAxis {
  int w, r;
  FastDiv dw, dw1;  // by w and by w + 1
  __host__ __device__ inline int origin(int t) const { return t * w + (t < r ? t : r); }
  __host__ __device__ inline int tile_of(int x) const {
    const int s = r * (w + 1);
    return x < s ? (int)dw1.div((uint32_t)x) : r + (int)dw.div((uint32_t)(x - s));
  }
};

inline TileAxis make_tile_axis(int N, int nt) {
  TileAxis a;
  a.w = N / nt;
  a.r = N - a.w * nt;
  a.dw = make_fastdiv((uint32_t)a.w);
  a.dw1 = make_fastdiv((uint32_t)a.w + 1u);
  return a;
}

// Runs of cell-ordered slots by tile (apt_runs.hpp).  off[row nt0 + tx] is the
// first slot of the cells of mesh row `row` (y fastest, guard rows included)
// from tile tx's first cell on; a row's guard cells in x belong to its first
// and last tile.  The last entry (rows nt0) is `end`.  work, right behind it:
// the number of work items, the slots in tiles (the others are in guard rows),
// then two words per item (tile, part | parts << 16): the tiles, those with many
// particles in several parts.
struct CellRuns {
  const uint32_t *off = nullptr, *work = nullptr;
  TileAxis ax[3];
  int nt[3];
  uint32_t ntiles;
  uint32_t items;  // most items there can be (a multiple of 8)
  uint32_t least;  // particles below which a tile is not shared
  uint64_t end;    // slots covered, known on the host
  uint64_t guard_slots;  // of these in guard rows (host counts)
};
// entries of the offsets; the table has 2 + 2 items more
inline uint64_t cell_runs_size(const Mesh &m, const CellRuns &cr) {
  return (uint64_t)m.dims[1] * m.dims[2] * cr.nt[0] + 1;
}
// tiles of at most T[d] cells
void cell_runs_shape(const Mesh &m, const int T[3], uint32_t least, CellRuns &cr);
// fills the table from n sorted keys (cell, or at least m.size() for empty
// slots)
hipError_t build_cell_runs(const Mesh &m, const CellRuns &cr, const uint32_t *keys, uint64_t n,
                           uint32_t *table, hipStream_t st);

// tile extents of the updates over cell runs, by dimension, and whether they are
// the faster ones: kept slots in `items` work items
void mixed_runs_tile(int dim, int T[3]);
bool mixed_runs_pay(int dim, uint64_t kept, uint32_t items);
void f64_runs_tile(int dim, int T[3]);
bool f64_runs_pay(int dim, uint64_t kept, uint32_t items);
// the update of the slots below cr.end, through LDS windows by tile
hipError_t launch_push_deposit_f64_runs(const Mesh &m, const Species &sp, double dt, int H,
                                        int rho, const PtcF64 &p, const FieldsF64 &f,
                                        const AccF64 &a, const CellRuns &cr,
                                        unsigned long long *counters, hipStream_t st);
hipError_t launch_push_deposit_f64(const Mesh &m, const Species &sp,
                                   double dt, int H, int rho, int nsp,
                                   const PtcF64 &p, const FieldsF64 &f,
                                   const AccF64 &a,
                                   unsigned long long *counters, uint64_t n,
                                   hipStream_t st);
hipError_t launch_finalize_f64(long long *hi, long long *lo, double *out,
                               uint64_t n, int H, hipStream_t st);

// ---- mixed form (FP32 push, int32 cell + FP32 offset, int64 J) -----
struct PtcF32 {
  uint32_t *cell;
  float *x1, *x2, *x3;
  float *u1, *u2, *u3;
  float *w;
  uint32_t *flag;
};

struct FieldsF32 {
  const float *E[3];
  const float *B[3];
};

// Tiling of the mixed deposit: particles sorted by tile; tile t owns
// particles [tile_off[t], tile_off[t+1]).  Particles past tile_off[ntiles]
// (appended since the last sort) go through the untiled path.
struct TileInfo {
  int T[3];       // largest tile extent in cells (the window is sized for it)
  int nt[3];      // tiles per dimension
  TileAxis ax[3];
  // every axis in tiles of one power-of-two extent: tile = cell >> sh (3D, 16.7 M
  // particles, us: count and scatter of a sort 83 + 475; 100 + 501 with a choice
  // between shift and division made axis by axis)
  bool shifts;
  uint32_t sh[3];
  int halo;       // cells of LDS halo around a tile
  int threads;    // threads per tile workgroup
  const uint32_t *tile_off;
  uint32_t ntiles;
  uint64_t tiled_end;  // tile_off[ntiles], known on the host
};

// int64 accumulators of the mixed form: J[c] always, R[s] when rho != 0
struct AccMixed {
  long long *J[3];
  long long *R[4];
  int rho;
};

// the update of the slots below cr.end, through LDS windows by tile
hipError_t launch_push_deposit_mixed_runs(const Mesh &m, const Species &sp, float dt, int S,
                                          const PtcF32 &p, const FieldsF32 &f, const AccMixed &a,
                                          const CellRuns &cr, unsigned long long *counters,
                                          hipStream_t st);
// first: the first slot (untiled meshes only)
hipError_t launch_push_deposit_mixed(const Mesh &m, const Species &sp,
                                     float dt, int S, const PtcF32 &p,
                                     const FieldsF32 &f, const AccMixed &a,
                                     const TileInfo &tiles,
                                     unsigned long long *counters,
                                     uint64_t n, hipStream_t st, uint64_t first = 0);

// ---- particle views shared by the forms -------------------------------
// E (stored gamma) and id exist in the FP64 form only; the mixed form
// recomputes gamma from u and carries no id.
template <typename R>
struct PtcView {
  uint32_t *cell;
  R *x1, *x2, *x3;
  R *p1, *p2, *p3;
  R *E;
  R *w;
  uint32_t *flag;
  uint64_t *id;
};
inline PtcView<double> view_of(const PtcF64 &p) {
  return {p.cell, p.x1, p.x2, p.x3, p.p1, p.p2, p.p3, p.E, p.w, p.flag, p.id};
}
inline PtcView<float> view_of(const PtcF32 &p) {
  return {p.cell, p.x1, p.x2, p.x3, p.u1, p.u2, p.u3, nullptr, p.w, p.flag,
          nullptr};
}

// ---- fields (T = double: FP64 form, T = float: mixed form) ----------
template <typename T>
struct FieldSet {
  T *E[3], *B[3];
  const T *Ebg[3], *Bbg[3];
  const T *J[3];
  T *divE, *divB;
  T *EdotB = nullptr;  // time-averaged E.B/|B| at cell centres (log-spherical)
  // Cartesian: a background that was never set (all zeros) is not read
  bool has_ebg = true, has_bbg = true;
};

// Accumulators to finalize in one launch (J and, on deposit steps, Rho) and
// arrays to clear.  lo is read in the FP64 form only.
template <typename T>
struct FinalizeSet {
  long long *hi[7], *lo[7];
  T *out[7];
  int n = 0;
  T *zero[4];
  int nzero = 0;
};
template <typename T>
hipError_t launch_finalize_set(const FinalizeSet<T> &fs, uint64_t n, int H, hipStream_t st);
// whether updates and filters can write guard images themselves: every axis
// with guard cells periodic and no shorter than its guard
bool guard_images_ok(const Mesh &m);
// one binomial pass of n (at most 4) components, src to dst with guard images;
// guard_images_ok meshes only
template <typename T>
hipError_t launch_filter_set(const Mesh &m, T *const *src, T *const *dst, int n, int fix3d,
                             hipStream_t st);

// the updates leave the guard cells of periodic axes refreshed
template <typename T>
hipError_t launch_update_e(const Mesh &m, const FieldSet<T> &f, double dt,
                           hipStream_t st);
template <typename T>
// ref3d: the reference's 3D stencil (forward differences), else staggered
hipError_t launch_update_b(const Mesh &m, const FieldSet<T> &f, double dt,
                           hipStream_t st, int ref3d = 0);
template <typename T>
hipError_t launch_divs(const Mesh &m, const FieldSet<T> &f, hipStream_t st);
template <typename T>
hipError_t launch_guard_copy(const Mesh &m, T *a, hipStream_t st);
template <typename T>
hipError_t launch_filter(const Mesh &m, T *j, T *tmp, int fix3d,
                         hipStream_t st);
template <typename T>
hipError_t launch_fill(T *a, T v, uint64_t n, hipStream_t st);

// ---- 2D log-spherical path (kern_logsph.hip) --------------------------
// the 13 Grid_LogSph coefficient arrays (grid_log_sph.h:45-49), FP64
enum LsCoefIdx {
  LS_L1E, LS_L2E, LS_L3E, LS_L1B, LS_L2B, LS_L3B,
  LS_A1E, LS_A2E, LS_A3E, LS_A1B, LS_A2B, LS_A3B, LS_DV,
  LS_NCOEF
};
struct LsCoef {
  const double *a[LS_NCOEF];
};
// the SimParams entries of the log-spherical path (sim_params.h:31-64);
// gravity is 0 when gravity_on is off
struct LsParams {
  double compactness, omega, gravity, rad_cooling_coef, B0, damping_coef,
      track_percent;
  int rad_cooling_on, damping_length, inject_ions;
};

void logsph_coef_host(const Mesh &m, std::vector<double> (&c)[LS_NCOEF]);
hipError_t launch_logsph_push_f64(const Mesh &m, const Species &sp,
                                  const LsParams &lp, double dt, int H,
                                  int rho, const PtcF64 &p,
                                  const FieldsF64 &f, const AccF64 &a,
                                  unsigned long long *counters, uint64_t n,
                                  hipStream_t st, const unsigned long long *dn = nullptr,
                                  const CellRuns *runs = nullptr);
hipError_t launch_logsph_push_f32(const Mesh &m, const Species &sp,
                                  const LsParams &lp, float dt, int S,
                                  const PtcF32 &p, const FieldsF32 &f,
                                  const AccMixed &a,
                                  unsigned long long *counters, uint64_t n,
                                  hipStream_t st, const unsigned long long *dn = nullptr,
                                  const CellRuns *runs = nullptr);
template <typename T>
hipError_t launch_logsph_process_j(const Mesh &m, const LsCoef &cf, double dt,
                                   int H, int limbs, long long *const (*J)[2],
                                   long long *const (*R)[2], int ns,
                                   T *const *Jout, T *const *Rout,
                                   int axis, hipStream_t st);
template <typename T>
hipError_t launch_logsph_filter(const Mesh &m, T *j, T *tmp, const double *A,
                                hipStream_t st);
template <typename T>
hipError_t launch_logsph_axis_j3(const Mesh &m, T *J3, hipStream_t st);
template <typename T>
hipError_t launch_logsph_field_update(const Mesh &m, const LsCoef &cf,
                                      const LsParams &lp,
                                      const FieldSet<T> &f, double dt,
                                      double edotb_delta, hipStream_t st);
template <typename T>
hipError_t launch_logsph_field_boundary(const Mesh &m, const LsParams &lp,
                                        const FieldSet<T> &f, double omega,
                                        hipStream_t st);
template <typename R>
hipError_t launch_logsph_inject(const Mesh &m, const LsParams &lp,
                                const PtcView<R> &p, uint64_t number, int inj,
                                double p1, double w, double q_e, uint64_t seed,
                                uint32_t epoch, int Hs, uint64_t id_base,
                                long long *surf, hipStream_t st, int r_cells = 0,
                                double theta = 0.0, unsigned long long *dc = nullptr,
                                uint64_t cap = 0, unsigned long long *counters = nullptr);

// ---- 3D log-spherical force-free / vacuum solver (kern_ffe.hip) -------
template <typename T>
struct FfeBuf {
  T *En[3], *Bn[3], *dE[3], *dB[3];
};
template <typename T>
hipError_t launch_ffe_update(const Mesh &m, const LsCoef &cf, int damping_length,
                             double damping_coef, const FieldSet<T> &f,
                             const FfeBuf<T> &b, double dt, double omega,
                             double time, hipStream_t st);
template <typename T>
hipError_t launch_ffe_boundary(const Mesh &m, int damping_length,
                               double damping_coef, const FieldSet<T> &f,
                               double omega, hipStream_t st);
// mode 0: clean_epar (E -> dE), mode 1: check_eGTb (dE -> E)
template <typename T>
hipError_t launch_ffe_clean(const Mesh &m, const FieldSet<T> &f,
                            const FfeBuf<T> &b, int mode, hipStream_t st);

// ---- photons and pair creation (kern_rt.hip) ----------------------------
// photon_data (src/data/particle_data.h:68-81); the mixed form recomputes
// the photon energy from |p| and carries no id
struct PhoF64 {
  uint32_t *cell;
  double *x1, *x2, *x3;
  double *p1, *p2, *p3;
  double *E, *w, *path;
  uint32_t *flag;
  uint64_t *id;
};
struct PhoF32 {
  uint32_t *cell;
  float *x1, *x2, *x3;
  float *p1, *p2, *p3;
  float *w, *path;
  uint32_t *flag;
};
template <typename R>
struct PhoView {
  uint32_t *cell;
  R *x1, *x2, *x3;
  R *p1, *p2, *p3;
  R *E, *w, *path;
  uint32_t *flag;
  uint64_t *id;
};
inline PhoView<double> view_of(const PhoF64 &p) {
  return {p.cell, p.x1, p.x2, p.x3, p.p1, p.p2, p.p3, p.E, p.w, p.path, p.flag,
          p.id};
}
inline PhoView<float> view_of(const PhoF32 &p) {
  return {p.cell, p.x1, p.x2, p.x3, p.p1, p.p2, p.p3, nullptr, p.w, p.path,
          p.flag, nullptr};
}

// model 0: the reference's default hooks; model 1: exponential free path
struct RtParams {
  int model;
  double gamma_thr, photon_path, E_secondary, r_cutoff, e_frac;
  uint64_t max_ptc, max_photon;
};

// Counts kept on the device (a context's device-count mode): the particle
// and photon numbers, the next ids, event totals since the mode was
// entered, the Philox epochs of emission and injection, and the events of
// the last call.  Slots from a count up to the capacity are empty, so a
// kernel may run over any upper bound of the count.
enum {
  DC_NUM = 0,
  DC_PH = 1,
  DC_ID = 2,
  DC_PH_ID = 3,
  DC_EMITTED = 4,
  DC_CONVERTED = 5,
  DC_RT_EPOCH = 6,
  DC_INJ_EPOCH = 7,
  DC_LAST = 8,
  DC_PUSHED = 9,  // particle slots pushed (the count at each push, summed)
  DC_N = 10
};

// scan scratch of the emit / pair passes
struct RtWork {
  uint32_t *flags = nullptr;
  unsigned long long *total = nullptr, *host_total = nullptr;  // the latter pinned
  uint64_t *bsum = nullptr;  // per-workgroup event prefixes
  uint64_t cap = 0;
  uint64_t most = 0;  // slots its owner can ever have: no room beyond
  hipError_t ensure(uint64_t n);
  hipError_t alloc(uint64_t c);
  void release();
};

// dc (nullable): device-count mode -- the photon / particle base, the id
// base and the epoch are read from dc, the counts and totals updated there
// by a kernel, and nothing is read back (*emitted / *made are left 0).
template <typename R>
hipError_t rt_emit(const Mesh &m, const RtParams &rt, const PtcView<R> &p,
                   uint64_t n, const PhoView<R> &ph, uint64_t ph_base,
                   uint64_t seed, uint32_t epoch, uint64_t id_base,
                   RtWork &w, unsigned long long *counters, hipStream_t st,
                   R *produced, uint64_t *emitted, unsigned long long *dc = nullptr);
template <typename R>
hipError_t rt_pairs(const Mesh &m, const RtParams &rt, const PtcView<R> &p,
                    uint64_t p_base, const PhoView<R> &ph, uint64_t nph,
                    uint64_t id_base, RtWork &w, unsigned long long *counters,
                    hipStream_t st, R *produced, uint64_t *made,
                    unsigned long long *dc = nullptr);
// device-count bookkeeping kernels (kern_rt.hip): the cells of slots
// [*kept, n) emptied; dc[which] = *src
hipError_t launch_fill_tail(uint32_t *cell, const unsigned long long *kept, uint64_t n,
                            hipStream_t st);
hipError_t launch_dc_set(unsigned long long *dc, int which, const unsigned long long *src,
                         hipStream_t st);
// dc[to] += dc[from]
hipError_t launch_dc_accum(unsigned long long *dc, int to, int from, hipStream_t st);
template <typename R>
hipError_t rt_move_photons(const Mesh &m, int logsph, double r_cutoff,
                           const PhoView<R> &ph, uint64_t n, double dt,
                           hipStream_t st, const unsigned long long *dn = nullptr);

// ---- loading, sort, diagnostics -------------------------------------
struct LoadParams {
  int ppc;
  double theta[2];
  double drift[2];
  double weight;
  uint64_t seed;
  uint64_t base;  // index of the first new particle
};
hipError_t launch_load_uniform_f64(const Mesh &m, const LoadParams &lp,
                                   const PtcF64 &p,
                                   unsigned long long *counters,
                                   hipStream_t st);
hipError_t launch_load_uniform_f32(const Mesh &m, const LoadParams &lp,
                                   const PtcF32 &p,
                                   unsigned long long *counters,
                                   hipStream_t st);

// dn (nullable, here and below): the device-resident count that bounds
// the slots processed in device-count mode (n is then an upper bound)
hipError_t launch_erase_guard(const Mesh &m, uint32_t *cell, uint64_t n,
                              hipStream_t st, const unsigned long long *dn = nullptr);
hipError_t launch_energy_histogram_f64(const double *E, const uint32_t *flag,
                                       uint64_t n, uint32_t *hist, int nbins,
                                       double E_max, int flag_bit,
                                       hipStream_t st);
hipError_t launch_energy_histogram_mixed(const float *u1, const float *u2,
                                         const float *u3, const uint32_t *flag,
                                         uint64_t n, uint32_t *hist, int nbins,
                                         double E_max, int flag_bit,
                                         hipStream_t st);

// ---- 3D Cartesian force-free solver (kern_ffe_cart.hip) ---------------
template <typename T>
hipError_t launch_ffe_cart_curl_add(const Mesh &m, T *const v[3], const T *const u[3], T q,
                                    hipStream_t st);
template <typename T>
hipError_t launch_ffe_cart_edotb(const Mesh &m, T *eb, const T *const e[3], const T *const b[3],
                                 T q, hipStream_t st);
template <typename T>
hipError_t launch_ffe_cart_j(const Mesh &m, T *const j[3], const T *f, const T *const e[3],
                             const T *const b[3], T q, hipStream_t st);
template <typename T>
hipError_t launch_ffe_cart_de(const Mesh &m, T *const eo[3], T *const j[3], const T *const e[3],
                              const T *const b[3], T dt, hipStream_t st);

// ---- 1D pulsar gap (kern_1dgap.hip) ---------------------------------
hipError_t launch_gap_push(const Mesh &m, const Species &sp, const PtcF64 &p,
                           const double *e3, const AccF64 &acc, double dt, int H, uint64_t n,
                           unsigned long long *counters, hipStream_t st);
hipError_t launch_gap_photons(const Mesh &m, const PhoF64 &ph, double dt, uint64_t n,
                              hipStream_t st);
hipError_t launch_gap_filter(const Mesh &m, const double *j, double *tmp, int bnd_lower,
                             int bnd_upper, hipStream_t st);
hipError_t launch_gap_update_e(const Mesh &m, double *e1, const double *j1, double j0,
                               double dt, hipStream_t st);

// ---- 1D GR gap (kern_1dgr.hip) --------------------------------------
// Grid_1dGR::mesh_ptrs (grid_1dgr.h:17-21), one dims[0] array each
enum {
  GR_D1 = 0, GR_D2, GR_D3, GR_ALPHA, GR_THETA, GR_K1, GR_K1J, GR_J0, GR_AGRR,
  GR_AGRF, GR_RHO0, GR_GRR, GR_GFF, GR_BETA, GR_B3B1, GR_NCOEF
};
struct Gr1dCoef {
  const double *a[GR_NCOEF];
};
hipError_t launch_1dgr_push(const Mesh &m, const Gr1dCoef &cf, const Species &sp,
                            const PtcF64 &p, const double *e3, const AccF64 &acc,
                            double dt, uint32_t step, int data_interval, double a,
                            double omega, int H, uint64_t n, hipStream_t st);
hipError_t launch_1dgr_photons(const Mesh &m, const Gr1dCoef &cf, const PhoF64 &ph,
                               double dt, uint32_t step, int data_interval, uint64_t n,
                               hipStream_t st);
hipError_t launch_1dgr_filter(const Mesh &m, const double *j, double *tmp, const double *k1,
                              hipStream_t st);
hipError_t launch_1dgr_update_e(const Mesh &m, const Gr1dCoef &cf, double *e1,
                                const double *j1, double dt, hipStream_t st);

// charge arrays of the species, for the Gauss-law residual (kern_diag.hip)
template <typename T>
struct RhoSet {
  const T *r[4];
};
// largest number of blocks (and of partial maxima pairs) of the residual
constexpr int DIVRES_MAX_BLOCKS = 2048;
template <typename T>
hipError_t launch_div_residual(const Mesh &m, const T *divE, const RhoSet<T> &rho, int ns,
                               double kappa, double *out, double *part, int max_blocks,
                               int *nblocks, hipStream_t st);

// per-cell moments of collect_diagnostics (kern_diag.hip): num[s], gamma[s]
// for the four species slots and photon_num, ncell values each
template <typename R>
struct DiagArrays {
  R *num[4], *gamma[4];
  R *photon_num;
};
template <typename R>
hipError_t launch_diagnostics(const PtcView<R> &p, uint64_t n, const PhoView<R> &ph,
                              uint64_t nph, const DiagArrays<R> &d, int ns,
                              uint64_t ncell, hipStream_t st);

}  // namespace apt
