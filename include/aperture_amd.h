/*
 * aperture_amd.h -- C ABI of the MI355X-native Aperture PIC time step.
 *
 * Plain C: opaque context, pointers and sizes, status codes, no exceptions
 * and no C++ or torch types.  One context owns the device fields,
 * particles and a HIP stream (the state sim_data owns in the reference,
 * src/sim_data.h:14-70).  Every call is stream ordered; calls that return
 * data to the host synchronise the context's stream first.  A context is
 * used from one host thread at a time.
 *
 * Each entry point cites the reference interface it replaces (paths relative
 * to the fizban007/Aperture3 tree).
 */
#ifndef APERTURE_AMD_H
#define APERTURE_AMD_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef struct apt_ctx apt_ctx;
typedef int apt_status;

/* Status codes.  The reference throws (cudaUtility.h:62-74), exits
 * (cudaUtility.h:35-58, sim_environment_impl.hpp:54-59) or traps
 * (ptc_updater.cu:43-50); here every failure is a return code plus
 * apt_last_error(). */
enum {
  APT_OK = 0,
  APT_ERR_INVALID_ARG = 1,
  APT_ERR_HIP = 2,
  APT_ERR_CAPACITY = 3,
  APT_ERR_STATE = 4,
  APT_ERR_UNSUPPORTED = 5
};

/* Numeric forms. */
enum {
  APT_PREC_FP64 = 0,  /* plain FP64: the drop-in */
  APT_PREC_MIXED = 1  /* FP32 push/fields, int32 cell + FP32 offset,
                         int64 fixed-point current */
};

/* Coordinate systems (SimParams::coord_system, sim_params.h:101). */
enum {
  APT_COORD_CARTESIAN = 0,
  APT_COORD_LOGSPH = 1, /* 2D (ln r, theta), Grid_LogSph (grid_log_sph.h) */
  APT_COORD_1DGR = 2,   /* 1D along a Kerr field line, Grid_1dGR (grid_1dgr.h),
                           FP64 form */
  APT_COORD_1DGAP = 3   /* 1D pulsar gap co-rotating with beta_phi(x) = x
                           (coord_system "1DGap", labs/1dgap/config.toml),
                           FP64 form */
};

/* Pair-creation models (radiative_transfer hooks). */
enum {
  APT_RT_DEFAULT = 0, /* user_radiative_functions.cu:13-125 */
  APT_RT_EXP_PATH = 1 /* photon energy e_frac gamma, free path
                         -photon_path ln u */
};

/* Field identifiers (the members of sim_data, src/sim_data.h:40-60). */
enum {
  APT_FIELD_E = 0,
  APT_FIELD_B = 1,
  APT_FIELD_EBG = 2,
  APT_FIELD_BBG = 3,
  APT_FIELD_J = 4,
  APT_FIELD_RHO = 5, /* component = species */
  APT_FIELD_DIVE = 6,
  APT_FIELD_DIVB = 7,
  /* sim_data::EdotB (sim_data.h:57): E.B/|B| at cell centres, accumulated
   * with weight 1/data_interval by every log-spherical field update
   * (compute_edotb, cuda/sim_data.cu:235-265); zero it with apt_field_set
   * after output, as the pulsar lab does (labs/pulsar/src/main.cpp:106-108) */
  APT_FIELD_EDOTB = 8,
  /* photon_produced / pair_produced (sim_data.h:58-59): summed weights of
   * the particles that emitted and the photons that converted, per cell
   * (radiative_transfer.cu:48-57, 120-130); zeroed the same way */
  APT_FIELD_PHOTON_PRODUCED = 9,
  APT_FIELD_PAIR_PRODUCED = 10,
  /* the moments of apt_collect_diagnostics (sim_data.h:45-46, 60):
   * summed weight per species (component = species), weight-averaged
   * gamma per species, summed photon weight; readable after the first
   * collection */
  APT_FIELD_PTC_NUM = 11,
  APT_FIELD_GAMMA = 12,
  APT_FIELD_PHOTON_NUM = 13,
  /* the work fields of field_solver_ffe (field_solver_ffe.h:40-44: m_Etmp,
   * m_Btmp) and a scalar work field, allocated on first use */
  APT_FIELD_FFE_E = 14,
  APT_FIELD_FFE_B = 15,
  APT_FIELD_FFE_F = 16
};

/* Timed kernels (apt_timing_get). */
enum {
  APT_KERNEL_PUSH_DEPOSIT = 0,
  APT_KERNEL_FIELD = 1,
  APT_KERNEL_SORT = 2,
  APT_KERNEL_NUM = 3
};

/* Grid section of the config (sim_params.h:90-96) plus periodic_boundary
 * (sim_params.h:38).  Absent dimensions have N = 1 and guard = 0; the
 * dimensionality is the number of leading dimensions with N > 1
 * (quadmesh.h:357). */
typedef struct {
  int N[3];
  int guard[3];
  double lower[3];
  double size[3];
  int periodic[3];
} apt_grid;

/* Physics and run parameters (SimParamsBase, sim_params.h:17-98). */
typedef struct {
  int precision;            /* APT_PREC_* */
  int num_species;          /* num_species (sim_params.h:28) */
  double q_e;               /* q_e (:20); electrons carry -q_e */
  double ion_mass;          /* ion_mass (:27), in units of q_e */
  int data_interval;        /* data_interval (:46): Rho deposit cadence */
  int current_smoothing;    /* current_smoothing (:42) filter passes */
  int fix_3d_filter;        /* 1: 3D filter edge weight 1/32 instead of
                               the reference's 0.03152 */
  uint64_t max_ptc_number;  /* max_ptc_number (:22) */
  uint64_t random_seed;     /* random_seed (:116) */
  int tile[3];              /* mixed form: largest tile extent in cells
                               (0 = auto); an axis that is no multiple of it
                               is split evenly over ceil(N / extent) tiles,
                               the first N % tiles of them one cell longer */
  int tile_halo;            /* mixed form: LDS halo in cells (0 = auto) */
  int tile_threads;         /* mixed form: threads per tile workgroup
                               (0 = auto) */
  /* ---- log-spherical path (sim_params.h:31-64) ---- */
  int coord;                /* APT_COORD_* (coord_system, :101) */
  double compactness;       /* compactness (:33): beta_phi, omega_LT */
  double omega;             /* omega (:62): beta_phi's rotation rate */
  int gravity_on;           /* gravity_on (:31) */
  double gravity;           /* gravity (:32) */
  int rad_cooling_on;       /* rad_cooling_on (:34) */
  double rad_cooling_coef;  /* rad_cooling_coef (:35) */
  double B0;                /* B0 (:58), the cooling field scale */
  int damping_length;       /* damping_length (:47), cells */
  double damping_coef;      /* damping_coef (:48) */
  int inject_ions;          /* inject_ions (:64) */
  double track_percent;     /* track_percent (:56) */
  /* ---- pair creation (sim_params.h:52-79) ---- */
  int rt_model;             /* APT_RT_* */
  double gamma_thr;         /* gamma_thr (:52) */
  double photon_path;       /* photon_path (:73) */
  double E_secondary;       /* E_secondary (:78) */
  double r_cutoff;          /* r_cutoff (:79) */
  double e_frac;            /* APT_RT_EXP_PATH: photon energy / gamma */
  uint64_t max_photon_number; /* max_photon_number (:23) */
  /* ---- 1D GR gap (sim_params.h:58-63) ---- */
  double spin_a;            /* a, the black hole spin; taken as float like the
                               reference's omega, B0 and track_percent */
  /* ---- reference compatibility ---- */
  int reference_3d_b_stencil; /* 1: the 3D Cartesian B update of
                               field_solver.cu:214-234 as written (forward
                               differences, one cell off the staggering of E);
                               0 (default): the staggered backward differences
                               of the 1D/2D kernels and of div B */
  /* ---- tiled mixed form ---- */
  int cell_order_interval;  /* 3D: between sorts, each tile's particles are
                               laid out again cell by cell before every
                               cell_order_interval-th push (their field taps
                               through L1 are then shared by the lanes of a
                               wave); 0 = auto (5), negative = only at sorts.
                               The push and the current do not depend on
                               it; pair-creation draws are keyed by slot, so
                               with pair creation on it changes the random
                               realization, as the sort interval does. */
} apt_params;

/* Particle flag bit 27 is reserved: the mixed form's tiled push marks
 * deferred particles with it.  apt_ptc_set clears it in the mixed form. */
#define APT_FLAG_RESERVED (1u << 27)

/* Host view of particle_data (src/data/particle_data.h:50-61) in FP64.
 * Any member may be NULL on apt_ptc_get to skip it. */
typedef struct {
  uint32_t *cell;
  double *x1, *x2, *x3;
  double *p1, *p2, *p3;
  double *E; /* gamma */
  double *weight;
  uint32_t *flag;
  uint64_t *id;
} apt_particles;

/* Host view of photon_data (src/data/particle_data.h:68-81) in FP64. */
typedef struct {
  uint32_t *cell;
  double *x1, *x2, *x3;
  double *p1, *p2, *p3;
  double *E;
  double *weight;
  double *path_left;
  uint32_t *flag;
  uint64_t *id;
} apt_photons;

/* Bookkeeping of a context (no reference counterpart; for tests and
 * tools): counts, fixed-point exponents, id and random-stream epochs. */
typedef struct {
  uint64_t number;       /* particles (including empty slots) */
  uint64_t ph_number;    /* photons */
  int H;                 /* current fixed-point exponent */
  int Hs;                /* surface-density fixed-point exponent */
  uint64_t id_next;      /* next particle id (FP64 form) */
  uint64_t ph_id_next;   /* next photon id (FP64 form) */
  uint32_t rt_epoch;     /* emit_photons calls so far */
  uint32_t inject_epoch; /* inject calls so far */
} apt_info;

/* Device-side event counters that replace the reference's trap/printf
 * diagnostics (ptc_updater.cu:43-50, 251-255). */
typedef struct {
  uint64_t nan_momenta;
  uint64_t multi_cell_moves;
  uint64_t capacity_overflow;
  uint64_t outside_tile;
  /* FP64 form: particles outside the LDS current window of their tile of
   * cell-sorted slots (or, before the first sort, of a chunk of slots that
   * spread over more cells than its window holds), so their current went
   * straight to the accumulators in HBM (same sums, slower) */
  uint64_t global_deposits;
} apt_counters;

/* Largest max_ptc_number and max_photon_number: sorts and event scans
 * count slots with 32-bit signed integers. */
#define APT_MAX_SLOTS 0x7fffffffu

/* ---- lifetime ------------------------------------------------------- */
/* sim_environment(int*, char***) + sim_data(env)
 * (sim_environment_impl.hpp:17-65, sim_data_impl.hpp:12-71).  Capacities
 * above APT_MAX_SLOTS are refused with APT_ERR_INVALID_ARG. */
apt_status apt_create(const apt_grid *grid, const apt_params *params,
                      apt_ctx **out);
apt_status apt_destroy(apt_ctx *ctx);
/* the context's last error; with ctx == NULL, the message of the last
 * failed apt_create on the calling thread */
const char *apt_last_error(const apt_ctx *ctx);
/* fixed-point exponent H of the current (J = hi 2^-H + lo 2^-(H+40) in
 * the FP64 form, J = acc 2^-H in the mixed form) */
apt_status apt_get_jexp(const apt_ctx *ctx, int *H);
apt_status apt_get_mesh(const apt_ctx *ctx, int dims[3], double delta[3]);
apt_status apt_get_info(const apt_ctx *ctx, apt_info *out);
/* Restores id_next, ph_id_next, rt_epoch, inject_epoch and the exponents H
 * and Hs from `in` (the counter part of a snapshot; the reference stores
 * its XORWOW states instead, data_exporter.cpp:463-468).  Call after the
 * particles are set. */
apt_status apt_set_counters(apt_ctx *ctx, const apt_info *in);
/* Log-spherical metric coefficient `which` (0..12 in the order l1_e, l2_e,
 * l3_e, l1_b, l2_b, l3_b, A1_e, A2_e, A3_e, A1_b, A2_b, A3_b, dV;
 * Grid_LogSph members, grid_log_sph.h:45-49), dims0*dims1 doubles. */
apt_status apt_get_coef(apt_ctx *ctx, int which, double *dst, uint64_t count);

/* ---- data movement (multi_array copy_to/from_device, fields.h) ------- */
/* field<N,T>::initialize / copy_to_device (core/fields.h:111-143) */
apt_status apt_field_set(apt_ctx *ctx, int which, int comp,
                         const double *src, uint64_t count);
/* field<N,T>::copy_to_host */
apt_status apt_field_get(apt_ctx *ctx, int which, int comp, double *dst,
                         uint64_t count);
/* particles_t::copy_from / set_num (cuda/core/particle_base_impl.cu) */
apt_status apt_ptc_set(apt_ctx *ctx, const apt_particles *src, uint64_t n);
/* particles_t::copy_to_host */
apt_status apt_ptc_get(apt_ctx *ctx, apt_particles *dst, uint64_t cap,
                       uint64_t *n);
/* particle_base::number() */
apt_status apt_ptc_number(apt_ctx *ctx, uint64_t *n);
/* sim_data::fill_multiplicity (cuda/sim_data.cu:268-293) with
 * Maxwell-Juttner momenta: ppc co-located e-/e+ pairs per bulk cell,
 * theta[s] and x-drift[s] per species (s = 0 electrons, 1 positrons). */
apt_status apt_ptc_load_uniform(apt_ctx *ctx, int ppc_pairs,
                                const double theta[2], const double drift[2],
                                double weight);

/* photons: particles_t<photon_data>::copy_from / copy_to_host / number */
apt_status apt_ph_set(apt_ctx *ctx, const apt_photons *src, uint64_t n);
apt_status apt_ph_get(apt_ctx *ctx, apt_photons *dst, uint64_t cap,
                      uint64_t *n);

/* ---- the time step -------------------------------------------------- */
/* ptc_updater::update_particles(sim_data&, double dt, uint32_t step)
 * (src/algorithms/ptc_updater.h:11-24, cuda/algorithms/ptc_updater.cu:
 * 748-841): zero J (and Rho on deposit steps), push, move, deposit,
 * periodic fold and wrap, smoothing. */
apt_status apt_ptc_update(apt_ctx *ctx, double dt, uint32_t step);
/* ptc_updater::smooth_current(sim_data&, uint32_t step)
 * (ptc_updater.cu:852-873): current_smoothing binomial passes over J (and
 * Rho on deposit steps); apt_ptc_update already runs them once. */
apt_status apt_smooth_current(apt_ctx *ctx, uint32_t step);
/* field_solver::update_fields(sim_data&, double dt, uint32_t step)
 * (src/algorithms/field_solver.h:11-25, field_solver.cu:334-358); in a
 * log-spherical context field_solver_logsph::update_fields(sim_data&,
 * double dt, double time) (field_solver_logsph.h:10-20,
 * field_solver_logsph.cu:354-398): B, E, divergences, no half step. */
apt_status apt_field_update(apt_ctx *ctx, double dt, uint32_t step);
/* field_solver_logsph::apply_boundary(sim_data&, double omega, double time)
 * (field_solver_logsph.cu:403-428): rotating conductor, absorbing layer,
 * axis.  A no-op in a Cartesian context, like
 * field_solver::apply_outflow_boundary (field_solver.cu:451-452). */
apt_status apt_field_boundary(apt_ctx *ctx, double omega, double time);
/* ptc_updater_logsph::inject_ptc(sim_data&, int inj_per_cell, Scalar p1,
 * Scalar p2, Scalar p3, Scalar w, Scalar omega) (ptc_updater_logsph.h:13-28,
 * ptc_updater_logsph.cu:848-870); log-spherical contexts only. */
apt_status apt_inject_ptc(apt_ctx *ctx, int inj_per_cell, double p1,
                          double p2, double p3, double w, double omega);
/* Thermal shell injection (no reference counterpart: inject_ptc above
 * injects into one radial cell with a fixed momentum; the magnetosphere
 * workload injects pairs "in the inner cells with a temperature").  For
 * every row inject_ptc fills, inj_per_cell pairs in each of r_cells radial
 * cells from inject_ptc's cell (guard + 2) outward, under inject_ptc's
 * surface-density gate; each member's momentum an isotropic Maxwell-Juttner
 * draw at temperature theta (> 0), position uniform in the cell (shared by
 * the pair), weight w sin(theta_position).  1 <= r_cells <= 16. */
apt_status apt_inject_ptc_thermal(apt_ctx *ctx, int r_cells, int inj_per_cell, double theta,
                                  double w, double omega);
/* ffe_solver_logsph::update_fields(sim_data&, double dt, double omega,
 * double time) (src/algorithms/ffe_solver_logsph.h:12-33,
 * ffe_solver_logsph.cu:880-930): SSP-RK3 vacuum / force-free step of a 3D
 * log-spherical context (N = r, theta, phi; guard >= 3; phi periodic). */
apt_status apt_ffe_update(apt_ctx *ctx, double dt, double omega, double time);
/* ffe_solver_logsph::apply_boundary (ffe_solver_logsph.cu:932-966) */
apt_status apt_ffe_boundary(apt_ctx *ctx, double omega, double time);
/* ffe_solver_logsph::clean_epar (:1029-1037): the solver's dE copy of E
 * minus its component along B; check_eGTb (:1039-1047): E := that copy,
 * scaled down where |E| > |B|. */
apt_status apt_ffe_clean_epar(apt_ctx *ctx);
apt_status apt_ffe_check_egtb(apt_ctx *ctx);
/* ---- field_solver_ffe: the 3D Cartesian force-free solver -------------
 * (src/algorithms/field_solver_ffe.h:11-45,
 * src/cuda/algorithms/field_solver_ffe.cu:17-331).  Vector fields are
 * named by APT_FIELD_E, _B, _EBG, _BBG, _J, _FFE_E or _FFE_B; scalar
 * fields by APT_FIELD_DIVE, _DIVB, _EDOTB, _FFE_F (component 0) or
 * APT_FIELD_RHO (component = species).  Every bulk cell is updated; guard
 * cells are not refreshed (as in the reference).  The reference's
 * update_fields and compute_J have empty bodies (:292-298), so they have no
 * entry point. */
/* field_solver_ffe::update_field_substep(E_out, B_out, J_out, E_in, B_in, dt)
 * (field_solver_ffe.cu:300-331): B_out += dt curl E_in (curl_add,
 * finite_diff.cu:508-525, with the reference's + sign), then the
 * force-free current (rho E x B + (B.curl B - E.curl E) B) / B^2 of
 * (E_in, B_in), rho = div E, into J_out, and E_out += dt curl B_in
 * (compute_FFE_dE, :145-283).  The reference writes the current into its
 * private m_Etmp and leaves J_out untouched.  B_in may name B_out (then the
 * updated B is read, the reference's order) and E_out may name E_in (E_in is
 * then read from a copy); any other overlap is refused. */
apt_status apt_ffe_cart_substep(apt_ctx *ctx, int e_out, int b_out, int j_out, int e_in,
                                int b_in, double dt);
/* field_solver_ffe::ffe_edotb (compute_FFE_EdotB, :17-69, 333-354):
 * out += q E.B at each cell */
apt_status apt_ffe_cart_edotb(apt_ctx *ctx, int out, int out_comp, int e, int b, double q);
/* field_solver_ffe::ffe_j (compute_FFE_J, :71-143, 356-383):
 * j_out = q (f B + (div E) E x B) / B^2 */
apt_status apt_ffe_cart_j(apt_ctx *ctx, int j_out, int f, int f_comp, int e, int b,
                          double q);

/* radiative_transfer::emit_photons(sim_data&) / produce_pairs(sim_data&)
 * (radiative_transfer.h:11-28, radiative_transfer.cu:198-301); the
 * optional outputs return the number of events (in device-count mode a
 * non-NULL output synchronises the stream to read it). */
apt_status apt_emit_photons(apt_ctx *ctx, uint64_t *emitted);
apt_status apt_produce_pairs(apt_ctx *ctx, uint64_t *pairs);

/* ---- counts on the device; a recorded step ----------------------------
 * No reference counterpart: the reference reads every event count back
 * to the host (radiative_transfer.cu:225-228, 279-282) and keeps the
 * particle number there.  In device-count mode (2D log-spherical
 * contexts) the particle and photon counts, next ids, emission and
 * injection epochs and the event totals stay in device memory: injection,
 * emission, pair creation and the sort read their bases from it and update
 * it with kernels, so a step issues no host synchronisation.  Calls that
 * return counts or particle data (apt_ptc_number, apt_get_info,
 * apt_ptc_get, apt_ph_get, histograms, diagnostics) synchronise and read
 * them.  In this mode, injected pairs past the particle capacity are
 * dropped and counted in capacity_overflow instead of failing the call. */
apt_status apt_set_device_counts(apt_ctx *ctx, int on);
/* photons emitted and pairs converted since device counts were turned on;
 * pushed (nullable): particle slots pushed, the count at each
 * apt_ptc_update summed */
apt_status apt_get_events(apt_ctx *ctx, uint64_t *emitted, uint64_t *converted,
                          uint64_t *pushed);
/* Records the calls made between apt_graph_begin and apt_graph_end (for
 * example one step: inject, update_particles, update_fields,
 * apply_boundary, emit_photons, produce_pairs) into a HIP graph that
 * apt_graph_launch replays `times` times.  In device-count mode the
 * recorded launches cover the whole capacity, so replays stay valid as the
 * counts grow.  With host counts a recording may hold only calls that
 * change no count (update_particles, update_fields, apply_boundary,
 * filters: a periodic Cartesian step); injection, emission and pair
 * creation then fail with APT_ERR_STATE.  Not recordable in either mode:
 * sorts and any call that reads counts back.
 * Arguments are fixed at recording: a replayed step keeps its step number
 * (the charge-deposit cadence), time and dt, and the particle buffers of
 * the current sort parity (record again after a sort).  In a 3D tiled
 * mixed run an eager push that lays the tiles out again by cell (see
 * cell_order_interval) swaps those buffers and drops the recording; on a
 * mesh with an axis that is no multiple of the tile extent the tiles are
 * not laid out again while there is a recording. */
apt_status apt_graph_begin(apt_ctx *ctx);
apt_status apt_graph_end(apt_ctx *ctx);
apt_status apt_graph_launch(apt_ctx *ctx, int times);
/* field_solver::update_e_field / update_b_field / compute_divs
 * (field_solver.cu:360-504) */
apt_status apt_field_update_e(apt_ctx *ctx, double dt);
apt_status apt_field_update_b(apt_ctx *ctx, double dt);
apt_status apt_field_compute_divs(apt_ctx *ctx);
/* sim_data::sort_particles -> particle_base::sort_by_cell for particles and
 * photons (sim_data_impl.hpp:78-89, cuda/core/particle_base_impl.cu:435-464) */
apt_status apt_sort_particles(apt_ctx *ctx);
/* particle_base::clear_guard_cells (particle_base_impl.cu:489-493) */
apt_status apt_clear_guard_cells(apt_ctx *ctx);

/* ---- 1D GR gap (APT_COORD_1DGR) -------------------------------------- */
/* Grid_1dGR::compute_coef (grid_1dgr.cpp:21-175) from the field-line
 * profile the reference reads from coef.h5 (datasets r, Bu1, Bu3, rho,
 * ju1, th, dpsidth; taken as float): the 15 arrays D1, D2, D3, alpha,
 * theta, K1, K1_j, j0, agrr, agrf, rho0, gamma_rr, gamma_ff, beta_phi,
 * B3B1 (read back with apt_get_coef, which = 0..14, dims[0] each). */
apt_status apt_1dgr_set_profile(apt_ctx *ctx, const double *r, const double *B1,
                                const double *B3, const double *rho, const double *jr,
                                const double *theta, const double *dpsidth, uint64_t n);
/* ptc_updater_1dgr::prepare_initial_condition (ptc_updater_1dgr.cu:16-72,
 * 491-503): `multiplicity` pairs per bulk cell at rest, weights from B0 and
 * rho0 K1, tracked with probability track_percent.  apt_ptc_update and
 * apt_field_update on a 1D GR context run ptc_updater_1dgr and
 * field_solver_1dgr. */
apt_status apt_1dgr_initial_condition(apt_ctx *ctx, int multiplicity);
/* ---- 1D pulsar gap (APT_COORD_1DGAP) ---------------------------------- */
/* ptc_updater_1dgap::prepare_initial_condition(sim_data&, int multiplicity)
 * (src/algorithms/ptc_updater_1dgap.h:12-25, ptc_updater_1dgap.cu:21-72,
 * 236-248): `multiplicity` co-located e-/e+ pairs per bulk cell at rest in
 * the rotating frame, weights 2 B0/multiplicity plus the Goldreich-Julian
 * excess B0 omega atan(2x)/multiplicity of their sign, tracked with
 * probability track_percent.  apt_ptc_update on a 1D gap context runs
 * ptc_updater_1dgap::update_particles (the rotating-frame pusher, J1 and
 * Rho on every step, current_smoothing passes of the 1-2-1 filter over E,
 * J1 and Rho, photons at c along p1); apt_field_update runs
 * field_solver_1dgap::update_fields (field_solver_1dgap.h:9-18,
 * field_solver_1dgap.cu:14-39): E1 += (j0 - J1) dt with j0 = 1.6 B0. */
apt_status apt_1dgap_initial_condition(apt_ctx *ctx, int multiplicity);
/* AdditionalDiagnostics::collect_diagnostics
 * (cuda/core/additional_diagnostics.cu:78-100): per cell and species the
 * summed weight (APT_FIELD_PTC_NUM) and the weight-averaged gamma
 * (APT_FIELD_GAMMA: 0 where the summed weight is below 1e-5, Op_DivAssign,
 * core/detail/op.hpp:42-49), and the summed photon weight
 * (APT_FIELD_PHOTON_NUM).  Indexed by the full cell in 3D (the reference
 * indexes (c1, c2) only).  Sums are device atomics, as in the reference. */
apt_status apt_collect_diagnostics(apt_ctx *ctx);
/* Kernels::compute_energy_histogram (cuda/kernels.cu:36-69); hist has nbins
 * entries and is overwritten.  flag_bit < 0: every particle slot. */
apt_status apt_energy_histogram(apt_ctx *ctx, uint32_t *hist, int nbins,
                                double E_max, int flag_bit);

/* Largest nbins of apt_energy_histogram_noalloc: the size, in uint32
 * counts, of the library's static device array (32 KiB per GPU, held until
 * the process ends). */
#define APT_NOALLOC_HIST_MAX_BINS 8192

/* apt_energy_histogram without any allocation.  No counterpart in the
 * reference: it is for callers that cannot allocate device memory (code
 * under HIP graph capture, tight serving loops, harnesses that forbid
 * hipMalloc).  The same histogram as apt_energy_histogram, counted in a
 * static device array of APT_NOALLOC_HIST_MAX_BINS entries (one per GPU,
 * its address resolved in apt_create) instead of a buffer allocated per
 * call; no hipMalloc, hipFree or allocating library call.  hist (host
 * memory, nbins entries) is overwritten; nbins above
 * APT_NOALLOC_HIST_MAX_BINS is refused with APT_ERR_INVALID_ARG.  Every
 * call on one GPU shares that GPU's array: calls that overlap in time on
 * one GPU (two host threads, two contexts on one device) race and must be
 * serialised by the caller. */
apt_status apt_energy_histogram_noalloc(apt_ctx *ctx, uint32_t *hist, int nbins,
                                        double E_max, int flag_bit);

/* The Gauss-law check of the step (the |div E - 4 pi rho| residual the
 * FP64 form must hold at round-off; no reference counterpart, the reference
 * writes div E and Rho out, field_solver.cu:454-504, ptc_updater.cu:
 * 379-382): r = div E - kappa sum_s Rho_s over the bulk cells, from the
 * context's div E (written by apt_field_update / apt_field_compute_divs)
 * and the charge of the last deposit step, summed in FP64 on the device.
 * kappa is the path's normalisation: dt/delta in a Cartesian context with
 * equal cell sizes (J carries no delta/dt, E -= dt J), 1 in a log-spherical
 * one (process_j).  Returns max |r| and max |div E| over the bulk; residual
 * (optional, count = the context's cell count) receives r, 0 in guard
 * cells. */
apt_status apt_div_residual(apt_ctx *ctx, double kappa, double *max_abs, double *scale,
                            double *residual, uint64_t count);

/* Mixed form: tile binning of the particle array (no reference
 * counterpart; the reference sorts by cell).  Writes ntiles + 1 offsets:
 * tile t owns slots [off[t], off[t+1]); *ntiles = 0 when the particles are
 * not binned (untiled mesh, or not sorted since the last apt_ptc_set).
 * tile_extent receives the largest extent of a tile (see apt_params::tile
 * for the even split of an axis that is no multiple of it). */
apt_status apt_tile_offsets(apt_ctx *ctx, uint32_t *off, uint64_t cap,
                            uint32_t *ntiles, int tile_extent[3]);

/* Measurement (no reference counterpart): the speed of light of the mixed
 * form's particle stream.  Runs `reps` launches of a kernel that reads the
 * 9 particle arrays of the first n particles and writes 7 of them back
 * (unchanged) -- the push's HBM traffic with no arithmetic -- and returns
 * the average milliseconds per launch. */
apt_status apt_stream_probe(apt_ctx *ctx, uint64_t n, int reps, double *ms);

/* ---- control -------------------------------------------------------- */
apt_status apt_sync(apt_ctx *ctx);
apt_status apt_get_counters(apt_ctx *ctx, apt_counters *out);
apt_status apt_reset_counters(apt_ctx *ctx);
/* HIP-event timing of the kernels named by APT_KERNEL_* on the context's
 * stream; apt_timing_get synchronises and returns the summed milliseconds
 * and launch count since the last enable. */
apt_status apt_timing_enable(apt_ctx *ctx, int on);
apt_status apt_timing_get(apt_ctx *ctx, int kernel, double *total_ms,
                          uint64_t *launches);

/* ---- batched ensemble of 1D gap boxes ----------------------------------
 * Many independent 1D open boxes of uneven sizes advanced together: the
 * loop of labs/1dgap/src/main.cpp:61-98 (update_particles, clear_guard_cells
 * of particles and photons, update_fields, emit_photons, produce_pairs,
 * sort_by_cell every sort_interval steps) per box, with wall injection of
 * `inj` e-/e+ pairs per step at the left wall before the push.  The
 * reference runs one box per process; there is no batched counterpart.
 * Physics per box: ptc_updater.cu:21-499 (1D Cartesian Vay push + deposit),
 * field_solver.cu:14-235 (1D Yee, half E step at step 0),
 * radiative_transfer.cu:28-301 with the exponential free-path model
 * (E_ph = e_frac gamma, path = -photon_path ln u).  Box k runs with its own
 * seed (apt_batch_inst_seed) and reproduces the single-box FP64 path. */
typedef struct apt_batch apt_batch;

typedef struct {
  int N;              /* bulk cells; the box is [0, 1), delta = 1/N */
  int guard;          /* guard cells per side, >= 2 */
  int ppc;            /* initial particles per cell per species */
  int inj;            /* wall-injected pairs per step */
  uint64_t cap;       /* particle slots of this box */
  uint64_t ph_cap;    /* photon slots of this box */
  double cfl;         /* dt = cfl * delta, 0 < cfl < 1 */
  double weight;      /* particle weight */
  double theta;       /* Maxwell-Juttner temperature (load and injection) */
  double gamma_thr;   /* emission threshold Lorentz factor */
  double Bx;          /* uniform B_x (and background B_x) */
  double j0;          /* imposed current of the gap: the E update is
                         E1 += (j0 - J1) dt (update_e_1dgap,
                         field_solver_1dgap.cu:14-23); 0: plain Yee */
} apt_batch_inst;

typedef struct {
  int precision;        /* APT_PREC_* */
  double q_e;           /* charge unit (electron -q_e) */
  double ion_mass;
  uint64_t seed;        /* box k uses seed + 0x9E3779B97F4A7C15 (k + 1) */
  int chunk;            /* particles per workgroup: 256, 512 or 1024
                           (FP64: 256 or 512) */
  int grid_mult;        /* persistent push workgroups per CU, 1..64 */
  int sort_interval;    /* 0: never */
  double photon_path;   /* mean free path */
  double e_frac;        /* photon energy / parent gamma */
  double r_cutoff;      /* photons with a longer path are dropped */
} apt_batch_params;

apt_status apt_batch_create(const apt_batch_inst *specs, int n,
                            const apt_batch_params *params, apt_batch **out);
apt_status apt_batch_destroy(apt_batch *b);
const char *apt_batch_last_error(const apt_batch *b);
/* number of boxes */
apt_status apt_batch_size(const apt_batch *b, int *n);
/* the fixed-point exponent of the current accumulators */
apt_status apt_batch_get_jexp(const apt_batch *b, int *H);
apt_status apt_batch_inst_seed(const apt_batch *b, int inst, uint64_t *seed);
/* initial state: 2 ppc N particles per box (the apt_ptc_load_uniform
 * loader on the box's slots with its seed and theta), B_x = Bbg_x = Bx */
apt_status apt_batch_load(apt_batch *b, const apt_batch_inst *specs);
/* nsteps steps of every box (graph replays after step 0 when enabled) */
apt_status apt_batch_step(apt_batch *b, int nsteps);
apt_status apt_batch_graph(apt_batch *b, int on);
apt_status apt_batch_sort(apt_batch *b);
apt_status apt_batch_sync(apt_batch *b);
apt_status apt_batch_counts(apt_batch *b, uint64_t *number, uint64_t *ph_number);
apt_status apt_batch_get_counters(apt_batch *b, apt_counters *out);
/* particles pushed (live at push time) over all steps so far */
apt_status apt_batch_pushes(apt_batch *b, uint64_t *total);
/* pair-creation events over all steps so far, summed over the boxes:
 * photons emitted (written to a photon slot) and photons converted into a
 * pair (radiative_transfer.cu:198-301 per box) */
apt_status apt_batch_events(apt_batch *b, uint64_t *emitted, uint64_t *converted);
/* on = 1 start, 0 stop, -1 read only; sums since the last switch */
apt_status apt_batch_timing(apt_batch *b, int on, double *step_ms, double *push_ms,
                            uint64_t *steps);
apt_status apt_batch_get_particles(apt_batch *b, int inst, apt_particles *dst,
                                   uint64_t cap, uint64_t *n);
apt_status apt_batch_set_particles(apt_batch *b, int inst, const apt_particles *src,
                                   uint64_t n);
apt_status apt_batch_get_photons(apt_batch *b, int inst, apt_photons *dst,
                                 uint64_t cap, uint64_t *n);
/* which = APT_FIELD_E/B/EBG/BBG/J, count = N + 2 guard */
apt_status apt_batch_get_field(apt_batch *b, int inst, int which, int comp,
                               double *dst, uint64_t count);
apt_status apt_batch_set_field(apt_batch *b, int inst, int which, int comp,
                               const double *src, uint64_t count);
/* the ensemble workload draw: per box, Philox4x32-10 keyed (seed, box)
 * gives N = exp(U[ln 1024, ln 16384]), ppc = U[50, 400], Bx = U[0.5, 2],
 * theta = U[0.01, 0.3], gamma_thr = U[1e2, 1e4], and the gap's imposed
 * current j0 = 2 gamma_thr N^2 / (cfl^2 n*^2), n* = U[300, 700]: with unit
 * charge and mass, a particle at rest in the unscreened gap
 * (E1 = n dt j0 after n steps) reaches gamma_thr after about n* steps */
apt_status apt_batch_sample(uint64_t seed, int n, apt_batch_inst *out);

/* ---- inverse-Compton tables (rt_ic.cu:22-547) ------------------------ */
/* The reference's inverse_compton: the IC scattering rate, the
 * gamma-gamma pair-creation rate and the lab-frame spectra of scattered
 * photons (as cumulative distributions over e1 = E_ph / gamma, linear and
 * logarithmic grids) on a grid of n_gamma Lorentz factors in [1.01, 1e15],
 * for a soft-photon spectrum of src/radiation/spectra.h.  Independent of a
 * PIC context. */
typedef struct apt_ic apt_ic;
enum {
  APT_SPEC_POWER_LAW_HARD = 0,   /* p = delta, emin, emax */
  APT_SPEC_POWER_LAW_SOFT = 1,   /* p = alpha, emin, emax */
  APT_SPEC_BROKEN_POWER_LAW = 2, /* p = alpha, delta, epeak, emin, emax */
  APT_SPEC_BLACK_BODY = 3,       /* p = kT */
  APT_SPEC_MONO_ENERGETIC = 4    /* p = e0, de */
};
typedef struct {
  int kind;
  double p[5];
} apt_ic_spectrum;
enum {
  APT_IC_GAMMAS = 0,       /* n_gamma */
  APT_IC_EP = 1,           /* n_ep, e1 = i / (n_ep - 1) */
  APT_IC_LOG_EP = 2,       /* n_ep, 1e-10 .. 1 logarithmic */
  APT_IC_RATE = 3,         /* n_gamma: ic_rate */
  APT_IC_GG_RATE = 4,      /* n_gamma: gg_rate */
  APT_IC_DNDE = 5,         /* n_gamma x n_ep (e1 fastest): CDF on EP */
  APT_IC_DNDE_THOMSON = 6  /* n_gamma x n_ep: CDF on LOG_EP */
};
/* inverse_compton(params) (rt_ic.cu:227-282): params.n_gamma, n_ep grids
 * (each at least 3, n_gamma * n_ep at most 2^27) */
apt_status apt_ic_create(int n_gamma, int n_ep, apt_ic **out);
apt_status apt_ic_destroy(apt_ic *h);
const char *apt_ic_last_error(const apt_ic *h);
/* inverse_compton::init(n_e, emin, emax, n0) (rt_ic.cu:279-421), on the GPU */
apt_status apt_ic_init(apt_ic *h, const apt_ic_spectrum *spec, double emin, double emax,
                       double n0);
apt_status apt_ic_get_table(apt_ic *h, int which, double *dst, uint64_t count);
/* Kernels::gen_photon_e (rt_ic.cu:127-153) for n Lorentz factors, with the
 * uniform draw from the Philox stream (seed, index, epoch); host arrays */
apt_status apt_ic_gen_photon_e(apt_ic *h, const double *gamma, double *eph, uint64_t n,
                               uint64_t seed, uint32_t epoch);
/* the same on device arrays, ordered on `stream` (a hipStream_t; NULL: the
 * handle's own stream) */
apt_status apt_ic_gen_photon_e_dev(apt_ic *h, const double *gamma, double *eph, uint64_t n,
                                   uint64_t seed, uint32_t epoch, void *stream);
/* inverse_compton::generate_photon_energies (rt_ic.cu:515-522): device
 * arrays; sample k scatters when the first uniform of its Philox block
 * (seed, k, epoch) is below find_ic_rate(gammas[k]) and then takes
 * gen_photon_e with the second; e_ph[k] = 0 otherwise */
apt_status apt_ic_generate_photon_energies(apt_ic *h, double *e_ph, const double *gammas,
                                           uint64_t n, uint64_t seed, uint32_t epoch,
                                           void *stream);
/* inverse_compton::generate_random_gamma (rt_ic.cu:524-529): device array
 * of n Lorentz factors log-uniform in [1.01, 1e10] */
apt_status apt_ic_generate_random_gamma(apt_ic *h, double *gammas, uint64_t n, uint64_t seed,
                                        uint32_t epoch, void *stream);
/* Kernels::find_ic_rate / find_gg_rate (rt_ic.cu:156-171); host arrays */
apt_status apt_ic_rates(apt_ic *h, const double *gamma, double *ic_rate, double *gg_rate,
                        uint64_t n);

/* ---- triplet pair-production tables (rt_tpp.cu:21-294) --------------- */
/* The reference's triplet_pairs (a file its build does not compile): the
 * triplet rate and mean pair energy per Lorentz factor on the
 * inverse-Compton gamma grid, and the cumulative pair-energy spectrum
 * (n_gamma x n_gamma, pair energy fastest).  Rows where some soft photon
 * has s = gamma e < 4 are NaN, as in the reference (E_plus_min takes the
 * square root of a negative number there). */
typedef struct apt_tpp apt_tpp;
enum {
  APT_TPP_GAMMAS = 0, /* n_gamma */
  APT_TPP_RATE = 1,   /* n_gamma */
  APT_TPP_EM = 2,     /* n_gamma: mean pair energy fraction */
  APT_TPP_DNDE = 3    /* n_gamma x n_gamma: CDF over pair energy = gammas[i] */
};
/* triplet_pairs(params) (rt_tpp.cu:147-184); 3 <= n_gamma <= 11585 */
apt_status apt_tpp_create(int n_gamma, apt_tpp **out);
apt_status apt_tpp_destroy(apt_tpp *h);
const char *apt_tpp_last_error(const apt_tpp *h);
/* triplet_pairs::init(n_e, emin, emax, n0) (rt_tpp.cu:188-275), on the GPU */
apt_status apt_tpp_init(apt_tpp *h, const apt_ic_spectrum *spec, double emin, double emax,
                        double n0);
apt_status apt_tpp_get_table(apt_tpp *h, int which, double *dst, uint64_t count);
/* Kernels::gen_tpp_Ep (rt_tpp.cu:132-143) for n Lorentz factors, the draw
 * of index k from the Philox stream (seed, k, epoch); host arrays */
apt_status apt_tpp_gen_ep(apt_tpp *h, const double *gamma, double *e_p, uint64_t n,
                          uint64_t seed, uint32_t epoch);
/* Kernels::find_tpp_rate / find_tpp_Em (rt_tpp.cu:114-130); host arrays */
apt_status apt_tpp_rates(apt_tpp *h, const double *gamma, double *rate, double *em,
                         uint64_t n);

/* ---- analytic emission models (inverse_compton_*.{h,cuh}) ------------ */
/* InverseComptonPL1D (inverse_compton_power_law.cuh:11-190) and
 * InverseComptonDummy (inverse_compton_dummy.cuh:7-40): for each particle
 * (gamma, p), emit_photon, then draw_photon_energy and
 * draw_photon_freepath (emit = 0 leaves eph = path = 0).  The four draws
 * of particle k are the uniforms of the Philox blocks (seed, k, epoch)
 * instead of a curand state.  Fields as SimParams: alpha =
 * spectral_alpha, e_s, e_min, photon_path, ic_rate = delta_t / ic_path,
 * E_cutoff, E_ph (the dummy's). */
enum { APT_ICM_DUMMY = 0, APT_ICM_POWER_LAW = 1 };
typedef struct {
  int kind;
  double alpha, e_s, e_min, photon_path, ic_rate, E_cutoff, E_ph;
} apt_ic_model;
/* device arrays, ordered on `stream` (a hipStream_t; NULL: the default
 * stream) */
apt_status apt_ic_model_emit(const apt_ic_model *model, const double *gamma, const double *p,
                             uint8_t *emit, double *eph, double *path, uint64_t n,
                             uint64_t seed, uint32_t epoch, void *stream);

#ifdef __cplusplus
}
#endif
#endif /* APERTURE_AMD_H */
