// kern_logsph.hip -- the 2D log-spherical (ln r, theta) path:
//   * Grid_LogSph::compute_coef (grid_log_sph.cpp:10-104) on the host, FP64;
//   * fused push + move + deposit: user_push_2d_logsph<1>
//     (user_push_2d_logsph.cuh:14-114: Vay, gravity, perpendicular cooling)
//     then deposit_and_move_2d_log_sph<1> (ptc_updater_logsph.cu:134-282:
//     straight line in Cartesian, back to (ln r, theta, phi), axis
//     reflection, Esirkepov in index space), one thread per particle;
//   * process_j (:284-299), filter_current_logsph (:616-666), the particle
//     boundaries of apply_boundary (:812-846);
//   * the integral-form Yee update, divergences and field boundaries of
//     field_solver_logsph.cu:28-345;
//   * measure_surface_density + inject_ptc (:301-395, 440-493).
// R = double is the FP64 form: contraction off, the shared elementary
// functions of apt_math.hpp, all nine interpolation taps in reference
// order, two-limb fixed-point current -- bit-identical to the CPU
// restatement.  R = float is the mixed form: FP32 arithmetic and library
// functions, two-tap gathers, single-limb int64 current; the metric
// coefficients stay FP64.
#include <type_traits>
#include <vector>

#include "apt_common.hpp"
#include "apt_f32.hpp"
#include "apt_f64.hpp"
#include "apt_kernels.hpp"
#include "apt_runs.hpp"
#include "apt_math.hpp"
#include "apt_mj.hpp"

#include <climits>

namespace apt {

constexpr double LS_PI = 3.14159265358979323846;

// Quadmesh::pos(i, n, pos_in_cell) (quadmesh.h:144-150)
__host__ __device__ inline double lpos(const Mesh &m, int d, int n, double x) {
  return m.lower[d] + m.delta[d] * ((double)(n - m.guard[d]) + x);
}
__host__ __device__ inline double spos(const Mesh &m, int d, int n, int st) {
  return lpos(m, d, n, st ? 1.0 : 0.5);
}

// ---------------------------------------------------------------------
// metric coefficients (host, FP64, C library -- like the reference)
// ---------------------------------------------------------------------
static double g_l1(double r, double rs) {
  double a = sqrt(1.0 - rs / r);
  return r * a + 0.5 * rs * log(2.0 * r * (1.0 + a) - rs);
}
static double g_A2(double r, double rs) {
  double a = sqrt(1.0 - rs / r);
  return 0.25 * r * a * (2.0 * r + 3.0 * rs) +
         0.375 * rs * rs * log(2.0 * r * (1.0 + a) - rs);
}
static double g_V3(double r, double rs) {
  double a = sqrt(1.0 - rs / r);
  return r * a * (8.0 * r * r + 10.0 * r * rs + 15.0 * rs * rs) / 24.0 +
         0.3125 * rs * rs * rs * log(2.0 * r * (1.0 + a) - rs);
}

void logsph_coef_host(const Mesh &m, std::vector<double> (&c)[LS_NCOEF]) {
  const double r_g = 0.0;  // grid_log_sph.cpp:14
  const int d0 = m.dims[0];
  const size_t n = (size_t)m.dims[0] * m.dims[1];
  for (int k = 0; k < LS_NCOEF; k++) c[k].assign(n, 0.0);
  const double D0 = m.delta[0], D1 = m.delta[1];
  for (int j = 0; j < m.dims[1]; j++) {
    double x2 = spos(m, 1, j, 0), x2s = spos(m, 1, j, 1);
    for (int i = 0; i < d0; i++) {
      size_t o = (size_t)i + (size_t)j * d0;
      double x1 = spos(m, 0, i, 0), x1s = spos(m, 0, i, 1);
      double r_plus = exp(x1 + D0), r = exp(x1), rs = exp(x1s),
             rs_minus = exp(x1s - D0);
      bool axis = fabs(x2s) < 1.0e-5 || fabs(x2s - LS_PI) < 1.0e-5;
      c[LS_L1E][o] = g_l1(rs, r_g) - g_l1(rs_minus, r_g);
      c[LS_L2E][o] = rs * D1;
      c[LS_L3E][o] = rs * sin(x2s);
      c[LS_L1B][o] = g_l1(r_plus, r_g) - g_l1(r, r_g);
      c[LS_L2B][o] = r * D1;
      c[LS_L3B][o] = r * sin(x2);
      c[LS_A1E][o] = r * r * (cos(x2) - cos(x2 + D1));
      if (axis) c[LS_A1E][o] = r * r * 2.0 * (1.0 - cos(0.5 * D1));
      c[LS_A2E][o] = (g_A2(r_plus, r_g) - g_A2(r, r_g)) * sin(x2);
      c[LS_A3E][o] = (g_A2(r_plus, r_g) - g_A2(r, r_g)) * D1;
      c[LS_A1B][o] = rs * rs * (cos(x2s - D1) - cos(x2s));
      c[LS_A2B][o] = (g_A2(rs, r_g) - g_A2(rs_minus, r_g)) * sin(x2s);
      c[LS_A3B][o] = (g_A2(rs, r_g) - g_A2(rs_minus, r_g)) * D1;
      c[LS_DV][o] = (g_V3(r_plus, r_g) - g_V3(r, r_g)) *
                    (cos(x2) - cos(x2 + D1)) / (D0 * D1);
      if (axis)
        c[LS_DV][o] = (g_V3(r_plus, r_g) - g_V3(r, r_g)) * 2.0 *
                      (1.0 - cos(0.5 * D1)) / (D0 * D1);
    }
  }
}

// ---------------------------------------------------------------------
// elementary functions per form
// ---------------------------------------------------------------------
template <typename R>
struct LsMath;
template <>
struct LsMath<double> {
  static __device__ double exp(double x) { return apt_exp(x); }
  static __device__ void sincos(double x, double &s, double &c) {
    apt_sincos(x, s, c);
  }
  static __device__ double sin(double x) { return apt_sin(x); }
  static __device__ double acos(double t) { return apt_acos(t); }
  static __device__ double atan2(double y, double x) { return apt_atan2(y, x); }
  static __device__ double log(double x) { return apt_log(x); }
};
template <>
struct LsMath<float> {
  static __device__ float exp(float x) { return expf(x); }
  static __device__ void sincos(float x, float &s, float &c) {
    sincosf(x, &s, &c);
  }
  static __device__ float sin(float x) { return sinf(x); }
  static __device__ float acos(float t) {
    return acosf(fminf(fmaxf(t, -1.0f), 1.0f));
  }
  static __device__ float atan2(float y, float x) { return atan2f(y, x); }
  static __device__ float log(float x) { return logf(x); }
};

// beta_phi (field_solver_logsph.cu:16-20); alpha_gr == 1 (:22-26)
template <typename R>
__device__ inline R beta_phi(const LsParams &lp, R r, R theta) {
  return (R)(-0.4) * (R)lp.compactness * (R)lp.omega * LsMath<R>::sin(theta) /
         (r * r);
}

// the s-th of four pointers (null past them) by selects: an array indexed by
// the species would be copied to scratch
__device__ __forceinline__ long long *pick4(int s, long long *a, long long *b, long long *c,
                                            long long *d) {
  return s == 0 ? a : s == 1 ? b : s == 2 ? c : s == 3 ? d : nullptr;
}

// current accumulation per form: a contribution to component c (or to
// the charge of species s) at mesh cell (x, y)
struct LsAccF64 {
  long long *J[3][2];
  long long *R[4][2];
  int H, d0;
  __device__ long long *at(int q, int l) const { return q < 3 ? J[q][l] : R[q - 3][l]; }
  __device__ void add(int c, int x, int y, double v) const {
    acc_add(J[c][0], J[c][1], (uint64_t)x + (uint64_t)y * d0, v, H);
  }
  __device__ void add_rho(int s, int x, int y, double v) const {
    // species without a charge array (s >= num_species) are not recorded
    long long *h = pick4(s, R[0][0], R[1][0], R[2][0], R[3][0]);
    if (h)
      acc_add(h, pick4(s, R[0][1], R[1][1], R[2][1], R[3][1]), (uint64_t)x + (uint64_t)y * d0, v,
              H);
  }
};
struct LsAccF32 {
  long long *J[3];
  long long *R[4];
  float scale;
  int d0;
  __device__ long long *at(int q, int) const { return q < 3 ? J[q] : R[q - 3]; }
  __device__ void add(int c, int x, int y, float v) const {
    acc_fx(J[c], (uint64_t)x + (uint64_t)y * d0, v, scale);
  }
  __device__ void add_rho(int s, int x, int y, float v) const {
    long long *h = pick4(s, R[0], R[1], R[2], R[3]);
    if (h) acc_fx(h, (uint64_t)x + (uint64_t)y * d0, v, scale);
  }
};
template <typename R>
struct LsAccOf;
template <>
struct LsAccOf<double> {
  using type = LsAccF64;
  static constexpr int limbs = 2;
};
template <>
struct LsAccOf<float> {
  using type = LsAccF32;
  static constexpr int limbs = 1;
};

// The same contributions into a workgroup's LDS window of W0 x W1 cells, the
// particle's cell (c1, c2) at (l1, l2): component q (J1..J3, then the charge of
// the first nq - 3 species) in elements [limbs q cells, limbs (q + 1) cells),
// limb l from l cells on.  A particle whose reach of two cells leaves the
// window adds to HBM.  The fixed-point value of each contribution is the HBM
// path's, so the sums are equal.
template <typename R>
struct LsAccWin {
  using G = typename LsAccOf<R>::type;
  long long *win;
  int cells, W0, W1, l1, l2, c1, c2, nq;
  G g;
  __device__ bool in() const { return l1 >= 2 && l1 <= W0 - 3 && l2 >= 2 && l2 <= W1 - 3; }
  __device__ void put(int q, int x, int y, R v) const {
    long long *e = win + LsAccOf<R>::limbs * q * cells + (x - c1 + l1) + (y - c2 + l2) * W0;
    if constexpr (std::is_same<R, double>::value) {
      long long h, l;
      fx_split(v, g.H, h, l);
      if (h != 0)
        __hip_atomic_fetch_add(e, h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      if (l != 0)
        __hip_atomic_fetch_add(e + cells, l, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    } else {
      const long long q1 = (long long)__float2int_rn(v * g.scale);
      if (q1 != 0)
        __hip_atomic_fetch_add(e, q1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  }
  __device__ void add(int c, int x, int y, R v) const {
    if (in()) put(c, x, y, v);
    else g.add(c, x, y, v);
  }
  __device__ void add_rho(int s, int x, int y, R v) const {
    if (in() && 3 + s < nq) put(3 + s, x, y, v);
    else g.add_rho(s, x, y, v);
  }
};

template <typename R>
__device__ inline R cicR(R d) {
  R a = (R)1 - fabs(d);
  return a > (R)0 ? a : (R)0;
}
template <typename R>
__device__ inline R center2dR(R sx0, R sx1, R sy0, R sy1) {
  return ((R)2 * sx1 * sy1 + sx0 * sy1 + sx1 * sy0 + (R)2 * sx0 * sy0) *
         ((R)1 / (R)6);
}
template <typename R>
__device__ inline R movement2dR(R sx0, R sx1, R sy0, R sy1) {
  return (sy1 - sy0) * (R)0.5 * (sx0 + sx1);
}

template <typename R>
__device__ inline R gatherR(const R *__restrict__ f, const Mesh &m, int c1,
                            int c2, R x1, R x2, int st) {
  if constexpr (std::is_same<R, double>::value)
    return gather2(f, m.dims[0], x1, x2, c1, c2, st);
  else
    return gatherf<2>(f, m, c1, c2, 0, x1, x2, 0.0f, st);
}

// ---------------------------------------------------------------------
// push + move + deposit of one live particle in bulk cell (c1, c2)
// ---------------------------------------------------------------------
template <typename R>
struct LsFields {
  const R *E1, *E2, *E3, *B1, *B2, *B3;
};

template <typename R, typename Acc>
__device__ __forceinline__ void logsph_push_one(const Mesh &m, const Species &sp,
                                                const LsParams &lp, R dt, int rho,
                                                const PtcView<R> &p, const LsFields<R> &F,
                                                const Acc &acc,
                                                unsigned long long *__restrict__ counters,
                                                uint64_t idx, int c1, int c2) {
  using M = LsMath<R>;
  const int d0 = m.dims[0];
  const R *E1f = F.E1, *E2f = F.E2, *E3f = F.E3, *B1f = F.B1, *B2f = F.B2, *B3f = F.B3;
  const uint32_t flag = p.flag[idx];
  const int s = ptc_species(flag);
  const R old_x1 = p.x1[idx], old_x2 = p.x2[idx], old_x3 = p.x3[idx];
  R p1 = p.p1[idx], p2 = p.p2[idx], p3 = p.p3[idx];
  if (p1 != p1 || p2 != p2 || p3 != p3) atomicAdd(&counters[CTR_NAN], 1ull);
  const R r = M::exp((R)lpos(m, 0, c1, (double)old_x1));
  const R q_over_m = (R)(dt * (R)0.5 * (R)sp.q[s] / (R)sp.m[s]);
  R gamma = sqrt((R)1 + p1 * p1 + p2 * p2 + p3 * p3);
  if (!(flag & FLAG_IGNORE_EM)) {
    R E1 = gatherR(E1f, m, c1, c2, old_x1, old_x2, ST_E1) * q_over_m;
    R E2 = gatherR(E2f, m, c1, c2, old_x1, old_x2, ST_E2) * q_over_m;
    R E3 = gatherR(E3f, m, c1, c2, old_x1, old_x2, ST_E3) * q_over_m;
    R B1 = gatherR(B1f, m, c1, c2, old_x1, old_x2, ST_B1) * q_over_m;
    R B2 = gatherR(B2f, m, c1, c2, old_x1, old_x2, ST_B2) * q_over_m;
    R B3 = gatherR(B3f, m, c1, c2, old_x1, old_x2, ST_B3) * q_over_m;
    if constexpr (std::is_same<R, double>::value)
      vay_push(p1, p2, p3, gamma, E1, E2, E3, B1, B2, B3);
    else
      vay_pushf(p1, p2, p3, gamma, E1, E2, E3, B1, B2, B3);
    // gravity (gravity.cuh:13-26)
    p1 -= dt * (R)lp.gravity * (R)sp.m[s] / (r * r * (R)fabs(sp.q[s]));
    gamma = sqrt((R)1 + p1 * p1 + p2 * p2 + p3 * p3);
    // sync_kill_perp (sync_cooling.cuh:41-68), leptons only
    if (lp.rad_cooling_on && s != 2) {
      B1 /= q_over_m;
      B2 /= q_over_m;
      B3 /= q_over_m;
      R B_sqr = B1 * B1 + B2 * B2 + B3 * B3;
      R pdotB = (p1 * B1 + p2 * B2 + p3 * B3);
      R k = (R)lp.rad_cooling_coef;
      R dp1 = -k * (p1 - B1 * pdotB / B_sqr);
      R dp2 = -k * (p2 - B2 * pdotB / B_sqr);
      R dp3 = -k * (p3 - B3 * pdotB / B_sqr);
      R fB = sqrt(B_sqr) / (R)lp.B0;
      p1 += dp1 * fB;
      p2 += dp2 * fB;
      p3 += dp3 * fB;
      R pp = sqrt(p1 * p1 + p2 * p2 + p3 * p3);
      gamma = sqrt((R)1 + pp * pp);
    }
    if (p.E) p.E[idx] = gamma;
  } else if (p.E) {
    gamma = p.E[idx];
  }

  // ---- move in Cartesian and back (ptc_updater_logsph.cu:163-230) ----
  const R w = p.w[idx];
  const R r1 = (R)lpos(m, 0, c1, (double)old_x1);
  const R exp_r1 = M::exp(r1);
  const R r2 = (R)lpos(m, 1, c2, (double)old_x2);
  R v1 = p1 / gamma, v2 = p2 / gamma, v3 = p3 / gamma;
  R v3_gr = v3 - beta_phi<R>(lp, exp_r1, r2);
  R s2, cs2;
  M::sincos(r2, s2, cs2);
  R np1, np2, np3, new_x1, new_x2, r3p;
  if constexpr (std::is_same<R, double>::value) {
    // FP64: the reference's expressions, operation for operation
    R s3, cs3;
    M::sincos(old_x3, s3, cs3);
    R x = exp_r1 * s2 * cs3;
    R y = exp_r1 * s2 * s3;
    R z = exp_r1 * cs2;
    {
      R a = v1, b = v2, cc = v3_gr;
      v1 = a * s2 * cs3 + b * cs2 * cs3 - cc * s3;
      v2 = a * s2 * s3 + b * cs2 * s3 + cc * cs3;
      v3_gr = a * cs2 - b * s2;
    }
    x += v1 * dt;
    y += v2 * dt;
    z += v3_gr * dt;
    R r1p = sqrt(x * x + y * y + z * z);
    const R r2p = M::acos(z / r1p);
    const R exp_r1p = r1p;
    r1p = M::log(r1p);
    r3p = M::atan2(y, x);
    {
      R ps2, pc2, ps3, pc3;
      M::sincos(r2p, ps2, pc2);
      M::sincos(r3p, ps3, pc3);
      R a = v1, b = v2, cc = v3_gr;
      v1 = a * ps2 * pc3 + b * ps2 * ps3 + cc * pc2;
      v2 = a * pc2 * pc3 + b * pc2 * ps3 - cc * ps2;
      v3_gr = -a * ps3 + b * pc3;
    }
    np1 = v1 * gamma;
    np2 = v2 * gamma;
    np3 = (v3_gr + beta_phi<R>(lp, exp_r1p, r2p)) * gamma;
    new_x1 = old_x1 + (r1p - r1) / (R)m.delta[0];
    new_x2 = old_x2 + (r2p - r2) / (R)m.delta[1];
  } else {
    // FP32: the same straight-line move, written in the particle's own
    // frame (azimuth measured from the particle, so phi's rounding never
    // enters) and for the changes of ln r, theta and phi directly: a step
    // moves a particle by ~1e-3 r, and taking ln|x| and the angles of the
    // moved Cartesian point, then subtracting the old ones, would leave
    // only a few correct bits of the change in FP32.  With d = v dt in the
    // local (r, theta, phi) components and the moved point
    // P = (r + d_r) r^ + d_th th^ + d_ph ph^:
    //   d ln r  = log1p((2 r d_r + |d|^2) / r^2) / 2
    //   d theta = atan2(rho cos th - Z sin th, rho sin th + Z cos th)
    //           = atan2(d_th + cos th t, r + d_r + sin th t),
    //             t = rho - X = d_ph^2 / (X + rho)
    //   d phi   = atan2(d_ph, X)
    // with X = (r + d_r) sin th + d_th cos th, Z = (r + d_r) cos th -
    // d_th sin th, rho = sqrt(X^2 + d_ph^2).  A move across the axis
    // (X <= 0) takes theta from atan2(rho, Z) directly.
    const float dr = v1 * dt, dth = v2 * dt, dph = v3_gr * dt;
    const float R1 = exp_r1 + dr;
    const float X = R1 * s2 + dth * cs2;
    const float Z = R1 * cs2 - dth * s2;
    const float rho = sqrtf(X * X + dph * dph);
    const float dlnr =
        0.5f * log1pf((2.0f * exp_r1 * dr + (dr * dr + dth * dth + dph * dph)) /
                      (exp_r1 * exp_r1));
    float r2p, dtheta;
    if (X > 0.0f) {
      const float t = dph * dph / (X + rho);
      dtheta = atan2f(dth + cs2 * t, R1 + s2 * t);
      r2p = r2 + dtheta;
    } else {
      r2p = atan2f(rho, Z);
      dtheta = r2p - r2;
    }
    const float dphi = atan2f(dph, X);
    const float exp_r1p = exp_r1 * expf(dlnr);
    // velocity: old local basis -> Cartesian (old azimuth 0) -> new basis
    const float a = v1 * s2 + v2 * cs2, b = v3_gr, cc = v1 * cs2 - v2 * s2;
    float ps2, pc2, ps3, pc3;
    sincosf(r2p, &ps2, &pc2);
    sincosf(dphi, &ps3, &pc3);
    v1 = a * ps2 * pc3 + b * ps2 * ps3 + cc * pc2;
    v2 = a * pc2 * pc3 + b * pc2 * ps3 - cc * ps2;
    v3_gr = -a * ps3 + b * pc3;
    np1 = v1 * gamma;
    np2 = v2 * gamma;
    np3 = (v3_gr + beta_phi<R>(lp, exp_r1p, r2p)) * gamma;
    new_x1 = old_x1 + dlnr / (float)m.delta[0];
    new_x2 = old_x2 + dtheta / (float)m.delta[1];
    // azimuth kept in (-pi, pi] like atan2's
    r3p = old_x3 + dphi;
    if (r3p > 3.14159265f) r3p -= 6.28318531f;
    else if (r3p <= -3.14159265f) r3p += 6.28318531f;
  }
  int dc1 = (int)floor(new_x1);
  int dc2 = (int)floor(new_x2);
  if (dc1 < -1 || dc1 > 1 || dc2 < -1 || dc2 > 1) {
    atomicAdd(&counters[CTR_MULTICELL], 1ull);
    p.cell[idx] = MAX_CELL;
    return;
  }
  new_x1 -= (R)dc1;
  new_x2 -= (R)dc2;
  if (lpos(m, 1, c2 + dc2, (double)new_x2) < 0.0) {
    dc2 += 1;
    new_x2 = (R)1 - new_x2;
    np2 = -np2;
    np3 = -np3;
  }
  if (lpos(m, 1, c2 + dc2, (double)new_x2) >= LS_PI) {
    dc2 -= 1;
    new_x2 = (R)1 - new_x2;
    np2 = -np2;
    np3 = -np3;
  }
  if constexpr (!std::is_same<R, double>::value) {
    // keep FP32 offsets inside [0, 1)
    if (new_x1 >= 1.0f) new_x1 = 0x1.fffffep-1f;
    if (new_x2 >= 1.0f) new_x2 = 0x1.fffffep-1f;
  }
  p.p1[idx] = np1;
  p.p2[idx] = np2;
  p.p3[idx] = np3;
  // what leaves the bulk is erased, what enters the outflow layer coasts on
  // (erase_ptc_in_guard_cells, kernels.cu:25-34; ptc_outflow,
  // ptc_updater_logsph.cu:397-412)
  const int n1 = c1 + dc1, n2 = c2 + dc2;
  const bool live = n1 >= m.guard[0] && n1 < d0 - m.guard[0] && n2 >= m.guard[1] &&
                    n2 < m.dims[1] - m.guard[1];
  p.cell[idx] = live ? (uint32_t)(n1 + n2 * d0) : MAX_CELL;
  if (live && !(flag & FLAG_IGNORE_EM) && n1 > d0 - lp.damping_length + 2)
    p.flag[idx] = flag | FLAG_IGNORE_EM;
  p.x1[idx] = new_x1;
  p.x2[idx] = new_x2;
  p.x3[idx] = r3p;

  if (flag & FLAG_IGNORE_CURRENT) return;
  const R weight = -(R)sp.q[s] * w;
  const int j0 = (dc2 == -1 ? -2 : -1), j1 = (dc2 == 1 ? 1 : 0);
  const int i0 = (dc1 == -1 ? -2 : -1), i1 = (dc1 == 1 ? 1 : 0);
  // the inner loop's trip count is fixed so that djy stays in registers
  R djy[3] = {(R)0, (R)0, (R)0};
#pragma unroll 1
  for (int j = j0; j <= j1; j++) {
    R sy0 = cicR<R>(-old_x2 + (R)j + (R)1);
    R sy1 = cicR<R>(-new_x2 + (R)(j + 1 - dc2));
    R djx = (R)0;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const int i = i0 + k;
      if (i > i1) break;
      R sx0 = cicR<R>(-old_x1 + (R)i + (R)1);
      R sx1 = cicR<R>(-new_x1 + (R)(i + 1 - dc1));
      const int x = i + c1, y = j + c2;
      djx += movement2dR<R>(sy0, sy1, sx0, sx1);
      acc.add(0, x + 1, y, weight * djx);
      djy[k] += movement2dR<R>(sx0, sx1, sy0, sy1);
      acc.add(1, x, y + 1, weight * djy[k]);
      R val2 = center2dR<R>(sx0, sx1, sy0, sy1);
      acc.add(2, x, y, -weight * v3_gr * val2);
      if (rho) {
        R s1 = sx1 * sy1;
        acc.add_rho(s, x, y, -weight * s1);
      }
    }
  }
}

// Shape of the update: a tile's cells per side, its halo, threads, slots per
// lane run, and the window in elements (a tile's window, or 40 KB).
constexpr uint32_t LS_DEV_TAIL = 4096;  // most workgroups behind the tiles, under a bound
constexpr int LS_T = 16, LS_HALO = 6, LS_NT = 512, LS_RUN = 4;
template <typename R, bool RHO>
constexpr int ls_win() {
  const int t = LsAccOf<R>::limbs * (RHO ? 5 : 3) * (LS_T + 2 * LS_HALO) * (LS_T + 2 * LS_HALO);
  return t > 5120 ? t : 5120;
}

// waves per SIMD asked of the compiler: two workgroups per CU (FP64: 126 VGPRs;
// with the 130 it takes unasked, one workgroup and 188 us for 131), except on
// FP64 charge steps, which do not fit in 128 VGPRs without spilling: compiled so,
// they gave wrong particles in all waves of a workgroup but the first, for a
// reason that was not found (the spill and its reloads read right), so that form
// is not built and the build refuses spills here (build.py)
template <typename R, bool RHO>
constexpr int ls_waves() {
  return std::is_same<R, double>::value && RHO ? 2 : 4;
}

// The log-spherical update with the current summed in LDS, on charge steps with
// the charge of two species.  The first nwork workgroups take the slots sorted
// by cell: one tile of 16 x 16 cells (or a share of its particles) each, with a
// window over the tile and a halo.  The others take the slots behind them
// (injected and created since, in cell order; every slot before the first
// sort), a slot a thread, with a window over the cells that the workgroup's
// particles occupy, if it fits.  The window is flushed once per element;
// particles outside it add to HBM (counted).  Integer sums: equal to the
// all-HBM path bit for bit.
// Bound by latency: long chains of transcendentals at four waves a SIMD.  In
// chunks of 1024 slots throughout, the cells of a chunk of a sparse cloud span
// several mesh rows and the windows did not fit: 800,000 particles at 7 per
// cell 130 us FP32 / 480 us FP64.  By tiles 52 / 107 us, and with the few slots
// behind them, a slot a thread in the same launch, 70 / 140 us (82 / 150 us in
// a launch of their own, 102 / 201 us at 4 slots a thread).  Halo 4: equal FP32,
// 3 % slower FP64; 256 threads equal / 9 % slower, 1024 9 / 13 % slower; runs
// of 16 slots 2 % slower than of 4 once the injected plasma has grown dense.
template <typename R, bool RHO>
__global__ void __launch_bounds__(LS_NT, (ls_waves<R, RHO>()))
    k_logsph_push(Mesh m, Species sp, LsParams lp, R dt, int nrho, PtcView<R> p, LsFields<R> F,
                  typename LsAccOf<R>::type acc, CellRuns cr, uint32_t nwork,
                  unsigned long long *__restrict__ counters, uint64_t n,
                  const unsigned long long *__restrict__ dn) {
  constexpr int LIMBS = LsAccOf<R>::limbs, W = LS_T + 2 * LS_HALO;
  constexpr uint32_t G = 64 / LS_RUN;
  __shared__ long long win[ls_win<R, RHO>()];
  __shared__ RunWalk<LS_T> walk;
  __shared__ uint32_t s_ref;
  __shared__ int s_lo[2], s_hi[2];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int d0 = m.dims[0];
  const int nq = 3 + (RHO ? (nrho < 2 ? nrho : 2) : 0);
  const bool tiled = blockIdx.x < nwork;  // uniform
  uint64_t base = 0;
  uint32_t cnt, lo = 0;
  int x0, y0, W0 = W, W1 = W;
  if (tiled) {
    uint32_t tile, part, parts, hi;
    if (!run_item(cr, blockIdx.x, tile, part, parts)) return;  // uniform
    int org[3];
    walk.open(m, cr, tile, part, parts, org, lo, hi);
    if (lo == hi) return;  // uniform
    cnt = hi - lo;
    x0 = org[0] - LS_HALO;
    y0 = org[1] - LS_HALO;
  } else {
    // The slots that no tile holds: one workgroup takes those sorted into the
    // guard rows below the tiles, the others those above them, which end where
    // the slots behind the sorted ones begin.  Each is judged by its own cell, as
    // a recorded step may be replayed on particles that were set since the sort.
    n = dev_n(n, dn);
    const bool lower = nwork > 0 && blockIdx.x == nwork;  // uniform
    const uint32_t first = lower ? nwork : nwork > 0 ? nwork + 1 : 0;
    uint64_t from = 0, groups = 1;
    if (lower) {
      const uint64_t end = cr.off[(uint64_t)m.guard[1] * cr.nt[0]];
      n = end < n ? end : n;
    } else {
      if (nwork > 0) from = cr.off[(uint64_t)(m.dims[1] - m.guard[1]) * cr.nt[0]];
      groups = gridDim.x - first;
    }
    if (from >= n) return;  // uniform
    // whole slots a thread: one, unless the grid is capped
    const uint64_t per = groups * LS_NT;
    const uint64_t chunk = (n - from + per - 1) / per * LS_NT;
    base = from + (uint64_t)(blockIdx.x - first) * chunk;
    if (base >= n) return;  // uniform: past the count
    cnt = (uint32_t)(n - base < chunk ? n - base : chunk);
    if (tid < 2) {
      s_lo[tid] = INT_MAX;
      s_hi[tid] = INT_MIN;
    }
    if (tid == 0) s_ref = MAX_CELL;
    __syncthreads();
    // the occupied cells' extent, about one of them
    uint32_t low = MAX_CELL;
    for (uint32_t i = tid; i < cnt; i += LS_NT) {
      const uint32_t c = p.cell[base + i];
      low = c < low ? c : low;
    }
    if (low != MAX_CELL) atomicMin(&s_ref, low);
    __syncthreads();
    if (s_ref == MAX_CELL) return;  // no live particle
    const int r1 = (int)(s_ref % (uint32_t)d0), r2 = (int)(s_ref / (uint32_t)d0);
    for (uint32_t i = tid; i < cnt; i += LS_NT) {
      const uint32_t c = p.cell[base + i];
      if (c == MAX_CELL) continue;
      const int a = (int)(c % (uint32_t)d0) - r1, b = (int)(c / (uint32_t)d0) - r2;
      atomicMin(&s_lo[0], a);
      atomicMax(&s_hi[0], a);
      atomicMin(&s_lo[1], b);
      atomicMax(&s_hi[1], b);
    }
    __syncthreads();
    // the deposit reaches cells -2 .. +2 of a particle's cell
    W0 = s_hi[0] - s_lo[0] + 5;
    W1 = s_hi[1] - s_lo[1] + 5;
    x0 = r1 + s_lo[0] - 2;
    y0 = r2 + s_lo[1] - 2;
    if ((int64_t)W0 * W1 * LIMBS * nq > ls_win<R, RHO>()) W0 = W1 = 0;
  }
  const int cells = W0 * W1;
  for (int e = tid; e < LIMBS * nq * cells; e += LS_NT) win[e] = 0;
  __syncthreads();
  // lanes take runs of consecutive slots spread over the share, so that a
  // wave's atomics fall on several cells
  const uint32_t seg = ((cnt + G - 1) / G + LS_RUN - 1) / LS_RUN * LS_RUN;
  unsigned far = 0;
#pragma unroll 1
  for (uint32_t k = wv * LS_RUN; k < seg; k += (LS_NT / 64) * LS_RUN) {
    const uint32_t kk = k + (uint32_t)(lane % LS_RUN), q = (uint32_t)(lane / LS_RUN) * seg + kk;
    if (kk >= seg || q >= cnt) continue;
    const uint64_t idx = tiled ? (uint64_t)walk.slot(lo + q) : base + q;
    const uint32_t c = p.cell[idx];
    if (c == MAX_CELL) continue;
    const int c1 = (int)(c % (uint32_t)d0), c2 = (int)(c / (uint32_t)d0);
    if (!(c1 >= m.guard[0] && c1 < d0 - m.guard[0] && c2 >= m.guard[1] &&
          c2 < m.dims[1] - m.guard[1])) {
      p.cell[idx] = MAX_CELL;  // particles outside the bulk are erased
      continue;
    }
    const LsAccWin<R> w{win, cells, W0, W1, c1 - x0, c2 - y0, c1, c2, nq, acc};
    if (!w.in()) far++;
    logsph_push_one<R>(m, sp, lp, dt, RHO, p, F, w, counters, idx, c1, c2);
  }
  if (far) atomicAdd(&counters[CTR_GLOBAL_DEP], (unsigned long long)far);
  if (cells == 0) return;  // uniform
  __syncthreads();
  // e / W0 by the reciprocal: exact, cells W0 < 2^32
  const uint32_t inv = 0xffffffffu / (uint32_t)W0 + 1u;
  for (int e = tid; e < cells; e += LS_NT) {
    const int y = (int)__umulhi((uint32_t)e, inv), x = e - y * W0;
    const int64_t o = (int64_t)(x0 + x) + (int64_t)(y0 + y) * d0;
#pragma unroll
    for (int q = 0; q < (RHO ? 5 : 3); q++) {
      if (q >= nq) break;
#pragma unroll
      for (int l = 0; l < LIMBS; l++) {
        const long long v = win[(LIMBS * q + l) * cells + e];
        if (v != 0)
          __hip_atomic_fetch_add(acc.at(q, l) + o, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
}

// the rows on either side of the two axis edges
__device__ __forceinline__ bool axis_row(const Mesh &m, int j) {
  const int g = m.guard[1], jl = m.dims[1] - m.guard[1];
  return j == g - 1 || j == g || j == jl - 1 || j == jl;
}

// process_j (ptc_updater_logsph.cu:284-299): J1,J2 *= (D0 D1/dt)/A,
// J3 and Rho /= dV over every cell; clears the accumulators.  With no smoothing
// pass to follow, J3's axis rows are set to zero here (axis_rho_lower/upper,
// ptc_updater_logsph.cu:414-438).  One pass for the current and the charge of
// every species: 512 x 512 took 6.1 + 4 x 4.9 us in five launches, 5.4 us here
// (the charge written on charge steps and the step after).
template <typename T>
struct LsProcess {
  long long *jh[3], *jl[3], *rh[4], *rl[4];
  T *J[3], *Rho[4];
  int ns;  // charge arrays to write
};
template <typename T>
__global__ void k_logsph_process(Mesh m, LsCoef cf, double wj, int H, int limbs, LsProcess<T> a,
                                 int axis, uint64_t n) {
  uint64_t o = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (o >= n) return;
  auto take = [&](long long *hi, long long *lo) {
    const long long h = hi[o];
    double v;
    if (limbs == 2) {
      const long long l = lo[o];
      v = fx_value(h, l, H);
      if (l != 0) lo[o] = 0;
    } else {
      v = ldexp((double)h, -H);
    }
    if (h != 0) hi[o] = 0;
    return v;
  };
  const double dv = cf.a[LS_DV][o];
  a.J[0][o] = (T)(take(a.jh[0], a.jl[0]) * (wj / cf.a[LS_A1E][o]));
  a.J[1][o] = (T)(take(a.jh[1], a.jl[1]) * (wj / cf.a[LS_A2E][o]));
  const T j3 = (T)(take(a.jh[2], a.jl[2]) / dv);
  a.J[2][o] = axis && axis_row(m, (int)(o / (uint32_t)m.dims[0])) ? (T)0 : j3;
#pragma unroll
  for (int s = 0; s < 4; s++)
    if (s < a.ns) a.Rho[s][o] = (T)(take(a.rh[s], a.rl[s]) / dv);
}

// filter_current_logsph (ptc_updater_logsph.cu:616-666), one rank: all
// four boundary offsets collapse at the domain edge.
template <typename T>
__global__ void k_logsph_filter(Mesh m, const T *__restrict__ j,
                                T *__restrict__ tmp,
                                const double *__restrict__ A) {
  const int N0 = m.dims[0] - 2 * m.guard[0], N1 = m.dims[1] - 2 * m.guard[1];
  uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (uint64_t)N0 * N1) return;
  const int d0 = m.dims[0];
  int n1 = m.guard[0] + (int)(t % N0), n2 = m.guard[1] + (int)(t / N0);
  uint64_t o = (uint64_t)n1 + (uint64_t)n2 * d0;
  uint64_t drp = n1 == m.dims[0] - m.guard[0] - 1 ? 0 : 1;
  uint64_t drm = n1 == m.guard[0] ? 0 : 1;
  uint64_t dtp = n2 == m.dims[1] - m.guard[1] - 1 ? 0 : (uint64_t)d0;
  uint64_t dtm = n2 == m.guard[1] ? 0 : (uint64_t)d0;
  T r = (T)0.25 * j[o] * (T)A[o];
  r += (T)0.125 * j[o + drp] * (T)A[o + drp];
  r += (T)0.125 * j[o - drm] * (T)A[o - drm];
  r += (T)0.125 * j[o + dtp] * (T)A[o + dtp];
  r += (T)0.125 * j[o - dtm] * (T)A[o - dtm];
  r += (T)0.0625 * j[o + drp + dtp] * (T)A[o + drp + dtp];
  r += (T)0.0625 * j[o - drm + dtp] * (T)A[o - drm + dtp];
  r += (T)0.0625 * j[o + drp - dtm] * (T)A[o + drp - dtm];
  r += (T)0.0625 * j[o - drm - dtm] * (T)A[o - drm - dtm];
  r /= (T)A[o];
  tmp[o] = r;
}

// axis_rho_lower/upper (ptc_updater_logsph.cu:414-438)
template <typename T>
__global__ void k_logsph_axis_j3(Mesh m, T *J3) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m.dims[0]) return;
  const int d0 = m.dims[0], g = m.guard[1], jl = m.dims[1] - m.guard[1];
  J3[i + (uint64_t)(g - 1) * d0] = (T)0;
  J3[i + (uint64_t)g * d0] = (T)0;
  J3[i + (uint64_t)jl * d0] = (T)0;
  J3[i + (uint64_t)(jl - 1) * d0] = (T)0;
}

// ---------------------------------------------------------------------
// field solver (field_solver_logsph.cu:28-345), alpha_gr = 1
// ---------------------------------------------------------------------
#define F2(a, i, j) (a)[(uint64_t)(i) + (uint64_t)(j) * d0]
#define C2(k, i, j) ((T)cf.a[k][(uint64_t)(i) + (uint64_t)(j) * d0])

// Thread t's cell: the bulk's nb cells in order, then the bulk's columns of the
// row below it (theta = 0), whose rules need no row that the bulk writes and
// run in the same launch.
template <typename T>
__device__ inline void bulk_ij(const Mesh &m, uint64_t t, uint64_t nb, int &i, int &j) {
  const uint32_t N0 = (uint32_t)(m.dims[0] - 2 * m.guard[0]);
  const bool axis = t >= nb;
  const uint32_t u = (uint32_t)(axis ? t - nb : t);
  i = m.guard[0] + (int)(u % N0);
  j = axis ? m.guard[1] - 1 : m.guard[1] + (int)(u / N0);
}

template <typename T>
__global__ void k_logsph_update_b(Mesh m, LsCoef cf, LsParams lp,
                                  FieldSet<T> f, T dt, uint64_t nb) {
  uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int i, j;
  bulk_ij<T>(m, t, nb, i, j);
  if (t >= nb + (uint64_t)(m.dims[0] - 2 * m.guard[0])) return;
  const int d0 = m.dims[0];
  const uint64_t o = (uint64_t)i + (uint64_t)j * d0;
  if (t >= nb) {  // (field_solver_logsph.cu:177-184)
    f.B[1][o] = f.Bbg[1][o];
    return;
  }
  const T *E1 = f.E[0], *E2 = f.E[1], *E3 = f.E[2];
  const T *G1 = f.Ebg[0], *G2 = f.Ebg[1], *G3 = f.Ebg[2];
  const T *H1 = f.Bbg[0], *H2 = f.Bbg[1];
  const double r1 = apt_exp(spos(m, 0, i, 1));
  const double r0 = apt_exp(spos(m, 0, i - 1, 1));
  const double r = apt_exp(spos(m, 0, i, 0));
  const double th0 = spos(m, 1, j, 0);
  const T b_r1 = (T)beta_phi<double>(lp, r1, th0);
  const T b_r0 = (T)beta_phi<double>(lp, r0, th0);
  const T b_m = (T)beta_phi<double>(lp, r, spos(m, 1, j - 1, 1));
  const T b_c = (T)beta_phi<double>(lp, r, spos(m, 1, j, 1));
  f.B[0][o] += -dt *
               ((F2(E3, i, j) - F2(G3, i, j)) * C2(LS_L3E, i, j) -
                (F2(E3, i, j - 1) - F2(G3, i, j - 1)) * C2(LS_L3E, i, j - 1)) /
               C2(LS_A1B, i, j);
  f.B[1][o] += -dt *
               ((F2(E3, i - 1, j) - F2(G3, i - 1, j)) * C2(LS_L3E, i - 1, j) -
                (F2(E3, i, j) - F2(G3, i, j)) * C2(LS_L3E, i, j)) /
               C2(LS_A2B, i, j);
  f.B[2][o] += -dt * ((((F2(E2, i, j) - F2(G2, i, j)) + F2(H1, i, j) * b_r1) *
                           C2(LS_L2E, i, j) -
                       ((F2(E2, i - 1, j) - F2(G2, i - 1, j)) +
                        F2(H1, i - 1, j) * b_r0) *
                           C2(LS_L2E, i - 1, j) +
                       ((F2(E1, i, j - 1) - F2(G1, i, j - 1)) -
                        F2(H2, i, j - 1) * b_m) *
                           C2(LS_L1E, i, j - 1) -
                       ((F2(E1, i, j) - F2(G1, i, j)) - F2(H2, i, j) * b_c) *
                           C2(LS_L1E, i, j)) /
                      C2(LS_A3B, i, j));
}

template <typename T>
__global__ void k_logsph_update_e(Mesh m, LsCoef cf, FieldSet<T> f, T dt,
                                  uint64_t nb) {
  uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int i, j;
  bulk_ij<T>(m, t, nb, i, j);
  if (t >= nb + (uint64_t)(m.dims[0] - 2 * m.guard[0])) return;
  const int d0 = m.dims[0];
  const uint64_t o = (uint64_t)i + (uint64_t)j * d0;
  const T *B1 = f.B[0], *B2 = f.B[1], *B3 = f.B[2];
  const T *H1 = f.Bbg[0], *H2 = f.Bbg[1], *H3 = f.Bbg[2];
  const T D1 = (T)m.delta[1];
  if (t >= nb) {  // (field_solver_logsph.cu:100-113)
    const int g = m.guard[1];
    const T r0 = (T)apt_exp(spos(m, 0, i, 0));
    f.E[2][o] = f.Ebg[2][o];
    f.E[0][o] += dt * ((T)4.0 * (F2(B3, i, g) - F2(H3, i, g)) / (D1 * r0) - f.J[0][o]);
    return;
  }
  if (fabs(spos(m, 1, j, 1) - LS_PI) < 1.0e-5) {
    const T r0 = (T)apt_exp(spos(m, 0, i, 0));
    f.E[0][o] += dt * ((T)(-4.0) * (B3[o] - H3[o]) / (D1 * r0) - f.J[0][o]);
  } else {
    f.E[0][o] += dt * (((F2(B3, i, j + 1) - F2(H3, i, j + 1)) *
                            C2(LS_L3B, i, j + 1) -
                        (F2(B3, i, j) - F2(H3, i, j)) * C2(LS_L3B, i, j)) /
                           C2(LS_A1E, i, j) -
                       f.J[0][o]);
  }
  f.E[1][o] += dt * (((F2(B3, i, j) - F2(H3, i, j)) * C2(LS_L3B, i, j) -
                      (F2(B3, i + 1, j) - F2(H3, i + 1, j)) *
                          C2(LS_L3B, i + 1, j)) /
                         C2(LS_A2E, i, j) -
                     f.J[1][o]);
  f.E[2][o] += dt * (((F2(B2, i + 1, j) - F2(H2, i + 1, j)) *
                          C2(LS_L2B, i + 1, j) -
                      (F2(B2, i, j) - F2(H2, i, j)) * C2(LS_L2B, i, j) +
                      (F2(B1, i, j) - F2(H1, i, j)) * C2(LS_L1B, i, j) -
                      (F2(B1, i, j + 1) - F2(H1, i, j + 1)) *
                          C2(LS_L1B, i, j + 1)) /
                         C2(LS_A3E, i, j) -
                     f.J[2][o]);
}

// compute_EdotB_2d (cuda/sim_data.cu:50-79): E and B interpolated to the
// cell centre (stagger 0b000) with interpolate2d's neighbour offsets, then
// EdotB += delta (E.B) / |B| with delta = 1.0f / data_interval
template <typename T>
__device__ inline T centre2d(const T *a, uint64_t o, int st, int d0) {
  const int64_t im = (st & 1) ? -1 : 0, jm = (st & 2) ? -(int64_t)d0 : 0;
  const T *p = a + o;
  const T f1 = (T)0.5 * (p[0] + p[jm]);
  const T f0 = (T)0.5 * (p[im] + p[im + jm]);
  return (T)0.5 * (f1 + f0);
}

// the divergences and E.B of the updated fields, one read of them
template <typename T>
__global__ void k_logsph_divs(Mesh m, LsCoef cf, FieldSet<T> f, T delta, uint64_t nb) {
  uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int i, j;
  bulk_ij<T>(m, t, nb, i, j);
  if (t >= nb + (uint64_t)(m.dims[0] - 2 * m.guard[0])) return;
  const int d0 = m.dims[0];
  const uint64_t o = (uint64_t)i + (uint64_t)j * d0;
  const T *E1 = f.E[0], *E2 = f.E[1], *B1 = f.B[0], *B2 = f.B[1];
  const T *G1 = f.Ebg[0], *G2 = f.Ebg[1], *H1 = f.Bbg[0], *H2 = f.Bbg[1];
  if (t >= nb) {
    const int g = m.guard[1];
    f.divE[o] = ((F2(E1, i + 1, g - 1) - F2(G1, i + 1, g - 1)) * C2(LS_A1E, i + 1, g - 1) -
                 (F2(E1, i, g - 1) - F2(G1, i, g - 1)) * C2(LS_A1E, i, g - 1) +
                 (T)2.0 * (F2(E2, i, g) - F2(G2, i, g)) * C2(LS_A2E, i, g)) /
                (C2(LS_DV, i, g - 1) * (T)m.delta[0] * (T)m.delta[1]);
    return;
  }
  const T den = C2(LS_DV, i, j) * (T)m.delta[0] * (T)m.delta[1];
  const double size1 = m.delta[1] * (double)(m.dims[1] - 2 * m.guard[1]);
  if (spos(m, 0, i, 1) > m.delta[0]) {
    if (fabs(spos(m, 1, j, 1) - size1 + m.lower[1]) < 1.0e-5)
      f.divE[o] = ((F2(E1, i + 1, j) - F2(G1, i + 1, j)) * C2(LS_A1E, i + 1, j) -
                   (F2(E1, i, j) - F2(G1, i, j)) * C2(LS_A1E, i, j) -
                   (T)2.0 * (F2(E2, i, j) - F2(G2, i, j)) * C2(LS_A2E, i, j)) /
                  den;
    else
      f.divE[o] = ((F2(E1, i + 1, j) - F2(G1, i + 1, j)) * C2(LS_A1E, i + 1, j) -
                   (F2(E1, i, j) - F2(G1, i, j)) * C2(LS_A1E, i, j) +
                   (F2(E2, i, j + 1) - F2(G2, i, j + 1)) * C2(LS_A2E, i, j + 1) -
                   (F2(E2, i, j) - F2(G2, i, j)) * C2(LS_A2E, i, j)) /
                  den;
  }
  f.divB[o] = ((F2(B1, i, j) - F2(H1, i, j)) * C2(LS_A1B, i, j) -
               (F2(B1, i - 1, j) - F2(H1, i - 1, j)) * C2(LS_A1B, i - 1, j) +
               (F2(B2, i, j) - F2(H2, i, j)) * C2(LS_A2B, i, j) -
               (F2(B2, i, j - 1) - F2(H2, i, j - 1)) * C2(LS_A2B, i, j - 1)) /
              den;
  if (!f.EdotB) return;
  const T e1 = centre2d<T>(f.E[0], o, 0b110, d0);
  const T e2 = centre2d<T>(f.E[1], o, 0b101, d0);
  const T e3 = centre2d<T>(f.E[2], o, 0b011, d0);
  const T b1 = centre2d<T>(f.B[0], o, 0b001, d0);
  const T b2 = centre2d<T>(f.B[1], o, 0b010, d0);
  const T b3 = centre2d<T>(f.B[2], o, 0b100, d0);
  f.EdotB[o] += delta * (e1 * b1 + e2 * b2 + e3 * b3) / sqrt(b1 * b1 + b2 * b2 + b3 * b3);
}

// stellar_boundary (field_solver_logsph.cu:252-275): i < guard0, every j
template <typename T>
__device__ inline void stellar_cell(const Mesh &m, const LsParams &lp, const FieldSet<T> &f,
                                    double omega, int i, int j) {
  const uint64_t o = (uint64_t)i + (uint64_t)j * m.dims[0];
  const double theta_s = spos(m, 1, j, 1), theta = spos(m, 1, j, 0);
  const double r_s = apt_exp(spos(m, 0, i, 1)), r = apt_exp(spos(m, 0, i, 0));
  const double omega_LT = 0.4 * omega * lp.compactness;
  f.B[0][o] = f.Bbg[0][o];
  f.B[1][o] = f.Bbg[1][o];
  f.B[2][o] = f.Bbg[2][o];
  if constexpr (std::is_same<T, double>::value) {
    f.E[1][o] = -(omega - omega_LT) * apt_sin(theta) * f.Bbg[0][o] / r_s / r_s +
                f.Ebg[1][o];
    f.E[0][o] = (omega - omega_LT) * apt_sin(theta_s) * f.Bbg[1][o] / r / r +
                f.Ebg[0][o];
  } else {
    f.E[1][o] = (T)(-(omega - omega_LT) * apt_sin(theta) * (double)f.Bbg[0][o] /
                    r_s / r_s) +
                f.Ebg[1][o];
    f.E[0][o] = (T)((omega - omega_LT) * apt_sin(theta_s) *
                    (double)f.Bbg[1][o] / r / r) +
                f.Ebg[0][o];
  }
}

// outflow_boundary_sph (field_solver_logsph.cu:322-345): the outermost
// damping_length columns
template <typename T>
__device__ inline void damping_cell(const Mesh &m, const LsParams &lp, const FieldSet<T> &f,
                                    int i, int j) {
  const int L = lp.damping_length;
  const uint64_t o = (uint64_t)i + (uint64_t)j * m.dims[0];
  const double x = (double)(i - (m.dims[0] - L)) / L;
  const T lambda = (T)(1.0 - lp.damping_coef * (x * x));
  for (int c = 0; c < 3; c++)
    f.E[c][o] = lambda * (f.E[c][o] - f.Ebg[c][o]) + f.Ebg[c][o];
  f.B[2][o] = lambda * (f.B[2][o] - f.Bbg[2][o]) + f.Bbg[2][o];
}

// axis_boundary_lower / upper (field_solver_logsph.cu:277-320) of column i
template <typename T>
__device__ inline void axis_lower(const Mesh &m, const FieldSet<T> &f, int i) {
  T *E2 = f.E[1], *E3 = f.E[2], *B1 = f.B[0], *B2 = f.B[1], *B3 = f.B[2];
  const T *G2 = f.Ebg[1], *G3 = f.Ebg[2], *H1 = f.Bbg[0], *H2 = f.Bbg[1], *H3 = f.Bbg[2];
  const uint64_t a = (uint64_t)i + (uint64_t)(m.guard[1] - 1) * m.dims[0], b = a + m.dims[0];
  E3[a] = G3[a];
  E2[a] = -(E2[b] - G2[b]) + G2[a];
  B3[a] = H3[a];
  B3[b] = H3[b];
  B2[a] = H2[a];
  B1[a] = (B1[b] - H1[b]) + H1[a];
}
template <typename T>
__device__ inline void axis_upper(const Mesh &m, const FieldSet<T> &f, int i) {
  T *E2 = f.E[1], *E3 = f.E[2], *B1 = f.B[0], *B2 = f.B[1], *B3 = f.B[2];
  const T *G2 = f.Ebg[1], *G3 = f.Ebg[2], *H1 = f.Bbg[0], *H2 = f.Bbg[1], *H3 = f.Bbg[2];
  const uint64_t a = (uint64_t)i + (uint64_t)(m.dims[1] - m.guard[1] - 1) * m.dims[0],
                 b = a + m.dims[0];
  E3[a] = G3[a];
  E2[b] = -(E2[a] - G2[a]) + G2[b];
  B3[b] = H3[b];
  B3[a] = H3[a];
  B2[a] = H2[a];
  B1[b] = (B1[a] - H1[a]) + H1[b];
}

// The boundary rules in one launch (512 x 512: 16 us in four, 9.6 in one).  A
// column's axis rows go through every rule, in order, in one thread; the star's
// and the outflow layer's other cells have a thread each.
template <typename T>
__global__ void k_logsph_boundary(Mesh m, LsParams lp, FieldSet<T> f, double omega) {
  const int d0 = m.dims[0], d1 = m.dims[1], g0 = m.guard[0], L = lp.damping_length;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < d0) {
    const int i = (int)t;
    int last = -1;
    const int rows[4] = {m.guard[1] - 1, m.guard[1], d1 - m.guard[1] - 1, d1 - m.guard[1]};
    for (int k = 0; k < 4; k++) {
      if (rows[k] <= last) continue;  // a mesh of one or two rows
      last = rows[k];
      if (i < g0) stellar_cell(m, lp, f, omega, i, rows[k]);
      if (i >= d0 - L) damping_cell(m, lp, f, i, rows[k]);
    }
    axis_lower(m, f, i);
    axis_upper(m, f, i);
    return;
  }
  const int per = g0 + L;  // the other cells, a row at a time
  if (per == 0) return;
  const int64_t u = t - d0;
  const int j = (int)(u / per), q = (int)(u - (int64_t)j * per);
  if (j >= d1 || axis_row(m, j)) return;
  if (q < g0) {
    stellar_cell(m, lp, f, omega, q, j);
    if (q >= d0 - L) damping_cell(m, lp, f, q, j);
  } else {
    const int i = d0 - L + (q - g0);
    if (i >= g0) damping_cell(m, lp, f, i, j);
  }
}
#undef F2
#undef C2

// ---------------------------------------------------------------------
// injection (ptc_updater_logsph.cu:301-395, 440-493)
// ---------------------------------------------------------------------
// measure_surface_density: every electron and ion in the radial cells from
// the injection cell - 1 adds its weight, spread 1-4-6-4-1 / 16 over the
// neighbouring rows, to its species' surface density.  A workgroup reads a
// chunk of consecutive slots (16 B a lane) and leaves at once if nothing in it
// is near the surface.  Otherwise it adds the three distinct taps, in their two
// limbs, to LDS sums per row and species over the rows from the chunk's lowest
// on (a chunk of sorted or injected slots covers few rows; rows past the window
// go to HBM), and adds each sum to its rows at the end: integer sums, any order.
// Wave sums over one (row, species) at a time took 40 us at 512 rows and
// 850,000 slots, nearly all in the unsorted slots at the end; 22 us here.
constexpr int SURF_E = 8, SURF_ROWS = 192;
template <typename R>
__global__ void __launch_bounds__(256)
    k_logsph_surface(Mesh m, const uint32_t *__restrict__ cell, const uint32_t *__restrict__ flag,
                     const R *__restrict__ w, uint64_t n, long long *surf, int Hs,
                     const unsigned long long *__restrict__ dn) {
  __shared__ unsigned long long s_sum[2][6][SURF_ROWS];  // species, tap and limb, row
  __shared__ int s_row;
  n = dev_n(n, dn);
  const int d0 = m.dims[0], g0 = m.guard[0], g1 = m.guard[1], tid = threadIdx.x;
  const int N1 = m.dims[1] - 2 * g1;
  const int inject_cell = g0 + 2, sum_cells = 3;
  const double cw[3] = {1.0, 4.0, 6.0};
  // value of tap v, limb l of row r and species s added to its five rows
  auto spread = [&](int s, int r, int vl, unsigned long long v) {
    unsigned long long *to = (unsigned long long *)surf + (s == 0 ? 0 : 2 * N1) + (vl & 1) * N1;
    for (int t = vl >> 1; t < 5; t += 4 - 2 * (vl >> 1)) {
      int q = r - 2 + t;
      q = q < 0 ? 0 : (q > N1 - 1 ? N1 - 1 : q);
      __hip_atomic_fetch_add(to + q, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (vl >= 4) break;  // the middle tap
    }
  };
  const uint64_t chunk = 256 * SURF_E, stride = (uint64_t)gridDim.x * chunk;
  for (uint64_t b = (uint64_t)blockIdx.x * chunk; b < n; b += stride) {
    uint32_t c[SURF_E];
    const uint64_t i0 = b + (uint64_t)tid * SURF_E;
    if (i0 + SURF_E <= n) {
      const uint4 *v = reinterpret_cast<const uint4 *>(cell + i0);
#pragma unroll
      for (int k = 0; k < SURF_E / 4; k++) {
        const uint4 u = v[k];
        c[4 * k] = u.x;
        c[4 * k + 1] = u.y;
        c[4 * k + 2] = u.z;
        c[4 * k + 3] = u.w;
      }
    } else {
#pragma unroll
      for (int k = 0; k < SURF_E; k++) c[k] = i0 + k < n ? cell[i0 + k] : MAX_CELL;
    }
    unsigned near = 0;
    int low = INT_MAX;
#pragma unroll
    for (int k = 0; k < SURF_E; k++) {
      if (c[k] == MAX_CELL) continue;
      const int c2 = (int)(c[k] / (uint32_t)d0), c1 = (int)(c[k] - (uint32_t)c2 * (uint32_t)d0);
      if (c1 < inject_cell - 1 || c1 > inject_cell - 1 + sum_cells) continue;
      near |= 1u << k;
      low = c2 < low ? c2 : low;
      c[k] = (uint32_t)c2;
    }
    if (!__syncthreads_or((int)near)) continue;
    if (tid == 0) s_row = INT_MAX;
    for (int e = tid; e < 12 * SURF_ROWS; e += 256) (&s_sum[0][0][0])[e] = 0;
    __syncthreads();
    if (near) atomicMin(&s_row, low);
    __syncthreads();
    const int row0 = s_row;
#pragma unroll
    for (int k = 0; k < SURF_E; k++) {
      if (!(near >> k & 1)) continue;
      const int s = ptc_species(flag[i0 + k]);
      if (s != 0 && s != 2) continue;
      const double wp = (double)w[i0 + k];
      const int r = (int)c[k] - row0;
#pragma unroll
      for (int v = 0; v < 3; v++) {
        long long hl[2];
        fx_split(cw[v] * wp / (double)sum_cells / 16.0, Hs, hl[0], hl[1]);
#pragma unroll
        for (int l = 0; l < 2; l++) {
          if (hl[l] == 0) continue;
          if (r < SURF_ROWS)
            __hip_atomic_fetch_add(&s_sum[s >> 1][2 * v + l][r], (unsigned long long)hl[l],
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          else
            spread(s, (int)c[k] - g1, 2 * v + l, (unsigned long long)hl[l]);
        }
      }
    }
    __syncthreads();
    for (int e = tid; e < 12 * SURF_ROWS; e += 256) {
      const unsigned long long v = (&s_sum[0][0][0])[e];
      if (v == 0) continue;
      const int r = e % SURF_ROWS, vl = e / SURF_ROWS % 6, s = e / (6 * SURF_ROWS) * 2;
      spread(s, row0 + r - g1, vl, v);
    }
    __syncthreads();  // the sums are cleared for the next chunk
  }
}

template <typename R>
__global__ void k_logsph_inject(Mesh m, LsParams lp, PtcView<R> p,
                                uint64_t base, int inj, double p1, double w,
                                double q_e, uint64_t seed, uint32_t epoch,
                                int Hs, uint64_t id_base,
                                const long long *__restrict__ surf,
                                const unsigned long long *__restrict__ dc, uint64_t cap) {
  const int g0 = m.guard[0], g1 = m.guard[1], d0 = m.dims[0];
  const int N1 = m.dims[1] - 2 * g1;
  const int rows = N1 - 2;
  uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (uint64_t)rows * inj) return;
  if (dc) {  // device-count mode: base, ids and epoch from the device
    base = dc[DC_NUM];
    id_base = dc[DC_ID];
    epoch = (uint32_t)dc[DC_INJ_EPOCH];
  }
  const int i = g1 + 1 + (int)(t / inj), nn = (int)(t % inj);
  const uint64_t off = base + (uint64_t)(i - g1 - 1) * inj * 2 + 2 * (uint64_t)nn;
  if (dc && off + 1 >= cap) return;  // past the capacity: dropped, counted
  const long long *seh = surf, *sel = surf + N1, *sph = surf + 2 * N1,
                  *spl = surf + 3 * N1;
  const double de = fx_value(seh[i - g1], sel[i - g1], Hs);
  const double dp = fx_value(sph[i - g1], spl[i - g1], Hs);
  const double dens = de > dp ? de : dp;
  const double sgate = (1.0 / m.delta[1]) * (1.0 / m.delta[1]);
  const double sin_theta = apt_sin(lpos(m, 1, i, 0.5));
  const bool gated = q_e * dens > 1.5 * sgate * sin_theta;
  for (int s = 0; s < 2; s++) {
    p.cell[off + s] = MAX_CELL;
    if (p.id) p.id[off + s] = id_base + (off + s - base);
  }
  if (gated) return;
  double u0, u1;
  uniform2(seed, ((uint64_t)epoch << 32) | (uint32_t)i, (uint32_t)nn, 4, u0, u1);
  const double x2 = 1.0 - u0;
  const double theta = lpos(m, 1, i, x2);
  double st, ct;
  apt_sincos(theta, st, ct);
  const double vphi = 0.0;
  const double w_ptc = w * st;
  const double gamma = sqrt(1.0 + p1 * p1 + vphi * vphi);
  const double sg = (double)((0.0 < ct) - (ct < 0.0));
  const uint32_t fl = FLAG_PRIMARY | (u1 < lp.track_percent ? FLAG_TRACKED : 0u);
  for (int s = 0; s < 2; s++) {
    const uint64_t o = off + s;
    R x2r = (R)x2;
    if constexpr (!std::is_same<R, double>::value)
      if (x2r >= 1.0f) x2r = 0x1.fffffep-1f;
    p.x1[o] = (R)0.5;
    p.x2[o] = x2r;
    p.x3[o] = (R)0;
    p.p1[o] = (R)(p1 * 2.0 * fabs(ct));
    p.p2[o] = (R)(p1 * st * sg);
    p.p3[o] = (R)vphi;
    if (p.E) p.E[o] = (R)gamma;
    p.w[o] = (R)w_ptc;
    const uint32_t type = s == 0 ? 0u : (lp.inject_ions ? 2u : 1u);
    p.flag[o] = fl | (type << 29);
    p.cell[o] = (uint32_t)(g0 + 2 + i * d0);
  }
}

// Thermal shell injection (no reference counterpart; the magnetosphere
// workload's "pairs injected in the inner cells with a temperature"): for
// every row the reference injects into (inject_ptc above), `inj` pairs in
// each of the r_cells radial cells from the reference's injection cell
// g0 + 2 outward, with the reference's surface-density gate per row.  A
// pair shares a uniformly drawn position in its cell; each member's
// momentum is an isotropic Maxwell-Juttner draw of temperature theta;
// weights w sin(theta) as in inject_ptc.  Pair t of the launch (row-major
// over rows, radial cells, pairs) takes slots base + 2t and base + 2t + 1, a
// thread each: the rejection loops of the momentum draw are all of the time,
// and two draws in turn took twice one (510 rows x 4 pairs: 19 -> 10 us).
template <typename R>
__global__ void k_logsph_inject_shell(Mesh m, LsParams lp, PtcView<R> p, uint64_t base,
                                      int r_cells, int inj, double theta, double w,
                                      double q_e, uint64_t seed, uint32_t epoch, int Hs,
                                      uint64_t id_base, const long long *__restrict__ surf,
                                      const unsigned long long *__restrict__ dc, uint64_t cap) {
  const int g0 = m.guard[0], g1 = m.guard[1], d0 = m.dims[0];
  const int N1 = m.dims[1] - 2 * g1;
  const uint64_t per_row = (uint64_t)r_cells * inj;
  const uint64_t tt = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, t = tt >> 1;
  const int s = (int)(tt & 1);
  if (t >= (uint64_t)(N1 - 2) * per_row) return;
  if (dc) {  // device-count mode: base, ids and epoch from the device
    base = dc[DC_NUM];
    id_base = dc[DC_ID];
    epoch = (uint32_t)dc[DC_INJ_EPOCH];
  }
  const int i = g1 + 1 + (int)(t / per_row);
  const int ir = (int)((t % per_row) / inj);
  const uint64_t off = base + 2 * t;
  if (dc && off + 1 >= cap) return;  // past the capacity: dropped, counted
  const double de = fx_value(surf[i - g1], surf[N1 + i - g1], Hs);
  const double dp = fx_value(surf[2 * N1 + i - g1], surf[3 * N1 + i - g1], Hs);
  const double dens = de > dp ? de : dp;
  const double sgate = (1.0 / m.delta[1]) * (1.0 / m.delta[1]);
  const bool gated = q_e * dens > 1.5 * sgate * apt_sin(lpos(m, 1, i, 0.5));
  const uint64_t o = off + s;
  if (p.id) p.id[o] = id_base + (o - base);
  if (gated) {
    p.cell[o] = MAX_CELL;
    return;
  }
  const uint64_t pid = ((uint64_t)epoch << 32) | (t & 0xffffffffull);
  double u0, u1, u2, u3;
  uniform2(seed, pid, 0, 14, u0, u1);
  uniform2(seed, pid, 1, 14, u2, u3);
  const double x1 = 1.0 - u0, x2 = 1.0 - u1;
  double st, ct;
  apt_sincos(lpos(m, 1, i, x2), st, ct);
  const uint32_t fl = FLAG_PRIMARY | (u2 < lp.track_percent ? FLAG_TRACKED : 0u);
  double ux, uy, uz;
  sample_mj(theta, 0.0, seed,
            (1ull << 62) | ((uint64_t)(epoch & 0x1fffffffu) << 33) | (t << 1) | (uint64_t)s,
            ux, uy, uz);
  R x1r = (R)x1, x2r = (R)x2;
  if constexpr (!std::is_same<R, double>::value) {
    if (x1r >= 1.0f) x1r = 0x1.fffffep-1f;
    if (x2r >= 1.0f) x2r = 0x1.fffffep-1f;
  }
  p.x1[o] = x1r;
  p.x2[o] = x2r;
  p.x3[o] = (R)0;
  p.p1[o] = (R)ux;
  p.p2[o] = (R)uy;
  p.p3[o] = (R)uz;
  if (p.E) p.E[o] = (R)sqrt(1.0 + ux * ux + uy * uy + uz * uz);
  p.w[o] = (R)(w * st);
  const uint32_t type = s == 0 ? 0u : (lp.inject_ions ? 2u : 1u);
  p.flag[o] = fl | (type << 29);
  p.cell[o] = (uint32_t)(g0 + 2 + ir + i * d0);
}

// Device-count mode: the pairs of an injection that fitted below the
// capacity (the first ones in slot order) are added to the count and ids,
// the rest counted as overflow; the injection epoch advances.
__global__ void k_inject_finish(unsigned long long *__restrict__ dc, uint64_t npairs,
                                uint64_t cap, unsigned long long *__restrict__ counters) {
  if (blockIdx.x != 0 || threadIdx.x != 0) return;
  const unsigned long long room = cap > dc[DC_NUM] ? (cap - dc[DC_NUM]) / 2 : 0ull;
  const unsigned long long made = npairs < room ? npairs : room;
  if (made < npairs && counters) atomicAdd(&counters[CTR_OVERFLOW], npairs - made);
  dc[DC_NUM] += 2 * made;
  dc[DC_ID] += 2 * made;
  dc[DC_INJ_EPOCH] += 1;
}

// ---------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------
static inline dim3 grid1(uint64_t n, int b = 256) {
  return dim3((unsigned)((n + b - 1) / b));
}

// runs: the slots sorted by cell, if there are any (their end is known on the
// host exactly with host counts, else as a bound)
template <typename R>
static hipError_t launch_logsph_push(const Mesh &m, const Species &sp, const LsParams &lp, R dt,
                                     int rho, int nrho, const PtcView<R> &p,
                                     const LsFields<R> &F, const typename LsAccOf<R>::type &acc,
                                     unsigned long long *counters, uint64_t n, hipStream_t st,
                                     const unsigned long long *dn, const CellRuns *runs) {
  if (n == 0) return hipSuccess;
  const uint32_t nwork = runs ? runs->items : 0;
  const uint64_t rest = runs && !dn ? n - runs->end : n;
  // Slots of a workgroup behind the tiles, a slot a thread if they can be: the
  // cells of many do not fit the window.  Before a sort every slot is there, and
  // from 16 to a cell on two a thread cover no more cells (us per push, slots in
  // cell order, FP32, 1024 x 1024: 4 M 468 with 512, 577 with 1024; 24 M 2355,
  // 2086; 512 x 512: 8 M 820, 762).
  // Under a bound nearly all of the workgroups behind sorted slots are past the
  // count, and each holds 40 KB of LDS while it finds out: there are at most 4096
  // (1024 x 1024 with pairs, 0.42 -> 0.32 ms a push) or one for 4096 slots of the
  // bound, and a thread takes several slots where the count needs it.
  uint64_t slots = runs == nullptr && rest >= 16 * m.size() ? 2 * LS_NT : LS_NT;
  if (dn && runs) {
    slots = (rest + LS_DEV_TAIL - 1) / LS_DEV_TAIL;
    slots = slots < LS_NT ? LS_NT : slots > 4096 ? 4096 : slots;
  }
  uint64_t tail = (rest + slots - 1) / slots;
  if (tail == 0) tail = 1;  // the guard rows above the tiles
  const uint64_t grid = nwork + (runs ? 1 : 0) + tail;
  const CellRuns cr = runs ? *runs : CellRuns{};
  if (rho)
    k_logsph_push<R, true><<<(unsigned)grid, LS_NT, 0, st>>>(m, sp, lp, dt, nrho, p, F, acc, cr,
                                                             nwork, counters, n, dn);
  else
    k_logsph_push<R, false><<<(unsigned)grid, LS_NT, 0, st>>>(m, sp, lp, dt, nrho, p, F, acc, cr,
                                                              nwork, counters, n, dn);
  return hipGetLastError();
}

// species whose charge the window holds: those with a charge array, at
// most 4 (nrho <= 4)
static int rho_species(long long *const *R0) {
  int k = 0;
  while (k < 4 && R0[k]) k++;
  return k;
}

hipError_t launch_logsph_push_f64(const Mesh &m, const Species &sp,
                                  const LsParams &lp, double dt, int H,
                                  int rho, const PtcF64 &p,
                                  const FieldsF64 &f, const AccF64 &a,
                                  unsigned long long *counters, uint64_t n,
                                  hipStream_t st, const unsigned long long *dn,
                                  const CellRuns *runs) {
  LsAccF64 acc;
  for (int c = 0; c < 3; c++)
    for (int l = 0; l < 2; l++) acc.J[c][l] = a.J[c][l];
  long long *r0[4];
  for (int s = 0; s < 4; s++) {
    for (int l = 0; l < 2; l++) acc.R[s][l] = a.R[s][l];
    r0[s] = a.R[s][0];
  }
  acc.H = H;
  acc.d0 = m.dims[0];
  const LsFields<double> F{f.E[0], f.E[1], f.E[2], f.B[0], f.B[1], f.B[2]};
  return launch_logsph_push<double>(m, sp, lp, dt, rho, rho_species(r0), view_of(p), F, acc,
                                   counters, n, st, dn, runs);
}

hipError_t launch_logsph_push_f32(const Mesh &m, const Species &sp,
                                  const LsParams &lp, float dt, int S,
                                  const PtcF32 &p, const FieldsF32 &f,
                                  const AccMixed &a,
                                  unsigned long long *counters, uint64_t n,
                                  hipStream_t st, const unsigned long long *dn,
                                  const CellRuns *runs) {
  LsAccF32 acc;
  for (int c = 0; c < 3; c++) acc.J[c] = a.J[c];
  long long *r0[4];
  for (int s = 0; s < 4; s++) {
    acc.R[s] = a.R[s];
    r0[s] = a.R[s];
  }
  acc.scale = ldexpf(1.0f, S);
  acc.d0 = m.dims[0];
  const LsFields<float> F{f.E[0], f.E[1], f.E[2], f.B[0], f.B[1], f.B[2]};
  return launch_logsph_push<float>(m, sp, lp, dt, a.rho, rho_species(r0), view_of(p), F, acc,
                                  counters, n, st, dn, runs);
}

template <typename T>
hipError_t launch_logsph_process_j(const Mesh &m, const LsCoef &cf, double dt,
                                   int H, int limbs, long long *const (*J)[2],
                                   long long *const (*Rr)[2], int ns, T *const *Jout,
                                   T *const *Rout, int axis, hipStream_t st) {
  const uint64_t n = m.size();
  const double wj = m.delta[0] * m.delta[1] / dt;
  LsProcess<T> a{};
  for (int c = 0; c < 3; c++) {
    a.jh[c] = J[c][0];
    a.jl[c] = J[c][1];
    a.J[c] = Jout[c];
  }
  for (int s = 0; s < ns; s++) {
    a.rh[s] = Rr[s][0];
    a.rl[s] = Rr[s][1];
    a.Rho[s] = Rout[s];
  }
  a.ns = ns;
  k_logsph_process<T><<<grid1(n), 256, 0, st>>>(m, cf, wj, H, limbs, a, axis, n);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_logsph_filter(const Mesh &m, T *j, T *tmp, const double *A,
                                hipStream_t st) {
  const uint64_t nb = (uint64_t)(m.dims[0] - 2 * m.guard[0]) *
                      (m.dims[1] - 2 * m.guard[1]);
  k_logsph_filter<T><<<grid1(nb), 256, 0, st>>>(m, j, tmp, A);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  // whole-array copy back (ptc_updater_logsph.cu:752): guards take tmp's
  return hipMemcpyAsync(j, tmp, m.size() * sizeof(T), hipMemcpyDeviceToDevice,
                        st);
}

template <typename T>
hipError_t launch_logsph_axis_j3(const Mesh &m, T *J3, hipStream_t st) {
  k_logsph_axis_j3<T><<<grid1(m.dims[0]), 256, 0, st>>>(m, J3);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_logsph_field_update(const Mesh &m, const LsCoef &cf,
                                      const LsParams &lp, const FieldSet<T> &f,
                                      double dt, double edotb_delta, hipStream_t st) {
  const uint64_t nb = (uint64_t)(m.dims[0] - 2 * m.guard[0]) *
                      (m.dims[1] - 2 * m.guard[1]);
  // the bulk and the theta = 0 row below it
  const dim3 grid = grid1(nb + (uint64_t)(m.dims[0] - 2 * m.guard[0]));
  k_logsph_update_b<T><<<grid, 256, 0, st>>>(m, cf, lp, f, (T)dt, nb);
  k_logsph_update_e<T><<<grid, 256, 0, st>>>(m, cf, f, (T)dt, nb);
  k_logsph_divs<T><<<grid, 256, 0, st>>>(m, cf, f, (T)edotb_delta, nb);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_logsph_field_boundary(const Mesh &m, const LsParams &lp,
                                        const FieldSet<T> &f, double omega,
                                        hipStream_t st) {
  const uint64_t cells = (uint64_t)m.dims[1] * (m.guard[0] + lp.damping_length);
  k_logsph_boundary<T><<<grid1(m.dims[0] + cells, 64), 64, 0, st>>>(m, lp, f, omega);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_logsph_inject(const Mesh &m, const LsParams &lp,
                                const PtcView<R> &p, uint64_t number, int inj,
                                double p1, double w, double q_e, uint64_t seed,
                                uint32_t epoch, int Hs, uint64_t id_base,
                                long long *surf, hipStream_t st, int r_cells, double theta,
                                unsigned long long *dc, uint64_t cap,
                                unsigned long long *counters) {
  const int N1 = m.dims[1] - 2 * m.guard[1];
  hipError_t e = launch_fill<long long>(surf, 0, 4 * (uint64_t)N1, st);
  if (e != hipSuccess) return e;
  if (number > 0)
    k_logsph_surface<R><<<slot_blocks((number + SURF_E - 1) / SURF_E, dc), 256, 0, st>>>(
        m, p.cell, p.flag, p.w, number, surf, Hs, dc ? dc + DC_NUM : nullptr);
  const uint64_t nt = (uint64_t)(N1 - 2) * (r_cells > 0 ? r_cells : 1) * inj;
  if (nt > 0) {
    if (r_cells > 0)
      k_logsph_inject_shell<R><<<grid1(2 * nt, 64), 64, 0, st>>>(
          m, lp, p, number, r_cells, inj, theta, w, q_e, seed, epoch, Hs, id_base, surf, dc, cap);
    else
      k_logsph_inject<R><<<grid1(nt), 256, 0, st>>>(m, lp, p, number, inj, p1, w, q_e, seed,
                                                    epoch, Hs, id_base, surf, dc, cap);
  }
  if (dc) k_inject_finish<<<1, 64, 0, st>>>(dc, nt, cap, counters);
  return hipGetLastError();
}

#define INST(T)                                                                \
  template hipError_t launch_logsph_process_j<T>(                              \
      const Mesh &, const LsCoef &, double, int, int, long long *const (*)[2], \
      long long *const (*)[2], int, T *const *, T *const *, int, hipStream_t); \
  template hipError_t launch_logsph_filter<T>(const Mesh &, T *, T *,          \
                                              const double *, hipStream_t);    \
  template hipError_t launch_logsph_axis_j3<T>(const Mesh &, T *, hipStream_t); \
  template hipError_t launch_logsph_field_update<T>(                           \
      const Mesh &, const LsCoef &, const LsParams &, const FieldSet<T> &,     \
      double, double, hipStream_t);                                            \
  template hipError_t launch_logsph_field_boundary<T>(                         \
      const Mesh &, const LsParams &, const FieldSet<T> &, double,             \
      hipStream_t);                                                            \
  template hipError_t launch_logsph_inject<T>(                                 \
      const Mesh &, const LsParams &, const PtcView<T> &, uint64_t, int,       \
      double, double, double, uint64_t, uint32_t, int, uint64_t, long long *,  \
      hipStream_t, int, double, unsigned long long *, uint64_t,                \
      unsigned long long *);
INST(double)
INST(float)
#undef INST

}  // namespace apt
