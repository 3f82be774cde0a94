// kern_cart_f64.hip -- plain FP64 Cartesian particle update (the drop-in
// form).  One fused pass per particle: push (ptc_push_cart_{1,2,3}d,
// ptc_updater.cu:21-218), then move + Esirkepov deposit
// (deposit_current_cart_{1,2,3}d, ptc_updater.cu:220-499), then the periodic
// wrap that the reference does through send_particles.  Expressions keep the
// reference's operation order and this file is built with -ffp-contract=off,
// so every particle's arithmetic is bit-identical to the CPU restatement.
// The current goes through two-limb int64 fixed point (order independent):
// in 1D with device-scope atomics on the wrapped (periodic) index, the lanes
// of a wave that add to the same element summed first (one atomic pair per
// element: 4.4x faster at 200 particles per cell); in 2D and 3D into an LDS
// window per workgroup chunk of cell-sorted particles, flushed once per
// element (k_push_deposit_f64_win below).  Slots sorted by cell, with a table
// of their runs by tile, take k_push_deposit_f64_runs instead.
#include "apt_common.hpp"
#include "apt_f64.hpp"
#include "apt_kernels.hpp"
#include "apt_runs.hpp"

#include <climits>

// LDS-window shapes of the 2D and 3D updates: R consecutive slots per lane
// run, K slots per lane, window capacity in int64 elements
#ifndef F64_WIN2_R
#define F64_WIN2_R 16
#endif
#ifndef F64_WIN2_K
#define F64_WIN2_K 8
#endif
#ifndef F64_WIN2_CAP
#define F64_WIN2_CAP 6144
#endif
#ifndef F64_WIN3_R
#define F64_WIN3_R 4
#endif
#ifndef F64_WIN3_K
#define F64_WIN3_K 1
#endif
#ifndef F64_WIN3_CAP
#define F64_WIN3_CAP 10240
#endif
// waves per SIMD the 2D / 3D updates are compiled for (0: the compiler's
// choice); the LDS window must leave room for that many workgroups per CU
#ifndef F64_WIN2_WAVES
#define F64_WIN2_WAVES 0
#endif
#ifndef F64_WIN3_WAVES
#define F64_WIN3_WAVES 0
#endif

namespace apt {

// A particle as its push reads it (gamma is recomputed from the momenta).
struct Ptc64Regs {
  uint32_t cell, flag;
  double x1, x2, x3, p1, p2, p3, w;
};

__device__ __forceinline__ void load_ptc64(const PtcF64 &p, uint64_t i, Ptc64Regs &r) {
  r.cell = p.cell[i];
  r.flag = p.flag[i];
  r.x1 = p.x1[i];
  r.x2 = p.x2[i];
  r.x3 = p.x3[i];
  r.p1 = p.p1[i];
  r.p2 = p.p2[i];
  r.p3 = p.p3[i];
  r.w = p.w[i];
}

// Push (ptc_push_cart_1d, ptc_updater.cu:21-76) and move (the first part
// of deposit_current_cart_1d, :220-245) of one live particle: stores
// momenta, gamma, cell and offsets, and returns what the deposit needs.
template <class Gather>
__device__ __forceinline__ void push_move_1d_f64(const Mesh &m, const double *qdt, const double *qs,
                                                 double dt, const PtcF64 &p, const Gather &gather,
                                                 unsigned long long *counters, uint64_t idx,
                                                 const Ptc64Regs &r, int &s, bool &dep,
                                                 double &weight, double &old_x1, double &new_x1,
                                                 int &dc1, double &v2, double &v3) {
  const uint32_t flag = r.flag, c = r.cell;
  s = ptc_species(flag);
  double x1 = r.x1, x2 = r.x2, x3 = r.x3;
  double p1 = r.p1, p2 = r.p2, p3 = r.p3;
  double q_over_m = qdt[s];
  if (p1 != p1 || p2 != p2 || p3 != p3)
    atomicAdd(&counters[CTR_NAN], 1ull);
  double gamma = sqrt(1.0 + p1 * p1 + p2 * p2 + p3 * p3);
  if (!(flag & FLAG_IGNORE_EM)) {
    double F[6];
    gather(x1, F);
    vay_push(p1, p2, p3, gamma, F[0] * q_over_m, F[1] * q_over_m, F[2] * q_over_m,
             F[3] * q_over_m, F[4] * q_over_m, F[5] * q_over_m);
    p.p1[idx] = p1;
    p.p2[idx] = p2;
    p.p3[idx] = p3;
    p.E[idx] = gamma;
  } else {
    gamma = p.E[idx];  // ignore_EM: stored momenta and gamma are left as they were
  }
  double v1 = p1 / gamma;
  v2 = p2 / gamma;
  v3 = p3 / gamma;
  double w = r.w;
  old_x1 = x1;
  new_x1 = old_x1 + (v1 * dt) / m.delta[0];
  dc1 = (int)floor(new_x1);
  if (dc1 > 1 || dc1 < -1) atomicAdd(&counters[CTR_MULTICELL], 1ull);
  new_x1 -= (double)dc1;
  p.cell[idx] = (uint32_t)m.wrap(0, (int)c + dc1);
  p.x1[idx] = new_x1;
  p.x2[idx] = x2 + v2 * dt;
  p.x3[idx] = x3 + v3 * dt;
  weight = qs[s] * w;
  dep = !(flag & FLAG_IGNORE_CURRENT);
}


// Where a particle's current contributions go.  add(q, di, dj, dk, v) adds
// v to component q (0..2: J1..J3; 3 + s: Rho of species s) at offset
// (di, dj, dk) from the particle's cell (before the move).

// Straight to the fixed-point accumulators in HBM, on the wrapped index.
struct DepGlobal {
  const Mesh &m;
  const AccF64 &a;
  int H, c1, c2, c3;
  __device__ __forceinline__ void add(int q, int di, int dj, int dk, double v) const {
    long long *hi = q < 3 ? a.J[q][0] : a.R[q - 3][0];
    long long *lo = q < 3 ? a.J[q][1] : a.R[q - 3][1];
    acc_add(hi, lo, m.widx(c1 + di, c2 + dj, c3 + dk), v, H);
  }
};

// The same with the accumulators' addresses (two limbs per component) in
// LDS, which keeps them out of the scalar registers of a kernel that rarely
// needs them.
struct DepGlobalL {
  const Mesh &m;
  long long *const *dst;
  int H, c1, c2, c3;
  __device__ __forceinline__ void add(int q, int di, int dj, int dk, double v) const {
    acc_add(dst[2 * q], dst[2 * q + 1], m.widx(c1 + di, c2 + dj, c3 + dk), v, H);
  }
};

// Into the workgroup's LDS window: `cells` elements per limb and component,
// x fastest; `base` is the particle's cell in the window.  Components past
// the window's (Rho of a species it does not hold) go to HBM.
struct DepWindow {
  long long *win;
  int cells, W0, W01, base, H, nq;
  DepGlobal g;
  __device__ __forceinline__ void add(int q, int di, int dj, int dk, double v) const {
    if (q >= nq) {
      g.add(q, di, dj, dk, v);
      return;
    }
    long long h, l;
    fx_split(v, H, h, l);
    long long *e = win + 2 * q * cells + base + di + W0 * dj + W01 * dk;
    if (h != 0)
      __hip_atomic_fetch_add(e, h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (l != 0)
      __hip_atomic_fetch_add(e + cells, l, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
};

// What the deposit of a 2D or 3D particle needs of its push and move.
struct Moved {
  double old_x[3], new_x[3], v3, weight;  // weight = -q w
  int dc[3], s;
  bool on;  // deposits current
};

// Push (ptc_push_cart_2d/3d, ptc_updater.cu:78-218) and move (:295-330,
// :400-440) of one live particle in bulk cell (c1, c2, c3); gather(x, F) fills
// the six interpolated fields; qdt, qs are dt q / 2m and q by species.
template <int DIM, class Gather>
__device__ __forceinline__ void push_move_f64(const Mesh &m, const double *qdt, const double *qs,
                                              double dt, const PtcF64 &p,
                                              unsigned long long *counters,
                                              uint64_t idx, const Ptc64Regs &r, int c1, int c2,
                                              int c3, const Gather &gather, Moved &mv) {
  const uint32_t flag = r.flag;
  int s = ptc_species(flag);
  double x1 = r.x1, x2 = r.x2, x3 = r.x3;
  double p1 = r.p1, p2 = r.p2, p3 = r.p3;
  double q_over_m = qdt[s];
  if (p1 != p1 || p2 != p2 || p3 != p3)
    atomicAdd(&counters[CTR_NAN], 1ull);
  double gamma = sqrt(1.0 + p1 * p1 + p2 * p2 + p3 * p3);
  if (!(flag & FLAG_IGNORE_EM)) {
    double F[6];
    gather(x1, x2, x3, F);
    vay_push(p1, p2, p3, gamma, F[0] * q_over_m, F[1] * q_over_m, F[2] * q_over_m,
             F[3] * q_over_m, F[4] * q_over_m, F[5] * q_over_m);
    p.p1[idx] = p1;
    p.p2[idx] = p2;
    p.p3[idx] = p3;
    p.E[idx] = gamma;
  } else {
    gamma = p.E[idx];  // ignore_EM: stored momenta and gamma are left as they were
  }
  // ---- move (reads the stored momenta / gamma) ----
  double v1 = p1 / gamma, v2 = p2 / gamma, v3 = p3 / gamma;
  double w = r.w;
  const double old_x[3] = {x1, x2, x3}, v[3] = {v1, v2, v3};
  bool multi = false;
#pragma unroll
  for (int d = 0; d < 3; d++) {
    mv.old_x[d] = old_x[d];
    mv.dc[d] = 0;
    if (d < DIM) {
      double n = old_x[d] + (v[d] * dt) * m.inv_delta[d];
      const int dc = (int)floor(n);
      multi = multi || dc > 1 || dc < -1;
      n -= (double)dc;
      mv.new_x[d] = n;
      mv.dc[d] = dc;
    } else {
      mv.new_x[d] = old_x[d] + v[d] * dt;
    }
  }
  if (multi) atomicAdd(&counters[CTR_MULTICELL], 1ull);
  p.cell[idx] = (uint32_t)m.idx(m.wrap(0, c1 + mv.dc[0]), m.wrap(1, c2 + mv.dc[1]),
                                DIM == 3 ? m.wrap(2, c3 + mv.dc[2]) : 0);
  p.x1[idx] = mv.new_x[0];
  p.x2[idx] = mv.new_x[1];
  p.x3[idx] = mv.new_x[2];
  mv.v3 = v3;
  mv.s = s;
  mv.weight = -qs[s] * w;
  mv.on = !(flag & FLAG_IGNORE_CURRENT);
}

// every tap of the reference's interpolators
template <int DIM>
__device__ __forceinline__ void gather_f64(const Mesh &m, const FieldsF64 &f, double x1,
                                           double x2, double x3, int c1, int c2, int c3,
                                           double F[6]) {
  const int d0 = m.dims[0], d1 = m.dims[1];
  constexpr int st[6] = {ST_E1, ST_E2, ST_E3, ST_B1, ST_B2, ST_B3};
#pragma unroll
  for (int q = 0; q < 6; q++) {
    const double *a = q < 3 ? f.E[q] : f.B[q - 3];
    F[q] = DIM == 1 ? gather1(a, x1, c1, st[q])
           : DIM == 2 ? gather2(a, d0, x1, x2, c1, c2, st[q])
                      : gather3(a, d0, d1, x1, x2, x3, c1, c2, c3, st[q]);
  }
}

// Esirkepov deposit of a moved particle (deposit_current_cart_2d/3d,
// :331-384, :441-499) through `dep`
template <int DIM, class Dep>
__device__ __forceinline__ void deposit_loops_f64(const Moved &mv, int rho, const Dep &dep) {
  const double weight = mv.weight, v3 = mv.v3;
  const double old_x1 = mv.old_x[0], old_x2 = mv.old_x[1], old_x3 = mv.old_x[2];
  const double new_x1 = mv.new_x[0], new_x2 = mv.new_x[1], new_x3 = mv.new_x[2];
  const int dc1 = mv.dc[0], dc2 = mv.dc[1], dc3 = mv.dc[2], s = mv.s;
  const int j0 = (dc2 == -1 ? -2 : -1), j1 = (dc2 == 1 ? 1 : 0);
  const int i0 = (dc1 == -1 ? -2 : -1), i1 = (dc1 == 1 ? 1 : 0);
  if (DIM == 2) {
    double djy[3] = {0.0, 0.0, 0.0};
    for (int j = j0; j <= j1; j++) {
      double sy0 = cic(-old_x2 + j + 1);
      double sy1 = cic(-new_x2 + (j + 1 - dc2));
      double djx = 0.0;
      for (int i = i0; i <= i1; i++) {
        double sx0 = cic(-old_x1 + i + 1);
        double sx1 = cic(-new_x1 + (i + 1 - dc1));
        djx += movement2d(sy0, sy1, sx0, sx1);
        dep.add(0, i + 1, j, 0, weight * djx);
        djy[i - i0] += movement2d(sx0, sx1, sy0, sy1);
        dep.add(1, i, j + 1, 0, weight * djy[i - i0]);
        double val2 = center2d(sx0, sx1, sy0, sy1);
        dep.add(2, i, j, 0, -weight * v3 * val2);
        if (rho) {
          double s1 = sx1 * sy1;
          dep.add(3 + s, i, j, 0, -weight * s1);
        }
      }
    }
  } else {
    const int k0 = (dc3 == -1 ? -2 : -1), k1 = (dc3 == 1 ? 1 : 0);
    double djz[3][3] = {{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}};
    for (int k = k0; k <= k1; k++) {
      double sz0 = cic(-old_x3 + k + 1);
      double sz1 = cic(-new_x3 + (k + 1 - dc3));
      double djy[3] = {0.0, 0.0, 0.0};
      for (int j = j0; j <= j1; j++) {
        double sy0 = cic(-old_x2 + j + 1);
        double sy1 = cic(-new_x2 + (j + 1 - dc2));
        double djx = 0.0;
        for (int i = i0; i <= i1; i++) {
          double sx0 = cic(-old_x1 + i + 1);
          double sx1 = cic(-new_x1 + (i + 1 - dc1));
          djx += movement3d(sy0, sy1, sz0, sz1, sx0, sx1);
          dep.add(0, i + 1, j, k, weight * djx);
          djy[i - i0] += movement3d(sx0, sx1, sz0, sz1, sy0, sy1);
          dep.add(1, i, j + 1, k, weight * djy[i - i0]);
          djz[j - j0][i - i0] += movement3d(sx0, sx1, sy0, sy1, sz0, sz1);
          dep.add(2, i, j, k + 1, weight * djz[j - j0][i - i0]);
          if (rho) {
            double s1 = sx1 * sy1 * sz1;
            dep.add(3 + s, i, j, k, -weight * s1);
          }
        }
      }
    }
  }
}

// Push, move and deposit of one live particle in bulk cell (c1, c2, c3).
template <int DIM, class Dep>
__device__ __forceinline__ void push_deposit_f64(const Mesh &m, const Species &sp, double dt,
                                                 int rho, const PtcF64 &p, const FieldsF64 &f,
                                                 unsigned long long *counters, uint64_t idx,
                                                 int c1, int c2, int c3, const Dep &dep) {
  Moved mv;
  Ptc64Regs r;
  load_ptc64(p, idx, r);
  push_move_f64<DIM>(
      m, sp.qdt, sp.q, dt, p, counters, idx, r, c1, c2, c3,
      [&](double x1, double x2, double x3, double F[6]) {
        gather_f64<DIM>(m, f, x1, x2, x3, c1, c2, c3, F);
      },
      mv);
  if (mv.on) deposit_loops_f64<DIM>(mv, rho, dep);
}

template <int DIM>
__global__ void __launch_bounds__(256)
    k_push_deposit_f64(Mesh m, Species sp, double dt, int H, int rho,
                       PtcF64 p, FieldsF64 f, AccF64 a,
                       unsigned long long *__restrict__ counters,
                       uint64_t n) {
  uint64_t idx = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  // the 1D deposit goes through wave_acc_add, which every lane of the wave
  // enters: lanes without a particle take part with nothing to add
  bool live = idx < n;
  uint32_t c = live ? p.cell[idx] : MAX_CELL;
  live = live && c != MAX_CELL;
  int c1 = 0, c2 = 0, c3 = 0;
  if (live) {
    m.split(c, c1, c2, c3);
    if (!m.in_bulk(c1, c2, c3)) {
      p.cell[idx] = MAX_CELL;
      live = false;
    }
  }
  if (DIM != 1 && !live) return;
  if (DIM == 1) {
    bool dep = false;
    int s = 0, dc1 = 0;
    double weight = 0.0, old_x1 = 0.0, new_x1 = 0.0, v2 = 0.0, v3 = 0.0;
    if (live) {
      Ptc64Regs r;
      load_ptc64(p, idx, r);
      push_move_1d_f64(
          m, sp.qdt, sp.q, dt, p,
          [&](double x1, double F[6]) { gather_f64<1>(m, f, x1, 0.0, 0.0, (int)c, 0, 0, F); },
          counters, idx, r, s, dep, weight, old_x1, new_x1, dc1, v2, v3);
    }
    {
      // deposit_current_cart_1d (ptc_updater.cu:220-293): i over i0..i1
      const int i0 = (dc1 == -1 ? -2 : -1), i1 = (dc1 == 1 ? 1 : 0);
      double djx = 0.0;
      for (int i = -2; i <= 1; i++) {
        const bool in = dep && i >= i0 && i <= i1;
        double vj1 = 0.0, vj2 = 0.0, vj3 = 0.0, vr = 0.0;
        uint64_t o1 = 0, o = 0;
        if (in) {
          double sx0 = cic(-old_x1 + i + 1);
          double sx1 = cic(-new_x1 + (i + 1 - dc1));
          djx += sx1 - sx0;
          o1 = m.widx(i + (int)c + 1, 0, 0);
          o = m.widx(i + (int)c, 0, 0);
          vj1 = -weight * djx;
          double val1 = 0.5 * (sx0 + sx1);
          vj2 = weight * v2 * val1;
          vj3 = weight * v3 * val1;
          vr = weight * sx1;
        }
        wave_acc_add(a.J[0][0], a.J[0][1], o1, o1, vj1, H, in);
        wave_acc_add(a.J[1][0], a.J[1][1], o, o, vj2, H, in);
        wave_acc_add(a.J[2][0], a.J[2][1], o, o, vj3, H, in);
        if (rho)
          wave_acc_add(a.R[s][0], a.R[s][1], o, o | ((uint64_t)s << 56), vr, H, in);
      }
    }
    return;
  }
  if constexpr (DIM > 1)
    push_deposit_f64<DIM>(m, sp, dt, rho, p, f, counters, idx, c1, c2, c3,
                          DepGlobal{m, a, H, c1, c2, c3});
}

// The 2D/3D FP64 update with the current summed in LDS (J and, in 2D, Rho;
// 80 KB of LDS in 3D, 48 KB in 2D).  A workgroup takes
// a chunk of 256 K consecutive slots.  The particles are kept sorted by
// cell, so a chunk covers a short run of cells: the workgroup finds the
// extent of its particles' cells (differences to the chunk's lowest cell,
// taken the short way round periodic axes), pads it by the deposit's reach
// of two cells, and, when the two-limb J (and Rho) window fits in LDS,
// adds every contribution there with workgroup-scope int64 atomics and
// flushes each non-zero element once to HBM.  A chunk whose particles are
// too spread out for the window deposits straight to HBM (counted).
// Lanes are arranged so that one instruction of a wave covers 64 / R runs
// of R consecutive slots, spaced R K slots apart: a wave's lanes then sit in
// several cells instead of one, which spreads the LDS atomics over more
// addresses, while each run still reads R consecutive elements.  The sums
// are of integers, so the result equals the HBM path bit for bit.
template <int DIM, int R, int K, int WCAP, int WAVES>
__attribute__((amdgpu_waves_per_eu(WAVES > 0 ? WAVES : 1))) __global__ void __launch_bounds__(256)
    k_push_deposit_f64_win(Mesh m, Species sp, double dt, int H, int rho, int nsp, PtcF64 p,
                           FieldsF64 f, AccF64 a, unsigned long long *__restrict__ counters,
                           uint64_t n) {
  static_assert(64 % R == 0, "R divides the wave");
  __shared__ long long win[WCAP];
  __shared__ long long *s_dst[14];
  __shared__ uint32_t s_ref;
  __shared__ int s_lo[2][3], s_hi[2][3];  // window extents under the two offset maps
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const uint64_t first = (uint64_t)blockIdx.x * (256 * K) + (uint64_t)wv * (64 * K) +
                         (uint64_t)(lane / R) * (R * K) + (uint64_t)(lane % R);
  if (tid < 6) {
    (&s_lo[0][0])[tid] = INT_MAX;
    (&s_hi[0][0])[tid] = INT_MIN;
  }
  if (tid == 0) s_ref = MAX_CELL;
  if (tid < 6) s_dst[tid] = a.J[tid >> 1][tid & 1];
  if (tid >= 6 && tid < 14) s_dst[tid] = a.R[(tid - 6) >> 1][tid & 1];
  __syncthreads();
  // cells of this lane's particles; particles outside the bulk are erased
  uint32_t cl[K];
  uint32_t mine = MAX_CELL;
#pragma unroll
  for (int k = 0; k < K; k++) {
    const uint64_t idx = first + (uint64_t)R * k;
    uint32_t c = idx < n ? p.cell[idx] : MAX_CELL;
    if (c != MAX_CELL) {
      int c1, c2, c3;
      m.split(c, c1, c2, c3);
      if (!m.in_bulk(c1, c2, c3)) {
        p.cell[idx] = MAX_CELL;
        c = MAX_CELL;
      }
    }
    cl[k] = c;
    mine = c < mine ? c : mine;
  }
  if (mine != MAX_CELL) atomicMin(&s_ref, mine);
  __syncthreads();
  const uint32_t ref = s_ref;
  if (ref == MAX_CELL) return;  // no live particle in the chunk
  int r[3];
  m.split(ref, r[0], r[1], r[2]);
  // Offset of a cell from the chunk's lowest cell along one axis.  On a
  // periodic axis the offset is taken in [-T, N - T) for one of two T, the
  // one that gives the chunk the narrower window on that axis:
  //   T = N/2 (the short way round), which keeps particles a few cells on
  //   either side of the reference together (cells sorted by linear index
  //   put the reference anywhere along x when the chunk covers two rows);
  //   T = min(8, N/2), which keeps a chunk that runs past the end of a short
  //   row (or plane) contiguous when it spans more than half the period.
  auto relT = [&](int ax, int c, int T) {
    int d = c - r[ax];
    if (m.periodic[ax]) {
      const int N = m.N[ax];
      if (d < -T) d += N;
      else if (d >= N - T) d -= N;
    }
    return d;
  };
  auto Tof = [&](int ax, int v) {
    const int h = m.N[ax] / 2;
    return v == 0 ? h : (h < 8 ? h : 8);
  };
  {
    int lo[2][3], hi[2][3];
#pragma unroll
    for (int v = 0; v < 2; v++)
#pragma unroll
      for (int ax = 0; ax < 3; ax++) {
        lo[v][ax] = INT_MAX;
        hi[v][ax] = INT_MIN;
      }
#pragma unroll
    for (int k = 0; k < K; k++) {
      if (cl[k] == MAX_CELL) continue;
      int c[3];
      m.split(cl[k], c[0], c[1], c[2]);
#pragma unroll
      for (int v = 0; v < 2; v++)
#pragma unroll
        for (int ax = 0; ax < DIM; ax++) {
          const int d = relT(ax, c[ax], Tof(ax, v));
          lo[v][ax] = d < lo[v][ax] ? d : lo[v][ax];
          hi[v][ax] = d > hi[v][ax] ? d : hi[v][ax];
        }
    }
#pragma unroll
    for (int v = 0; v < 2; v++)
#pragma unroll
      for (int ax = 0; ax < DIM; ax++)
        if (lo[v][ax] <= hi[v][ax]) {
          atomicMin(&s_lo[v][ax], lo[v][ax]);
          atomicMax(&s_hi[v][ax], hi[v][ax]);
        }
  }
  __syncthreads();
  int W[3] = {1, 1, 1}, lo[3] = {0, 0, 0}, T[3] = {0, 0, 0};
  bool fit = true;
#pragma unroll
  for (int ax = 0; ax < DIM; ax++) {
    // the deposit reaches cells -2 .. +2; a window wider than the period
    // holds some mesh cells twice: each copy is flushed with its own add,
    // so the sums stay exact
    const int wa = s_hi[0][ax] - s_lo[0][ax] + 5, wb = s_hi[1][ax] - s_lo[1][ax] + 5;
    const int v = wb < wa ? 1 : 0;
    lo[ax] = s_lo[v][ax];
    W[ax] = v ? wb : wa;
    T[ax] = Tof(ax, v);
  }
  auto rel = [&](int ax, int c) { return relT(ax, c, T[ax]); };
  // the product in 64 bits: a spread-out chunk can span most of the grid
  const int64_t cells64 = (int64_t)W[0] * W[1] * W[2];
  // 2D windows also hold Rho; in 3D, Rho (deposited on output steps only)
  // goes to HBM so the window holds J alone: two workgroups per CU
  const int nq = 3 + (rho && DIM == 2 ? (nsp < 4 ? nsp : 4) : 0);
  fit = fit && cells64 * 2 * nq <= WCAP;
  const int cells = fit ? (int)cells64 : 0;
  if (fit)
    for (int e = tid; e < 2 * nq * cells; e += 256) win[e] = 0;
  __syncthreads();
  unsigned global_pushes = 0;
#pragma unroll 1
  for (int k = 0; k < K; k++) {
    if (cl[k] == MAX_CELL) continue;
    const uint64_t idx = first + (uint64_t)R * k;
    int c[3];
    m.split(cl[k], c[0], c[1], c[2]);
    const DepGlobal g{m, a, H, c[0], c[1], c[2]};
    if (fit) {
      int b = 0;
#pragma unroll
      for (int ax = DIM - 1; ax >= 0; ax--) b = b * W[ax] + (rel(ax, c[ax]) - lo[ax] + 2);
      const DepWindow w{win, cells, W[0], W[0] * W[1], b, H, nq, g};
      push_deposit_f64<DIM>(m, sp, dt, rho, p, f, counters, idx, c[0], c[1], c[2], w);
    } else {
      push_deposit_f64<DIM>(m, sp, dt, rho, p, f, counters, idx, c[0], c[1], c[2], g);
      global_pushes++;
    }
  }
  if (!fit) {
    if (global_pushes) atomicAdd(&counters[CTR_GLOBAL_DEP], (unsigned long long)global_pushes);
    return;
  }
  __syncthreads();
  // flush: element e = (2 q + limb) cells + window cell
  for (int e = tid; e < 2 * nq * cells; e += 256) {
    const long long v = win[e];
    if (v == 0) continue;
    const int ql = e / cells, cc = e - ql * cells;
    const int w0 = cc % W[0], w12 = cc / W[0];
    const int w1 = w12 % W[1], w2 = w12 / W[1];
    const int u0 = fold_axis(m, 0, r[0] + lo[0] - 2 + w0);
    const int u1 = DIM > 1 ? fold_axis(m, 1, r[1] + lo[1] - 2 + w1) : r[1];
    const int u2 = DIM > 2 ? fold_axis(m, 2, r[2] + lo[2] - 2 + w2) : r[2];
    __hip_atomic_fetch_add(s_dst[ql] + m.idx(u0, u1, u2), v, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
  }
}

// The two taps of an axis whose weights are not exactly zero, with the weights
// interp_cell gives them (0 <= x <= 1).
__device__ __forceinline__ void two_taps(double x, int c, int st, int &t, double &w0,
                                         double &w1) {
  t = (st || x < 0.5) ? c - 1 : c;
  w0 = interp_cell(x, c, t, st);
  w1 = interp_cell(x, c, t + 1, st);
}

// gather_f64 without the taps of zero weight: 2, 4 or 8 of 3, 9 or 27.  A tap
// of zero weight adds +-0 to a sum that starts at +0, so for finite fields the
// result is the same bit for bit.
template <int DIM>
__device__ __forceinline__ void gather_two_taps(const Mesh &m, const FieldsF64 &f, double x1,
                                                double x2, double x3, int c1, int c2, int c3,
                                                double F[6]) {
  constexpr int st[6] = {ST_E1, ST_E2, ST_E3, ST_B1, ST_B2, ST_B3};
  // per axis, the taps of both staggers
  int t1[2], t2[2] = {0, 0}, t3[2] = {0, 0};
  double w1[2][2], w2[2][2], w3[2][2];
#pragma unroll
  for (int q = 0; q < 2; q++) {
    two_taps(x1, c1, q, t1[q], w1[q][0], w1[q][1]);
    if (DIM > 1) two_taps(x2, c2, q, t2[q], w2[q][0], w2[q][1]);
    if (DIM > 2) two_taps(x3, c3, q, t3[q], w3[q][0], w3[q][1]);
  }
  const int64_t d0 = m.dims[0], d01 = (int64_t)m.dims[0] * m.dims[1];
#pragma unroll
  for (int q = 0; q < 6; q++) {
    const int a = st[q] & 1, b = (st[q] >> 1) & 1, c = (st[q] >> 2) & 1;
    const double *g = (q < 3 ? f.E[q] : f.B[q - 3]) + t1[a];
    if (DIM > 1) g += t2[b] * d0;
    if (DIM > 2) g += t3[c] * d01;
    double r = 0.0;
#pragma unroll
    for (int kk = 0; kk < (DIM > 2 ? 2 : 1); kk++)
#pragma unroll
      for (int jj = 0; jj < (DIM > 1 ? 2 : 1); jj++)
#pragma unroll
        for (int ii = 0; ii < 2; ii++) {
          const double v = g[ii + jj * d0 + kk * d01] * w1[a][ii];
          r += DIM == 1 ? v : DIM == 2 ? v * w2[b][jj] : v * w2[b][jj] * w3[c][kk];
        }
    F[q] = r;
  }
}

// Whether every field value that the taps of particles inside a tile's window
// can touch is finite (uniform; ends with a barrier).  Along each axis the
// window's cells [w + 1, w + W - 2] and, on a periodic axis, their images a
// period away, all within the bulk and one guard cell.
template <int DIM>
__device__ __forceinline__ bool window_finite(const Mesh &m, const FieldsF64 &f, const int w[3],
                                              const int W[3], uint32_t *s_bad) {
  int base[3][3], len[3][3], n[3];
#pragma unroll
  for (int d = 0; d < 3; d++) {
    n[d] = 1;
    base[d][0] = d < DIM ? 0 : w[d];
    len[d][0] = 1;
    if (d >= DIM) continue;
    const int lo = m.guard[d] - 1, hi = m.guard[d] + m.N[d];
    n[d] = 0;
#pragma unroll
    for (int q = 0; q < 3; q++) {
      const int off = m.periodic[d] ? (q == 0 ? 0 : q == 1 ? m.N[d] : -m.N[d]) : 0;
      const int b = max(w[d] + 1 + off, lo), e = min(w[d] + W[d] - 2 + off, hi);
      base[d][q] = b;
      len[d][q] = (q > 0 && off == 0) || e < b ? 0 : e - b + 1;
      n[d] += len[d][q];
    }
    if (n[d] > hi - lo + 1) {  // an axis shorter than the window: all of it
      base[d][0] = lo;
      len[d][0] = n[d] = hi - lo + 1;
    }
  }
  auto at = [&](int d, int e) {
    if (d >= DIM) return base[d][0];
    if (e < len[d][0]) return base[d][0] + e;
    e -= len[d][0];
    return e < len[d][1] ? base[d][1] + e : base[d][2] + (e - len[d][1]);
  };
  if (threadIdx.x == 0) *s_bad = 0;
  __syncthreads();
  bool bad = false;
  for (int e = threadIdx.x; e < n[0] * n[1] * n[2]; e += blockDim.x) {
    const int r = e / n[0];
    const uint64_t o = m.idx(at(0, e - r * n[0]), DIM > 1 ? at(1, r % n[1]) : base[1][0],
                             DIM > 2 ? at(2, r / n[1]) : base[2][0]);
#pragma unroll
    for (int c = 0; c < 3; c++) bad = bad || !isfinite(f.E[c][o]) || !isfinite(f.B[c][o]);
  }
  if (bad) *s_bad = 1;
  __syncthreads();
  return *s_bad == 0;
}

// Deposit into an LDS window: e0 is the element of the particle's cell, limb
// arrays are WN elements apart, rows W0 and planes W01.  Adds of zero are
// issued too: they cost less than the branches around them.
template <int WN, int W0, int W01>
struct DepTile {
  unsigned long long *e0;
  int H;
  __device__ __forceinline__ void add(int q, int o, double v) const {
    long long h, l;
    fx_split(v, H, h, l);
    __hip_atomic_fetch_add(e0 + 2 * q * WN + o, (unsigned long long)h, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WORKGROUP);
    __hip_atomic_fetch_add(e0 + (2 * q + 1) * WN + o, (unsigned long long)l, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WORKGROUP);
  }
};

// deposit_loops_f64 unrolled over the three nodes i0, i0 + 1, i0 + 2 of each
// axis (the third only where the particle crossed), its shape factors and
// centred products evaluated once: the same expressions in the same order of
// summation, so the same bits.  Rho of species past the window's goes to HBM.
template <int DIM, int NQ, bool RHO, class Win>
__device__ __forceinline__ void deposit_unrolled_f64(const Moved &mv, Win d, const DepGlobalL &g,
                                                     int W0, int W01) {
  double s0[DIM][3], s1[DIM][3];
  int n0[DIM];
  bool third[DIM];
#pragma unroll
  for (int a = 0; a < DIM; a++) {
    const int dc = mv.dc[a];
    n0[a] = dc == -1 ? -2 : -1;
    third[a] = dc == -1 || dc == 1;
#pragma unroll
    for (int t = 0; t < 3; t++) {
      const int i = n0[a] + t;
      s0[a][t] = cic(-mv.old_x[a] + i + 1);
      s1[a][t] = cic(-mv.new_x[a] + (i + 1 - dc));
    }
  }
  const double weight = mv.weight;
  auto charge = [&](int i, int j, int k, int o, double v) {
    if (NQ >= 5 && mv.s < 2)
      d.add(3 + mv.s, o, v);
    else
      g.add(3 + mv.s, n0[0] + i, n0[1] + j, DIM > 2 ? n0[DIM - 1] + k : 0, v);
  };
  if constexpr (DIM == 2) {
    d.e0 += n0[0] + W0 * n0[1];
    double djy[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int j = 0; j < 3; j++) {
      if (j == 2 && !third[1]) continue;
      double djx = 0.0;
#pragma unroll
      for (int i = 0; i < 3; i++) {
        if (i == 2 && !third[0]) continue;
        const int o = i + W0 * j;
        djx += movement2d(s0[1][j], s1[1][j], s0[0][i], s1[0][i]);
        d.add(0, o + 1, weight * djx);
        djy[i] += movement2d(s0[0][i], s1[0][i], s0[1][j], s1[1][j]);
        d.add(1, o + W0, weight * djy[i]);
        d.add(2, o, -weight * mv.v3 * center2d(s0[0][i], s1[0][i], s0[1][j], s1[1][j]));
        if (RHO) charge(i, j, 0, o, -weight * (s1[0][i] * s1[1][j]));
      }
    }
  } else {
    d.e0 += n0[0] + W0 * n0[1] + W01 * n0[2];
    double cxy[3][3], djz[3][3];
#pragma unroll
    for (int j = 0; j < 3; j++)
#pragma unroll
      for (int i = 0; i < 3; i++) {
        cxy[j][i] = center2d(s0[0][i], s1[0][i], s0[1][j], s1[1][j]);
        djz[j][i] = 0.0;
      }
#pragma unroll
    for (int k = 0; k < 3; k++) {
      if (k == 2 && !third[2]) continue;
      double cxz[3], djy[3] = {0.0, 0.0, 0.0};
#pragma unroll
      for (int i = 0; i < 3; i++) cxz[i] = center2d(s0[0][i], s1[0][i], s0[2][k], s1[2][k]);
#pragma unroll
      for (int j = 0; j < 3; j++) {
        if (j == 2 && !third[1]) continue;
        const double cyz = center2d(s0[1][j], s1[1][j], s0[2][k], s1[2][k]);
        double djx = 0.0;
#pragma unroll
        for (int i = 0; i < 3; i++) {
          if (i == 2 && !third[0]) continue;
          const int o = i + W0 * j + W01 * k;
          djx += (s1[0][i] - s0[0][i]) * cyz;
          d.add(0, o + 1, weight * djx);
          djy[i] += (s1[1][j] - s0[1][j]) * cxz[i];
          d.add(1, o + W0, weight * djy[i]);
          djz[j][i] += (s1[2][k] - s0[2][k]) * cxy[j][i];
          d.add(2, o + W01, weight * djz[j][i]);
          if (RHO) charge(i, j, k, o, -weight * (s1[0][i] * s1[1][j] * s1[2][k]));
        }
      }
    }
  }
}

// Tile shapes of the update over cell runs: cells per tile, halo, threads,
// copies of the window, slots per lane run, waves per SIMD compiled for.
// The window is 48 B per cell (three components of two limbs), so the tile is
// what leaves two or more workgroups per CU beside a halo that holds most of a
// sort interval's drift.  Measured, us per push: 640 x 480 cells at 24 per cell
// 16 x 16 + 8 with 512 threads 466 (256 threads 549, 8 x 8 + 8 477, 16 x 16 + 6
// 840); 64 x 48 x 50 at 8 per cell 8 x 4 x 4 + 3 255 (+ 4 268, 4^3 + 3 285, 8^3
// + 3 368); 1D, 4096 cells at 200 per cell, 16 + 16 with 8 window copies 37.
#ifndef F64R1
#define F64R1 16, 1, 1, 16, 256, 8, 8, 4
#endif
#ifndef F64R2
#define F64R2 16, 16, 1, 8, 512, 1, 16, 4
#endif
#ifndef F64R3
#define F64R3 8, 4, 4, 3, 256, 1, 8, 2
#endif
template <int A, int B, int C, int HH, int TH, int NC, int RL, int WV>
struct F64Shape {
  static constexpr int T0 = A, T1 = B, T2 = C, H = HH, NT = TH, COPIES = NC, R = RL;
  static constexpr int WAVES = WV;
};
template <int DIM>
struct F64RunShape;
template <>
struct F64RunShape<1> : F64Shape<F64R1> {};
template <>
struct F64RunShape<2> : F64Shape<F64R2> {};
template <>
struct F64RunShape<3> : F64Shape<F64R3> {};

void f64_runs_tile(int dim, int T[3]) {
  T[0] = dim == 1 ? F64RunShape<1>::T0 : dim == 2 ? F64RunShape<2>::T0 : F64RunShape<3>::T0;
  T[1] = dim == 1 ? F64RunShape<1>::T1 : dim == 2 ? F64RunShape<2>::T1 : F64RunShape<3>::T1;
  T[2] = dim == 1 ? F64RunShape<1>::T2 : dim == 2 ? F64RunShape<2>::T2 : F64RunShape<3>::T2;
}

// As mixed_runs_pay, against the update of chunks of consecutive slots (us per
// push, that one / this one): 1D, 62,500 tiles, 16 slots a tile 319 / 576, 32
// 607 / 637, 64 1208 / 723; 2D, 65,536 tiles, 13 1398 / 2745, 64 3366 / 2977, but
// 4096 tiles, 13 217 / 155 (the chunks then are too few to fill the chip); 3D,
// 131,072 tiles, 6 2034 / 7001, 32 6164 / 7870, 16,384 tiles, 64 1654 / 1449.
bool f64_runs_pay(int dim, uint64_t kept, uint32_t items) {
  const uint64_t least = dim == 1 ? 40 : dim == 2 ? 48 : 64;
  return items <= (dim == 2 ? 4096u : 1024u) || kept >= least * items;
}

// The FP64 update of cell-sorted slots: one workgroup per tile (or share of a
// tile), the tile's current -- and, RHO, the charge of two species -- summed
// in an LDS window over the tile and a halo that holds the drift of a sort
// interval, flushed once per element.  The windows above follow a chunk of
// consecutive slots, a thin strip of a row, and stop fitting once the
// particles have drifted a few rows; a tile's window does not depend on the
// particles per cell.  A wave's lanes take 64 / R runs of R consecutive slots
// spread over the share, so neighbouring lanes read whole cache lines while
// the wave's atomics fall on many cells; in 1D, where a tile is a few cells
// wide, lanes also alternate between copies of the window.  Particles outside
// the window deposit straight to HBM (counted).  The slots of guard rows are
// k_push_guard_rows_f64's.
template <int DIM, bool RHO>
__attribute__((amdgpu_waves_per_eu(F64RunShape<DIM>::WAVES))) __global__ void
    __launch_bounds__(F64RunShape<DIM>::NT) k_push_deposit_f64_runs(Mesh m, Species sp, double dt, int H, PtcF64 p, FieldsF64 f, AccF64 a,
                            CellRuns cr, unsigned long long *__restrict__ counters) {
  using S = F64RunShape<DIM>;
  constexpr int NT = S::NT, HW = S::H, R = S::R, NC = S::COPIES;
  constexpr int W0 = S::T0 + 2 * HW, W1 = DIM > 1 ? S::T1 + 2 * HW : 1;
  constexpr int W2 = DIM > 2 ? S::T2 + 2 * HW : 1, WN = W0 * W1 * W2;
  // 3D: the window holds the current alone; Rho, on output steps, goes to HBM
  constexpr int NQ = 3 + (RHO && DIM < 3 ? 2 : 0), ROWS = S::T1 * S::T2;
  static_assert(64 % R == 0 && 64 % NC == 0, "lane runs and copies divide the wave");
  using Win = DepTile<WN, W0, W0 * W1>;
  __shared__ unsigned long long win[NC * 2 * NQ * WN];
  __shared__ RunWalk<ROWS> walk;
  constexpr int QCAP = 512;
  __shared__ uint32_t s_queue[QCAP];
  __shared__ uint32_t s_bad, s_nq;
  __shared__ long long *s_dst[14];
  __shared__ double s_qdt[8], s_q[8];  // dt q / 2m and q per species
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  uint32_t tile, part, parts;
  if (!run_item(cr, blockIdx.x, tile, part, parts)) return;  // uniform
  for (int e = tid; e < NC * 2 * NQ * WN; e += NT) win[e] = 0;
  if (tid == 0) s_nq = 0;
  if (tid < 14) s_dst[tid] = tid < 6 ? a.J[tid >> 1][tid & 1] : a.R[(tid - 6) >> 1][tid & 1];
  if (tid < 8) {
    s_qdt[tid] = sp.qdt[tid];
    s_q[tid] = sp.q[tid];
  }
  int org[3];
  uint32_t lo, hi;
  walk.open(m, cr, tile, part, parts, org, lo, hi);
  if (lo == hi) return;  // uniform
  const int w[3] = {org[0] - HW, DIM > 1 ? org[1] - HW : org[1],
                    DIM > 2 ? org[2] - HW : org[2]};
  const int WD[3] = {W0, W1, W2};
  const bool finite = window_finite<DIM>(m, f, w, WD, &s_bad);
  const uint32_t cnt = hi - lo;
  constexpr uint32_t G = 64 / R;
  const uint32_t seg = ((cnt + G - 1) / G + R - 1) / R * R;
  unsigned long long *const mine = win + (lane & (NC - 1)) * 2 * NQ * WN;
  unsigned outside = 0;
  // Two passes of one loop: the tile's particles, then those found outside the
  // window (queued, so that a wave does not run the HBM path for a lane or
  // two; past the queue's end they take it at once).  The next particle is
  // requested before the current one is processed.
#pragma unroll 1
  for (int pass = 0; pass < 2; pass++) {
  if (pass) __syncthreads();
  const uint32_t limit = pass ? min(s_nq, (uint32_t)QCAP) : seg;
  const uint32_t step = pass ? (uint32_t)NT : (uint32_t)(NT / 64) * R;
  auto locate = [&](uint32_t k, uint32_t &i) -> bool {  // lanes past the end: a valid slot
    if (pass) {
      const bool ok = k + lane < limit;
      i = s_queue[ok ? k + lane : 0];
      return ok;
    }
    const uint32_t kk = k + (uint32_t)(lane % R), q = (uint32_t)(lane / R) * seg + kk;
    const bool ok = kk < seg && q < cnt;
    i = walk.slot(ok ? lo + q : lo);
    return ok;
  };
  uint32_t i_nxt = 0;
  Ptc64Regs r_nxt;
  bool ok_nxt = false;
  uint32_t k = pass ? (uint32_t)wv * 64 : (uint32_t)wv * R;
  if (k < limit) {
    ok_nxt = locate(k, i_nxt);
    load_ptc64(p, i_nxt, r_nxt);
  }
#pragma unroll 1
  for (; k < limit; k += step) {
    const Ptc64Regs r = r_nxt;
    const uint64_t idx = i_nxt;
    const bool ok = ok_nxt;
    if (k + step < limit) {
      ok_nxt = locate(k + step, i_nxt);
      load_ptc64(p, i_nxt, r_nxt);
    }
    const uint32_t c = r.cell;
    if (!ok || c == MAX_CELL) continue;
    int c1, c2, c3;
    m.split(c, c1, c2, c3);
    if (!m.in_bulk(c1, c2, c3)) {
      p.cell[idx] = MAX_CELL;
      continue;
    }
    const int l0 = window_coord<W0>(c1, w[0], m.N[0], m.periodic[0]);
    const int l1 = DIM > 1 ? window_coord<W1>(c2, w[1], m.N[1], m.periodic[1]) : 0;
    const int l2 = DIM > 2 ? window_coord<W2>(c3, w[2], m.N[2], m.periodic[2]) : 0;
    bool in = l0 >= 2 && l0 <= W0 - 3;
    if (DIM > 1) in = in && l1 >= 2 && l1 <= W1 - 3;
    if (DIM > 2) in = in && l2 >= 2 && l2 <= W2 - 3;
    if (!in && pass == 0) {
      outside++;
      const uint32_t q = atomicAdd(&s_nq, 1u);
      if (q < QCAP) {
        s_queue[q] = (uint32_t)idx;
        continue;
      }
    }
    const Win dep{mine + (in ? l0 + W0 * (l1 + W1 * l2) : 0), H};
    const DepGlobalL g{m, s_dst, H, c1, c2, c3};
    auto gather = [&](double x1, double x2, double x3, double F[6]) {
      bool two = finite && in && x1 >= 0.0 && x1 <= 1.0;
      if (DIM > 1) two = two && x2 >= 0.0 && x2 <= 1.0;
      if (DIM > 2) two = two && x3 >= 0.0 && x3 <= 1.0;
      if (two)
        gather_two_taps<DIM>(m, f, x1, x2, x3, c1, c2, c3, F);
      else
        gather_f64<DIM>(m, f, x1, x2, x3, c1, c2, c3, F);
    };
    if constexpr (DIM == 1) {
      int s, dc1;
      bool on;
      double weight, old_x1, new_x1, v2, v3;
      push_move_1d_f64(
          m, s_qdt, s_q, dt, p, [&](double x1, double F[6]) { gather(x1, 0.0, 0.0, F); }, counters, idx,
          r, s, on, weight, old_x1, new_x1, dc1, v2, v3);
      if (!on) continue;
      // deposit_current_cart_1d (ptc_updater.cu:220-293)
      const int i0 = (dc1 == -1 ? -2 : -1);
      const bool third = dc1 == -1 || dc1 == 1;
      double djx = 0.0;
#pragma unroll
      for (int t = 0; t < 3; t++) {
        if (t == 2 && !third) continue;
        const int i = i0 + t;
        const double sx0 = cic(-old_x1 + i + 1);
        const double sx1 = cic(-new_x1 + (i + 1 - dc1));
        djx += sx1 - sx0;
        const double val1 = 0.5 * (sx0 + sx1);
        auto put = [&](int q, int o, double v) {
          if (in && q < NQ) dep.add(q, o, v);
          else g.add(q, o, 0, 0, v);
        };
        put(0, i + 1, -weight * djx);
        put(1, i, weight * v2 * val1);
        put(2, i, weight * v3 * val1);
        if (RHO) put(3 + s, i, weight * sx1);
      }
    } else {
      Moved mv;
      push_move_f64<DIM>(m, s_qdt, s_q, dt, p, counters, idx, r, c1, c2, c3, gather, mv);
      if (!mv.on) continue;
      if (in)
        deposit_unrolled_f64<DIM, NQ, RHO>(mv, dep, g, W0, W0 * W1);
      else
        deposit_loops_f64<DIM>(mv, RHO ? 1 : 0, g);
    }
  }
  }  // passes
  if (outside) atomicAdd(&counters[CTR_GLOBAL_DEP], (unsigned long long)outside);
  __syncthreads();
  for (int e = tid; e < 2 * NQ * WN; e += NT) {
    unsigned long long v = 0;
#pragma unroll
    for (int cpy = 0; cpy < NC; cpy++) v += win[cpy * 2 * NQ * WN + e];
    if (v == 0) continue;
    const int ql = e / WN, cc = e - ql * WN;
    const int u0 = fold_axis(m, 0, w[0] + cc % W0);
    const int u1 = DIM > 1 ? fold_axis(m, 1, w[1] + cc / W0 % W1) : w[1];
    const int u2 = DIM > 2 ? fold_axis(m, 2, w[2] + cc / (W0 * W1)) : w[2];
    __hip_atomic_fetch_add((unsigned long long *)s_dst[ql] + m.idx(u0, u1, u2), v, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
  }
}

// The slots that a sort left in guard rows, which belong to no tile (none on a
// periodic mesh: not launched then).  Each is judged by its own cell, not by the
// row it was sorted into: a recorded step may be replayed on particles that were
// set since.
template <int DIM>
__global__ void __launch_bounds__(64)
    k_push_guard_rows_f64(Mesh m, Species sp, double dt, int H, int rho, PtcF64 p, FieldsF64 f,
                          AccF64 a, CellRuns cr, unsigned long long *__restrict__ counters) {
  for_guard_row_slots(m, cr, [&](uint32_t idx) {
    const uint32_t c = p.cell[idx];
    if (c == MAX_CELL) return;
    int c1, c2, c3;
    m.split(c, c1, c2, c3);
    if (!m.in_bulk(c1, c2, c3)) {
      p.cell[idx] = MAX_CELL;
      return;
    }
    push_deposit_f64<DIM>(m, sp, dt, rho, p, f, counters, idx, c1, c2, c3,
                          DepGlobal{m, a, H, c1, c2, c3});
    atomicAdd(&counters[CTR_GLOBAL_DEP], 1ull);
  });
}

// J = hi 2^-H + lo 2^-(H+40), accumulators cleared for the next step.
__global__ void k_finalize_f64(long long *__restrict__ hi,
                               long long *__restrict__ lo,
                               double *__restrict__ out, uint64_t n, int H) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  out[i] = fx_value(hi[i], lo[i], H);
  hi[i] = 0;
  lo[i] = 0;
}

// ---------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------
hipError_t launch_push_deposit_f64(const Mesh &m, const Species &sp,
                                   double dt, int H, int rho, int nsp,
                                   const PtcF64 &p, const FieldsF64 &f,
                                   const AccF64 &a,
                                   unsigned long long *counters, uint64_t n,
                                   hipStream_t st) {
  if (n == 0) return hipSuccess;
  dim3 block(256);
  Species spd = sp;
  for (int i = 0; i < 8; i++) spd.qdt[i] = dt * 0.5 * sp.q[i] / sp.m[i];
  if (m.dim == 1) {
    k_push_deposit_f64<1><<<(unsigned)((n + 255) / 256), block, 0, st>>>(m, spd, dt, H, rho, p,
                                                                         f, a, counters, n);
  } else if (m.dim == 2) {
    // 2048 slots per workgroup: ~32 cells of a row at 64 particles per cell
    constexpr int R = F64_WIN2_R, K = F64_WIN2_K;
    k_push_deposit_f64_win<2, R, K, F64_WIN2_CAP, F64_WIN2_WAVES>
        <<<(unsigned)((n + 256 * K - 1) / (256 * K)), block, 0, st>>>(m, spd, dt, H, rho, nsp, p,
                                                                      f, a, counters, n);
  } else {
    constexpr int R = F64_WIN3_R, K = F64_WIN3_K;
    k_push_deposit_f64_win<3, R, K, F64_WIN3_CAP, F64_WIN3_WAVES>
        <<<(unsigned)((n + 256 * K - 1) / (256 * K)), block, 0, st>>>(m, spd, dt, H, rho, nsp, p,
                                                                      f, a, counters, n);
  }
  return hipGetLastError();
}

hipError_t launch_push_deposit_f64_runs(const Mesh &m, const Species &sp, double dt, int H,
                                        int rho, const PtcF64 &p, const FieldsF64 &f,
                                        const AccF64 &a, const CellRuns &cr,
                                        unsigned long long *counters, hipStream_t st) {
  if (cr.end == 0) return hipSuccess;
  Species spd = sp;
  for (int i = 0; i < 8; i++) spd.qdt[i] = dt * 0.5 * sp.q[i] / sp.m[i];
  auto go = [&](auto kern, int NT) {
    kern<<<cr.items, NT, 0, st>>>(m, spd, dt, H, p, f, a, cr, counters);
    return hipGetLastError();
  };
  if (cr.guard_slots > 0 && m.dim > 1) {
    if (m.dim == 2)
      k_push_guard_rows_f64<2><<<guard_row_blocks(m), 64, 0, st>>>(m, spd, dt, H, rho, p, f, a, cr,
                                                                   counters);
    else
      k_push_guard_rows_f64<3><<<guard_row_blocks(m), 64, 0, st>>>(m, spd, dt, H, rho, p, f, a, cr,
                                                                   counters);
  }
  if (m.dim == 1)
    return rho ? go(k_push_deposit_f64_runs<1, true>, F64RunShape<1>::NT)
               : go(k_push_deposit_f64_runs<1, false>, F64RunShape<1>::NT);
  if (m.dim == 2)
    return rho ? go(k_push_deposit_f64_runs<2, true>, F64RunShape<2>::NT)
               : go(k_push_deposit_f64_runs<2, false>, F64RunShape<2>::NT);
  return rho ? go(k_push_deposit_f64_runs<3, true>, F64RunShape<3>::NT)
             : go(k_push_deposit_f64_runs<3, false>, F64RunShape<3>::NT);
}

hipError_t launch_finalize_f64(long long *hi, long long *lo, double *out,
                               uint64_t n, int H, hipStream_t st) {
  dim3 block(256), grid((unsigned)((n + 255) / 256));
  k_finalize_f64<<<grid, block, 0, st>>>(hi, lo, out, n, H);
  return hipGetLastError();
}

}  // namespace apt
