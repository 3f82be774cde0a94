// kern_rt.hip -- pair creation and photon transport:
//   * radiative_transfer::emit_photons / produce_pairs
//     (radiative_transfer.cu:28-301) with the reference's default hooks
//     (user_radiative_functions.cu:13-125) and an exponential-free-path
//     model with a fixed photon energy fraction;
//   * move_photons_cart_{1,2,3}d (ptc_updater.cu:627-741) and the
//     log-spherical move_photons (ptc_updater_logsph.cu:58-132).
// Decide -> exclusive scan -> write: the k-th emitting particle (slot order)
// fills photon slot number + k and the k-th converting photon fills
// particle slots number + 2k, 2k+1, replacing the reference's per-block
// atomic counters, so events and their storage order do not depend on the
// launch shape.  Random draws are Philox4x32-10 keyed on (seed, particle
// slot, call epoch).  The one host read per call is the event count, as
// in the reference (radiative_transfer.cu:225-228, 279-282); in a
// context's device-count mode there is none: bases, ids and the epoch are
// read from device memory and the counts updated there.
#include <type_traits>

#include "apt_common.hpp"
#include "apt_kernels.hpp"
#include "apt_sort.hpp"
#include "apt_math.hpp"

namespace apt {

constexpr double RT_PI = 3.14159265358979323846;

template <typename R>
struct RtMath;
template <>
struct RtMath<double> {
  static __device__ double sin(double x) { return apt_sin(x); }
  static __device__ double log(double x) { return apt_log(x); }
  static __device__ double exp(double x) { return apt_exp(x); }
  static __device__ void sincos(double x, double &s, double &c) {
    apt_sincos(x, s, c);
  }
  static __device__ double acos(double t) { return apt_acos(t); }
  static __device__ double atan2(double y, double x) { return apt_atan2(y, x); }
};
template <>
struct RtMath<float> {
  static __device__ float sin(float x) { return sinf(x); }
  static __device__ float log(float x) { return logf(x); }
  static __device__ float exp(float x) { return expf(x); }
  static __device__ void sincos(float x, float &s, float &c) {
    sincosf(x, &s, &c);
  }
  static __device__ float acos(float t) {
    return acosf(fminf(fmaxf(t, -1.0f), 1.0f));
  }
  static __device__ float atan2(float y, float x) { return atan2f(y, x); }
};

// Quadmesh::pos (quadmesh.h:144-150), including the collapsed dimensions
__device__ inline double rt_pos(const Mesh &m, int d, int n, double x) {
  if (d < m.dim) return m.lower[d] + m.delta[d] * ((double)(n - m.guard[d]) + x);
  return x * m.delta[d];
}

template <typename R>
__device__ inline R ptc_gamma(const PtcView<R> &p, uint64_t i) {
  if (p.E) return p.E[i];
  R a = p.p1[i], b = p.p2[i], c = p.p3[i];
  return sqrt((R)1 + a * a + b * b + c * c);
}

// count_photon_produced: the emit decision (check_emit_photon) and the
// emitter's weight added to photon_produced of its cell
// (radiative_transfer.cu:48-57)
template <typename R>
__device__ inline uint32_t emit_decision(const Mesh &m, const RtParams &rt, const PtcView<R> &p,
                                         uint64_t i, R *produced) {
  uint32_t c = p.cell[i], f = 0;
  if (c != MAX_CELL) {
    int c1, c2, c3;
    m.split(c, c1, c2, c3);
    if (m.in_bulk(c1, c2, c3) && ptc_species(p.flag[i]) != 2 &&
        ptc_gamma(p, i) > (R)rt.gamma_thr)
      f = 1;
  }
  if (f && produced) atomicAdd(&produced[c], p.w[i]);
  return f;
}

// produce_photons + emit_photon for emitter i, the k-th emitter of the pass
template <typename R>
__device__ inline void emit_one(const Mesh &m, const RtParams &rt, const PtcView<R> &p,
                                const PhoView<R> &ph, uint64_t i, uint64_t k, uint64_t base,
                                uint64_t seed, uint32_t epoch, uint64_t id_base) {
  using M = RtMath<R>;
  const uint64_t slot = base + k;
  ph.cell[slot] = MAX_CELL;
  if (ph.id) ph.id[slot] = id_base + (slot - base);
  double u0, u1;
  uniform2(seed, i, epoch, 5, u0, u1);
  const uint32_t c = p.cell[i];
  const R gamma = ptc_gamma(p, i);
  const R p1 = p.p1[i], p2 = p.p2[i], p3 = p.p3[i];
  const R pi = sqrt(gamma * gamma - (R)1);
  R Eph;
  if (rt.model == 0)
    Eph = (R)2.5 + (R)u0 * ((R)rt.E_secondary - (R)1) * (R)2;
  else
    Eph = (R)rt.e_frac * gamma;
  const R ge = gamma - Eph;
  const R pf2 = ge * ge - (R)1;
  const R pf = sqrt(pf2 > (R)0 ? pf2 : (R)0);
  p.p1[i] = p1 * pf / pi;
  p.p2[i] = p2 * pf / pi;
  p.p3[i] = p3 * pf / pi;
  if (p.E) p.E[i] = ge;
  R path;
  if (rt.model == 0) {
    int c1, c2, c3;
    m.split(c, c1, c2, c3);
    const R theta = (R)rt_pos(m, 1, c2, (double)p.x2[i]);
    R lph = ((R)1 / M::sin(theta) - (R)1) * (R)rt.photon_path;
    if (lph > (R)10) lph = (R)10;
    if (theta < (R)0.005 || theta > (R)(RT_PI - 0.005)) return;
    path = lph * ((R)0.5 + (R)0.5 * (R)u1);
  } else {
    path = -(R)rt.photon_path * M::log((R)u1);
  }
  if (path > (R)rt.r_cutoff) return;
  ph.x1[slot] = p.x1[i];
  ph.x2[slot] = p.x2[i];
  ph.x3[slot] = p.x3[i];
  ph.p1[slot] = Eph * p1 / pi;
  ph.p2[slot] = Eph * p2 / pi;
  ph.p3[slot] = Eph * p3 / pi;
  if (ph.E) ph.E[slot] = Eph;
  ph.w[slot] = p.w[i];
  ph.path[slot] = path;
  ph.flag[slot] = 0;
  ph.cell[slot] = c;
}

// count_pairs_produced: check_produce_pair, and the photon's weight added
// to pair_produced of its cell (radiative_transfer.cu:120-130)
template <typename R>
__device__ inline uint32_t pair_decision(const Mesh &m, const PhoView<R> &ph, uint64_t t,
                                         R *produced) {
  uint32_t c = ph.cell[t], f = 0;
  if (c != MAX_CELL) {
    int c1, c2, c3;
    m.split(c, c1, c2, c3);
    if (m.in_bulk(c1, c2, c3) && ph.path[t] <= (R)0) f = 1;
  }
  if (f && produced) atomicAdd(&produced[c], ph.w[t]);
  return f;
}

// produce_pairs + produce_pair for photon t, the k-th converting photon of
// the pass; its pair goes to slots base + 2k, base + 2k + 1
template <typename R>
__device__ inline void pair_one(const PtcView<R> &p, const PhoView<R> &ph, uint64_t t,
                                uint64_t k, uint64_t base, uint64_t id_base) {
  const uint64_t off = base + 2 * k;
  const R p1 = ph.p1[t], p2 = ph.p2[t], p3 = ph.p3[t];
  R E_ph2 = p1 * p1 + p2 * p2 + p3 * p3;
  if (E_ph2 <= (R)4.01) E_ph2 = (R)4.01;
  const R ratio = sqrt((R)0.25 - (R)1 / E_ph2);
  const R gamma = sqrt((R)1 + ratio * ratio * E_ph2);
  const uint32_t c = ph.cell[t];
  for (int s = 0; s < 2; s++) {
    const uint64_t o = off + s;
    p.x1[o] = ph.x1[t];
    p.x2[o] = ph.x2[t];
    p.x3[o] = ph.x3[t];
    p.p1[o] = ratio * p1;
    p.p2[o] = ratio * p2;
    p.p3[o] = ratio * p3;
    if (p.E) p.E[o] = gamma;
    p.w[o] = ph.w[t];
    p.flag[o] = FLAG_SECONDARY | ((uint32_t)s << 29);
    if (p.id) p.id[o] = id_base + 2 * k + s;
    p.cell[o] = c;
  }
  ph.cell[t] = MAX_CELL;
}

// ---------------------------------------------------------------------
// An event pass over the slots below a count, on the host or on the device
// (device-count mode, where the host only holds an upper bound n).  Workgroups
// of EV_T threads own EV_T E consecutive slots; a workgroup wholly past the
// count exits at once.  Pass 1 stores the 0/1 decisions and each workgroup's
// event count; one workgroup turns the counts into exclusive prefixes (the
// total after the last); pass 2 ranks each event within its workgroup
// (ballots, slot order) on top of the prefix.  The k-th event in slot order
// gets rank k.
// A pass is launches and waits: with host counts the total goes straight to
// pinned host memory, so between decision and events there are one launch and
// one wait (a device-wide scan, a total and a copy before: 4 launches, and a
// copy through pageable memory).  E is 4 there, where n is the work (850,000
// slots fill the chip), and 16 under a bound, where most workgroups are empty.
// ---------------------------------------------------------------------
constexpr int EV_T = 256, EV_HOST_E = 4, EV_DEV_E = 16;
constexpr int EV_SCAN_T = 1024;

__host__ __device__ inline uint64_t ev_blocks(uint64_t n, int e) {
  return (n + (uint64_t)EV_T * e - 1) / ((uint64_t)EV_T * e);
}

// this thread's 0/1 flag ranked among the workgroup's (slot order):
// returns the number of set flags on lower threads; *tot the workgroup's
__device__ inline uint32_t ev_rank(uint32_t f, uint32_t *s_w, uint32_t *tot) {
  const unsigned long long b = __ballot(f != 0);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint32_t below = (uint32_t)__popcll(b & ((1ull << lane) - 1ull));
  if (lane == 0) s_w[w] = (uint32_t)__popcll(b);
  __syncthreads();
  uint32_t off = 0, t = 0;
#pragma unroll
  for (int k = 0; k < EV_T / 64; k++) {
    const uint32_t c = s_w[k];
    off += k < w ? c : 0u;
    t += c;
  }
  __syncthreads();  // s_w is written again by the next call
  *tot = t;
  return off + below;
}

template <typename R, bool PHOTONS, int E>
__global__ void __launch_bounds__(EV_T)
    k_ev_flags(Mesh m, RtParams rt, PtcView<R> p, PhoView<R> ph, uint64_t n,
               const unsigned long long *__restrict__ dn, uint32_t *__restrict__ flags,
               R *__restrict__ produced, uint64_t *__restrict__ bsum) {
  __shared__ uint32_t s_n;
  const uint64_t cnt = dev_n(n, dn), b0 = (uint64_t)blockIdx.x * (EV_T * E);
  if (b0 >= cnt) {
    if (threadIdx.x == 0) bsum[blockIdx.x] = 0;
    return;
  }
  if (threadIdx.x == 0) s_n = 0;
  __syncthreads();
  uint32_t mine = 0;
  for (int e = 0; e < E; e++) {
    const uint64_t i = b0 + (uint64_t)e * EV_T + threadIdx.x;
    if (i >= cnt) break;
    const uint32_t f = PHOTONS ? emit_decision(m, rt, p, i, produced)
                               : pair_decision(m, ph, i, produced);
    flags[i] = f;
    mine += f;
  }
  if (mine) atomicAdd(&s_n, mine);
  __syncthreads();
  if (threadIdx.x == 0) bsum[blockIdx.x] = s_n;
}

// exclusive prefixes of the workgroup counts below the count, in place, their
// sum behind them and in *total.  One workgroup; thread t owns a contiguous run.
__global__ void __launch_bounds__(EV_SCAN_T)
    k_ev_scan(uint64_t *__restrict__ bsum, uint64_t n, int E,
              const unsigned long long *__restrict__ dn,
              unsigned long long *__restrict__ total) {
  __shared__ uint64_t s[EV_SCAN_T];
  const uint64_t nb = ev_blocks(dev_n(n, dn), E);
  const uint64_t per = (nb + EV_SCAN_T - 1) / EV_SCAN_T;
  const uint64_t lo = threadIdx.x * per, hi = lo + per < nb ? lo + per : nb;
  uint64_t run = 0;
  for (uint64_t b = lo; b < hi; b++) run += bsum[b];
  s[threadIdx.x] = run;
  __syncthreads();
  for (int d = 1; d < EV_SCAN_T; d <<= 1) {
    const uint64_t v = threadIdx.x >= (unsigned)d ? s[threadIdx.x - d] : 0;
    __syncthreads();
    s[threadIdx.x] += v;
    __syncthreads();
  }
  uint64_t a = s[threadIdx.x] - run;
  for (uint64_t b = lo; b < hi; b++) {
    const uint64_t v = bsum[b];
    bsum[b] = a;
    a += v;
  }
  if (threadIdx.x == EV_SCAN_T - 1) *total = bsum[nb] = s[EV_SCAN_T - 1];
}

// pass 2: the events, with bases, ids and the epoch from the host or from dc
template <typename R, bool PHOTONS, int E>
__global__ void __launch_bounds__(EV_T)
    k_ev_apply(Mesh m, RtParams rt, PtcView<R> p, PhoView<R> ph, uint64_t n,
               const unsigned long long *__restrict__ dn,
               const uint32_t *__restrict__ flags, const uint64_t *__restrict__ bsum,
               uint64_t seed, uint64_t base, uint64_t id_base, uint32_t epoch,
               const unsigned long long *__restrict__ dc,
               unsigned long long *__restrict__ counters) {
  __shared__ uint32_t s_w[EV_T / 64];
  const uint64_t cnt = dev_n(n, dn), b0 = (uint64_t)blockIdx.x * (EV_T * E);
  if (b0 >= cnt) return;  // workgroup-uniform
  if (dc) {
    base = PHOTONS ? dc[DC_PH] : dc[DC_NUM];
    id_base = PHOTONS ? dc[DC_PH_ID] : dc[DC_ID];
    epoch = (uint32_t)dc[DC_RT_EPOCH];
  }
  const uint64_t cap = PHOTONS ? rt.max_photon : rt.max_ptc;
  uint64_t run = bsum[blockIdx.x];
  if (bsum[blockIdx.x + 1] == run) return;  // workgroup-uniform: no event here
  for (int e = 0; e < E; e++) {  // every thread takes every round (barriers)
    const uint64_t i = b0 + (uint64_t)e * EV_T + threadIdx.x;
    const uint32_t f = i < cnt ? flags[i] : 0u;
    uint32_t tot;
    const uint64_t k = run + ev_rank(f, s_w, &tot);
    run += tot;
    if (!f) continue;
    const bool over = PHOTONS ? base + k >= cap : base + 2 * k + 1 >= cap;
    wave_count(&counters[CTR_OVERFLOW], over);
    if (PHOTONS) {
      if (!over) emit_one(m, rt, p, ph, i, k, base, seed, epoch, id_base);
    } else {
      if (over)
        ph.cell[i] = MAX_CELL;
      else
        pair_one(p, ph, i, k, base, id_base);
    }
  }
}

// Device-count mode: the events of an emit (photons = 1) or pair pass
// that got slots, added to the counts, ids and totals on the device; the
// emission epoch advances.  room: photon (or particle) capacity.
__global__ void k_events_finish(const unsigned long long *__restrict__ ptotal, uint64_t cap,
                                int photons, unsigned long long *__restrict__ dc) {
  if (blockIdx.x != 0 || threadIdx.x != 0) return;
  const unsigned long long total = *ptotal;
  unsigned long long made;
  if (photons) {
    const unsigned long long room = cap > dc[DC_PH] ? cap - dc[DC_PH] : 0ull;
    made = total < room ? total : room;
    dc[DC_PH] += made;
    dc[DC_PH_ID] += made;
    dc[DC_EMITTED] += made;
    dc[DC_RT_EPOCH] += 1;
  } else {
    // pairs whose second slot fits: base + 2k + 1 < cap, k < L/2
    const unsigned long long L = cap > dc[DC_NUM] ? cap - dc[DC_NUM] : 0ull;
    made = total < L / 2 ? total : L / 2;
    dc[DC_NUM] += 2 * made;
    dc[DC_ID] += 2 * made;
    dc[DC_CONVERTED] += made;
  }
  dc[DC_LAST] = made;
}

__global__ void k_fill_tail(uint32_t *__restrict__ cell, const unsigned long long *kept,
                            uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && i >= *kept) cell[i] = MAX_CELL;
}

__global__ void k_dc_set(unsigned long long *dc, int which, const unsigned long long *src) {
  if (blockIdx.x == 0 && threadIdx.x == 0) dc[which] = *src;
}

__global__ void k_dc_accum(unsigned long long *dc, int to, int from) {
  if (blockIdx.x == 0 && threadIdx.x == 0) dc[to] += dc[from];
}

// move_photons_cart_{1,2,3}d (ptc_updater.cu:627-741) + periodic wrap
template <typename R>
__device__ inline void move_photon_cart(const Mesh &m, const PhoView<R> &ph, uint64_t t, R dt) {
  const uint32_t c = ph.cell[t];
  if (c == MAX_CELL) return;
  const R p1 = ph.p1[t], p2 = ph.p2[t], p3 = ph.p3[t];
  const R E = sqrt(p1 * p1 + p2 * p2 + p3 * p3);
  const R x1 = ph.x1[t], x2 = ph.x2[t], x3 = ph.x3[t];
  int c1, c2, c3;
  m.split(c, c1, c2, c3);
  int dc[3] = {0, 0, 0};
  R nx[3];
  if (m.dim == 1) {
    nx[0] = x1 + p1 / E * dt * (R)m.inv_delta[0];
    dc[0] = (int)floor(nx[0]);
    nx[0] -= (R)dc[0];
    nx[1] = x2 + p2 * dt / E;
    nx[2] = x3 + p3 * dt / E;
  } else {
    const R v1 = p1 / E, v2 = p2 / E, v3 = p3 / E;
    nx[0] = x1 + v1 * dt * (R)m.inv_delta[0];
    nx[1] = x2 + v2 * dt * (R)m.inv_delta[1];
    dc[0] = (int)floor(nx[0]);
    dc[1] = (int)floor(nx[1]);
    nx[0] -= (R)dc[0];
    nx[1] -= (R)dc[1];
    if (m.dim == 2) {
      nx[2] = x3 + v3 * dt;
    } else {
      nx[2] = x3 + v3 * dt * (R)m.inv_delta[2];
      dc[2] = (int)floor(nx[2]);
      nx[2] -= (R)dc[2];
    }
  }
  if (dc[0] < -1 || dc[0] > 1 || dc[1] < -1 || dc[1] > 1 || dc[2] < -1 ||
      dc[2] > 1) {
    ph.cell[t] = MAX_CELL;
    return;
  }
  int n1 = c1 + dc[0], n2 = c2 + dc[1], n3 = c3 + dc[2];
  if (m.dim >= 1) n1 = m.wrap(0, n1);
  if (m.dim >= 2) n2 = m.wrap(1, n2);
  if (m.dim >= 3) n3 = m.wrap(2, n3);
  ph.cell[t] = (uint32_t)m.idx(n1, n2, n3);
  ph.x1[t] = nx[0];
  ph.x2[t] = nx[1];
  ph.x3[t] = nx[2];
  ph.path[t] -= dt;
}

template <typename R>
__global__ void k_move_photons_cart(Mesh m, PhoView<R> ph, uint64_t n, R dt,
                                    const unsigned long long *__restrict__ dn) {
  const uint64_t cnt = dev_n(n, dn), stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < cnt; t += stride)
    move_photon_cart(m, ph, t, dt);
}

// move_photons (ptc_updater_logsph.cu:58-132); as in the reference the
// cell is taken before the axis reflection
template <typename R>
__device__ inline void move_photon_logsph(const Mesh &m, const PhoView<R> &ph, uint64_t t, R dt,
                                          double r_cutoff) {
  using M = RtMath<R>;
  const uint32_t c = ph.cell[t];
  if (c == MAX_CELL) return;
  const int d0 = m.dims[0];
  const int c1 = (int)(c % (uint32_t)d0), c2 = (int)(c / (uint32_t)d0);
  R v1 = ph.p1[t], v2 = ph.p2[t], v3 = ph.p3[t];
  const R E = sqrt(v1 * v1 + v2 * v2 + v3 * v3);
  v1 = v1 / E;
  v2 = v2 / E;
  v3 = v3 / E;
  const R old_x1 = ph.x1[t], old_x2 = ph.x2[t], old_x3 = ph.x3[t];
  const R r1 = (R)rt_pos(m, 0, c1, (double)old_x1);
  const R exp_r1 = M::exp(r1);
  if (exp_r1 > (R)r_cutoff || exp_r1 < (R)1.02) {
    ph.cell[t] = MAX_CELL;
    return;
  }
  const R r2 = (R)rt_pos(m, 1, c2, (double)old_x2);
  R s2, cs2, s3, cs3;
  M::sincos(r2, s2, cs2);
  M::sincos(old_x3, s3, cs3);
  R x = exp_r1 * s2 * cs3;
  R y = exp_r1 * s2 * s3;
  R z = exp_r1 * cs2;
  {
    R a = v1, b = v2, cc = v3;
    v1 = a * s2 * cs3 + b * cs2 * cs3 - cc * s3;
    v2 = a * s2 * s3 + b * cs2 * s3 + cc * cs3;
    v3 = a * cs2 - b * s2;
  }
  x += v1 * dt;
  y += v2 * dt;
  z += v3 * dt;
  R r1p = sqrt(x * x + y * y + z * z);
  R r2p;  // FP32: atan2 form, as in the particle mover
  if constexpr (std::is_same<R, double>::value)
    r2p = M::acos(z / r1p);
  else
    r2p = M::atan2(sqrt(x * x + y * y), z);
  r1p = M::log(r1p);
  const R r3p = M::atan2(y, x);
  {
    R ps2, pc2, ps3, pc3;
    M::sincos(r2p, ps2, pc2);
    M::sincos(r3p, ps3, pc3);
    R a = v1, b = v2, cc = v3;
    v1 = a * ps2 * pc3 + b * ps2 * ps3 + cc * pc2;
    v2 = a * pc2 * pc3 + b * pc2 * ps3 - cc * ps2;
    v3 = -a * ps3 + b * pc3;
  }
  ph.p1[t] = v1 * E;
  ph.p2[t] = v2 * E;
  ph.p3[t] = v3 * E;
  R new_x1 = old_x1 + (r1p - r1) / (R)m.delta[0];
  R new_x2 = old_x2 + (r2p - r2) / (R)m.delta[1];
  const int dc1 = (int)floor(new_x1);
  const int dc2 = (int)floor(new_x2);
  if (dc1 < -1 || dc1 > 1 || dc2 < -1 || dc2 > 1) {
    ph.cell[t] = MAX_CELL;
    return;
  }
  ph.cell[t] = (uint32_t)((c1 + dc1) + (c2 + dc2) * d0);
  new_x1 -= (R)dc1;
  new_x2 -= (R)dc2;
  if (rt_pos(m, 1, c2 + dc2, (double)new_x2) < 0.0)
    new_x2 = (R)1 - new_x2;
  else if (rt_pos(m, 1, c2 + dc2, (double)new_x2) >= RT_PI)
    new_x2 = (R)1 - new_x2;
  ph.x1[t] = new_x1;
  ph.x2[t] = new_x2;
  ph.x3[t] = r3p;
  ph.path[t] -= dt;
}

template <typename R>
__global__ void k_move_photons_logsph(Mesh m, PhoView<R> ph, uint64_t n, R dt,
                                      double r_cutoff,
                                      const unsigned long long *__restrict__ dn) {
  const uint64_t cnt = dev_n(n, dn), stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < cnt; t += stride)
    move_photon_logsph(m, ph, t, dt, r_cutoff);
}

// ---------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------
static inline unsigned rt_blocks(uint64_t n) {
  return (unsigned)((n + 255) / 256);
}

// A run's counts grow with every injection: sized to the count, the scratch was
// freed and allocated again on each call, ~100 us a step.  So room_for(n), or just
// n where memory is short.
hipError_t RtWork::ensure(uint64_t n) {
  if (n <= cap && host_total) return hipSuccess;
  const uint64_t least = n < 1024 ? 1024 : n, slack = room_for(least, most);
  if (slack > least) {
    if (alloc(slack) == hipSuccess) return hipSuccess;
    (void)hipGetLastError();
  }
  return alloc(least);
}

hipError_t RtWork::alloc(uint64_t c) {
  release();
  hipError_t e;
  if ((e = hipMalloc(&flags, c * 4)) != hipSuccess) return e;
  if ((e = hipMalloc(&total, sizeof(unsigned long long))) != hipSuccess)
    return e;
  if ((e = hipMalloc(&bsum, (ev_blocks(c, EV_HOST_E) + 1) * 8)) != hipSuccess) return e;
  if ((e = hipHostMalloc((void **)&host_total, sizeof(unsigned long long), hipHostMallocDefault)) !=
      hipSuccess)
    return e;
  cap = c;
  return hipSuccess;
}

void RtWork::release() {
  (void)hipFree(flags);
  (void)hipFree(total);
  (void)hipFree(bsum);
  (void)hipHostFree(host_total);
  bsum = nullptr;
  flags = nullptr;
  total = host_total = nullptr;
  cap = 0;
}

// the prefixes of the decided events and their number on the host
static hipError_t count_events(RtWork &w, uint64_t n, hipStream_t st, uint64_t *count) {
  k_ev_scan<<<1, EV_SCAN_T, 0, st>>>(w.bsum, n, EV_HOST_E, nullptr, w.host_total);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e == hipSuccess) *count = *(volatile unsigned long long *)w.host_total;
  return e;
}

template <typename R>
hipError_t rt_emit(const Mesh &m, const RtParams &rt, const PtcView<R> &p,
                   uint64_t n, const PhoView<R> &ph, uint64_t ph_base,
                   uint64_t seed, uint32_t epoch, uint64_t id_base,
                   RtWork &w, unsigned long long *counters, hipStream_t st,
                   R *produced, uint64_t *emitted, unsigned long long *dc) {
  *emitted = 0;
  if (n == 0) return hipSuccess;
  hipError_t e = w.ensure(n);
  if (e != hipSuccess) return e;
  if (dc) {  // no read-back: the counts stay on the device, n is a bound
    const unsigned nb = (unsigned)ev_blocks(n, EV_DEV_E);
    const unsigned long long *dn = dc + DC_NUM;
    k_ev_flags<R, true, EV_DEV_E><<<nb, EV_T, 0, st>>>(m, rt, p, ph, n, dn, w.flags, produced,
                                                       w.bsum);
    k_ev_scan<<<1, EV_SCAN_T, 0, st>>>(w.bsum, n, EV_DEV_E, dn, w.total);
    k_ev_apply<R, true, EV_DEV_E><<<nb, EV_T, 0, st>>>(m, rt, p, ph, n, dn, w.flags, w.bsum, seed,
                                                       0, 0, 0, dc, counters);
    k_events_finish<<<1, 64, 0, st>>>(w.total, rt.max_photon, 1, dc);
    return hipGetLastError();
  }
  const unsigned nb = (unsigned)ev_blocks(n, EV_HOST_E);
  k_ev_flags<R, true, EV_HOST_E><<<nb, EV_T, 0, st>>>(m, rt, p, ph, n, nullptr, w.flags, produced,
                                                      w.bsum);
  uint64_t total = 0;
  if ((e = count_events(w, n, st, &total)) != hipSuccess) return e;
  if (total == 0) return hipSuccess;
  k_ev_apply<R, true, EV_HOST_E><<<nb, EV_T, 0, st>>>(m, rt, p, ph, n, nullptr, w.flags, w.bsum,
                                                      seed, ph_base, id_base, epoch, nullptr,
                                                      counters);
  uint64_t room = rt.max_photon > ph_base ? rt.max_photon - ph_base : 0;
  *emitted = total < room ? total : room;
  return hipGetLastError();
}

template <typename R>
hipError_t rt_pairs(const Mesh &m, const RtParams &rt, const PtcView<R> &p,
                    uint64_t p_base, const PhoView<R> &ph, uint64_t nph,
                    uint64_t id_base, RtWork &w, unsigned long long *counters,
                    hipStream_t st, R *produced, uint64_t *made,
                    unsigned long long *dc) {
  *made = 0;
  if (nph == 0) return hipSuccess;
  hipError_t e = w.ensure(nph);
  if (e != hipSuccess) return e;
  if (dc) {  // no read-back: the counts stay on the device, nph is a bound
    const unsigned nb = (unsigned)ev_blocks(nph, EV_DEV_E);
    const unsigned long long *dn = dc + DC_PH;
    k_ev_flags<R, false, EV_DEV_E><<<nb, EV_T, 0, st>>>(m, rt, p, ph, nph, dn, w.flags, produced,
                                                        w.bsum);
    k_ev_scan<<<1, EV_SCAN_T, 0, st>>>(w.bsum, nph, EV_DEV_E, dn, w.total);
    k_ev_apply<R, false, EV_DEV_E><<<nb, EV_T, 0, st>>>(m, rt, p, ph, nph, dn, w.flags, w.bsum, 0,
                                                        0, 0, 0, dc, counters);
    k_events_finish<<<1, 64, 0, st>>>(w.total, rt.max_ptc, 0, dc);
    return hipGetLastError();
  }
  const unsigned nb = (unsigned)ev_blocks(nph, EV_HOST_E);
  k_ev_flags<R, false, EV_HOST_E><<<nb, EV_T, 0, st>>>(m, rt, p, ph, nph, nullptr, w.flags,
                                                       produced, w.bsum);
  uint64_t total = 0;
  if ((e = count_events(w, nph, st, &total)) != hipSuccess) return e;
  if (total == 0) return hipSuccess;
  k_ev_apply<R, false, EV_HOST_E><<<nb, EV_T, 0, st>>>(m, rt, p, ph, nph, nullptr, w.flags, w.bsum,
                                                       0, p_base, id_base, 0, nullptr, counters);
  // pairs whose second slot fits: base + 2k + 1 < max_ptc, k < L/2
  const uint64_t L = rt.max_ptc > p_base ? rt.max_ptc - p_base : 0;
  *made = total < L / 2 ? total : L / 2;
  return hipGetLastError();
}

template <typename R>
hipError_t rt_move_photons(const Mesh &m, int logsph, double r_cutoff,
                           const PhoView<R> &ph, uint64_t n, double dt,
                           hipStream_t st, const unsigned long long *dn) {
  if (n == 0) return hipSuccess;
  if (logsph)
    k_move_photons_logsph<R><<<slot_blocks(n, dn), 256, 0, st>>>(m, ph, n, (R)dt,
                                                                 r_cutoff, dn);
  else
    k_move_photons_cart<R><<<slot_blocks(n, dn), 256, 0, st>>>(m, ph, n, (R)dt, dn);
  return hipGetLastError();
}

hipError_t launch_fill_tail(uint32_t *cell, const unsigned long long *kept, uint64_t n,
                            hipStream_t st) {
  if (n == 0) return hipSuccess;
  k_fill_tail<<<rt_blocks(n), 256, 0, st>>>(cell, kept, n);
  return hipGetLastError();
}

hipError_t launch_dc_set(unsigned long long *dc, int which, const unsigned long long *src,
                         hipStream_t st) {
  k_dc_set<<<1, 64, 0, st>>>(dc, which, src);
  return hipGetLastError();
}

hipError_t launch_dc_accum(unsigned long long *dc, int to, int from, hipStream_t st) {
  k_dc_accum<<<1, 64, 0, st>>>(dc, to, from);
  return hipGetLastError();
}

#define INST(R)                                                               \
  template hipError_t rt_emit<R>(const Mesh &, const RtParams &,              \
                                 const PtcView<R> &, uint64_t,                \
                                 const PhoView<R> &, uint64_t, uint64_t,      \
                                 uint32_t, uint64_t, RtWork &,                \
                                 unsigned long long *, hipStream_t, R *,      \
                                 uint64_t *, unsigned long long *);           \
  template hipError_t rt_pairs<R>(const Mesh &, const RtParams &,             \
                                  const PtcView<R> &, uint64_t,               \
                                  const PhoView<R> &, uint64_t, uint64_t,     \
                                  RtWork &, unsigned long long *,             \
                                  hipStream_t, R *, uint64_t *,               \
                                  unsigned long long *);                      \
  template hipError_t rt_move_photons<R>(const Mesh &, int, double,           \
                                         const PhoView<R> &, uint64_t,        \
                                         double, hipStream_t,                 \
                                         const unsigned long long *);
INST(double)
INST(float)
#undef INST

}  // namespace apt
