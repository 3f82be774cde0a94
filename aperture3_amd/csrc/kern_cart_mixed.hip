// kern_cart_mixed.hip -- mixed-precision Cartesian particle update: the
// same fused push + move + Esirkepov deposit as the FP64 form
// (ptc_updater.cu:21-499), computed in FP32 on the 36-byte particle layout
// (int32 cell, FP32 in-cell offsets, FP32 u = gamma v, FP32 weight, flag).
// gamma is recomputed from u instead of stored.  Every current
// contribution is rounded to 2^-H and summed in int64, so the deposit is
// deterministic and charge conserving to the round-off of the FP32 shapes.
#include "apt_common.hpp"
#include "apt_f32.hpp"
#include "apt_kernels.hpp"
#include "apt_runs.hpp"
#include "apt_tiles.hpp"

namespace apt {

#pragma clang fp contract(fast)

// shape arrays over the four node offsets -2..1 around the old cell:
// s0 = old position, s1 = new position (moved by dc in {-1,0,1})
__device__ __forceinline__ void shapes(float xo, float xn, int dc, float s0[4],
                                       float s1[4]) {
#pragma unroll
  for (int t = 0; t < 4; t++) {
    s0[t] = 0.0f;
    s1[t] = 0.0f;
  }
  s0[1] = 1.0f - xo;
  s0[2] = xo;
  s1[1 + dc] = 1.0f - xn;
  s1[2 + dc] = xn;
}

// Push, move and deposit of one live particle in bulk cell (c1, c2, c3);
// add(q, di, dj, dk, v) adds v to component q (0..2: J1..J3; 3 + s: Rho of
// species s) at an offset of -2 .. 1 (J: .. 2) cells from that cell.
template <int DIM, class Add>
__device__ __forceinline__ void push_deposit_mixed(const Mesh &m, const Species &sp, float dt,
                                                   int rho, const PtcF32 &p, const FieldsF32 &f,
                                                   unsigned long long *__restrict__ counters,
                                                   uint64_t idx, int c1, int c2, int c3,
                                                   const Add &add) {
  uint32_t flag = p.flag[idx];
  int s = ptc_species(flag);
  float x1 = p.x1[idx], x2 = p.x2[idx], x3 = p.x3[idx];
  float u1 = p.u1[idx], u2 = p.u2[idx], u3 = p.u3[idx];
  float w = p.w[idx];
  if (u1 != u1 || u2 != u2 || u3 != u3) atomicAdd(&counters[CTR_NAN], 1ull);
  float gamma = sqrtf(1.0f + u1 * u1 + u2 * u2 + u3 * u3);
  if (!(flag & FLAG_IGNORE_EM)) {
    float qm = (float)(0.5 * sp.q[s] / sp.m[s]) * dt;
    float E1 = gatherf<DIM>(f.E[0], m, c1, c2, c3, x1, x2, x3, ST_E1) * qm;
    float E2 = gatherf<DIM>(f.E[1], m, c1, c2, c3, x1, x2, x3, ST_E2) * qm;
    float E3 = gatherf<DIM>(f.E[2], m, c1, c2, c3, x1, x2, x3, ST_E3) * qm;
    float B1 = gatherf<DIM>(f.B[0], m, c1, c2, c3, x1, x2, x3, ST_B1) * qm;
    float B2 = gatherf<DIM>(f.B[1], m, c1, c2, c3, x1, x2, x3, ST_B2) * qm;
    float B3 = gatherf<DIM>(f.B[2], m, c1, c2, c3, x1, x2, x3, ST_B3) * qm;
    vay_pushf(u1, u2, u3, gamma, E1, E2, E3, B1, B2, B3);
    gamma = sqrtf(1.0f + u1 * u1 + u2 * u2 + u3 * u3);
    p.u1[idx] = u1;
    p.u2[idx] = u2;
    p.u3[idx] = u3;
  }
  float ig = 1.0f / gamma;
  float v1 = u1 * ig, v2 = u2 * ig, v3 = u3 * ig;
  float qw = (float)sp.q[s] * w;

  // ---- move ----
  float n1 = x1 + v1 * dt * (float)m.inv_delta[0];
  int dc1 = (int)floorf(n1);
  n1 -= (float)dc1;
  float n2 = x2, n3 = x3;
  int dc2 = 0, dc3 = 0;
  if (DIM >= 2) {
    n2 = x2 + v2 * dt * (float)m.inv_delta[1];
    dc2 = (int)floorf(n2);
    n2 -= (float)dc2;
  } else {
    n2 = x2 + v2 * dt;
  }
  if (DIM == 3) {
    n3 = x3 + v3 * dt * (float)m.inv_delta[2];
    dc3 = (int)floorf(n3);
    n3 -= (float)dc3;
  } else {
    n3 = x3 + v3 * dt;
  }
  // an offset that rounds to 1.0f belongs to the next cell
  if (n1 >= 1.0f) { n1 -= 1.0f; dc1 += 1; }
  if (DIM >= 2 && n2 >= 1.0f) { n2 -= 1.0f; dc2 += 1; }
  if (DIM == 3 && n3 >= 1.0f) { n3 -= 1.0f; dc3 += 1; }
  if (dc1 > 1 || dc1 < -1 || dc2 > 1 || dc2 < -1 || dc3 > 1 || dc3 < -1) {
    atomicAdd(&counters[CTR_MULTICELL], 1ull);
    dc1 = max(-1, min(1, dc1));
    dc2 = max(-1, min(1, dc2));
    dc3 = max(-1, min(1, dc3));
  }
  p.cell[idx] = (uint32_t)m.idx(m.wrap(0, c1 + dc1),
                                DIM >= 2 ? m.wrap(1, c2 + dc2) : c2,
                                DIM == 3 ? m.wrap(2, c3 + dc3) : c3);
  p.x1[idx] = n1;
  p.x2[idx] = n2;
  p.x3[idx] = n3;
  if (flag & FLAG_IGNORE_CURRENT) return;

  // ---- Esirkepov deposit (ptc_updater.cu:264-291, 343-384, 443-497) ----
  float sx0[4], sx1[4];
  shapes(x1, n1, dc1, sx0, sx1);
  if (DIM == 1) {
    float acc = 0.0f;
#pragma unroll
    for (int t = 0; t < 4; t++) {
      acc += sx1[t] - sx0[t];
      if (t < 3) add(0, t - 1, 0, 0, -qw * acc);
      float val = 0.5f * (sx0[t] + sx1[t]);
      if (val != 0.0f) {
        add(1, t - 2, 0, 0, qw * v2 * val);
        add(2, t - 2, 0, 0, qw * v3 * val);
        if (rho && sx1[t] != 0.0f) add(3 + s, t - 2, 0, 0, qw * sx1[t]);
      }
    }
    return;
  }
  float sy0[4], sy1[4];
  shapes(x2, n2, dc2, sy0, sy1);
  if (DIM == 2) {
    const float wt = -qw;  // reference sign convention (ptc_updater.cu:345)
    float djy[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int tj = 0; tj < 4; tj++) {
      float ay = 0.5f * (sy0[tj] + sy1[tj]);
      float dsy = sy1[tj] - sy0[tj];
      float djx = 0.0f;
#pragma unroll
      for (int ti = 0; ti < 4; ti++) {
        djx += (sx1[ti] - sx0[ti]) * ay;
        if (ti < 3 && djx != 0.0f) add(0, ti - 1, tj - 2, 0, wt * djx);
        djy[ti] += dsy * 0.5f * (sx0[ti] + sx1[ti]);
        if (tj < 3 && djy[ti] != 0.0f)
          add(1, ti - 2, tj - 1, 0, wt * djy[ti]);
        float cen = (2.0f * sx1[ti] * sy1[tj] + sx0[ti] * sy1[tj] +
                     sx1[ti] * sy0[tj] + 2.0f * sx0[ti] * sy0[tj]) *
                    (1.0f / 6.0f);
        if (cen != 0.0f) add(2, ti - 2, tj - 2, 0, -wt * v3 * cen);
        if (rho && sx1[ti] * sy1[tj] != 0.0f)
          add(3 + s, ti - 2, tj - 2, 0, qw * (sx1[ti] * sy1[tj]));
      }
    }
    return;
  }
  float sz0[4], sz1[4];
  shapes(x3, n3, dc3, sz0, sz1);
  {
    const float wt = -qw;
    float djz[4][4];
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
      for (int b = 0; b < 4; b++) djz[a][b] = 0.0f;
#pragma unroll
    for (int tk = 0; tk < 4; tk++) {
      float djy[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int tj = 0; tj < 4; tj++) {
        float djx = 0.0f;
        float cyz = (2.0f * sy1[tj] * sz1[tk] + sy0[tj] * sz1[tk] +
                     sy1[tj] * sz0[tk] + 2.0f * sy0[tj] * sz0[tk]) *
                    (1.0f / 6.0f);
#pragma unroll
        for (int ti = 0; ti < 4; ti++) {
          djx += (sx1[ti] - sx0[ti]) * cyz;
          if (ti < 3 && djx != 0.0f)
            add(0, ti - 1, tj - 2, tk - 2, wt * djx);
          float cxz = (2.0f * sx1[ti] * sz1[tk] + sx0[ti] * sz1[tk] +
                       sx1[ti] * sz0[tk] + 2.0f * sx0[ti] * sz0[tk]) *
                      (1.0f / 6.0f);
          djy[ti] += (sy1[tj] - sy0[tj]) * cxz;
          if (tj < 3 && djy[ti] != 0.0f)
            add(1, ti - 2, tj - 1, tk - 2, wt * djy[ti]);
          float cxy = (2.0f * sx1[ti] * sy1[tj] + sx0[ti] * sy1[tj] +
                       sx1[ti] * sy0[tj] + 2.0f * sx0[ti] * sy0[tj]) *
                      (1.0f / 6.0f);
          djz[tj][ti] += (sz1[tk] - sz0[tk]) * cxy;
          if (tk < 3 && djz[tj][ti] != 0.0f)
            add(2, ti - 2, tj - 2, tk - 1, wt * djz[tj][ti]);
          float s3 = sx1[ti] * sy1[tj] * sz1[tk];
          if (rho && s3 != 0.0f) add(3 + s, ti - 2, tj - 2, tk - 2, qw * s3);
        }
      }
    }
  }
}

template <int DIM>
__global__ void __launch_bounds__(256)
    k_push_deposit_mixed(Mesh m, Species sp, float dt, float scale, PtcF32 p,
                         FieldsF32 f, AccMixed a,
                         unsigned long long *__restrict__ counters,
                         uint64_t first, uint64_t n) {
  uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const uint64_t idx = first + t;
  uint32_t c = p.cell[idx];
  if (c == MAX_CELL) return;
  int c1, c2, c3;
  m.split(c, c1, c2, c3);
  if (!m.in_bulk(c1, c2, c3)) {
    p.cell[idx] = MAX_CELL;
    return;
  }
  push_deposit_mixed<DIM>(m, sp, dt, a.rho, p, f, counters, idx, c1, c2, c3,
                          [&](int q, int di, int dj, int dk, float v) {
                            acc_fx(q < 3 ? a.J[q] : a.R[q - 3], m.widx(c1 + di, c2 + dj, c3 + dk),
                                   v, scale);
                          });
}

// Tile shapes of the update over cell runs: cells per tile, halo, threads,
// copies of the window, slots per lane run.
template <int A, int B, int C, int HH, int TH, int NC, int RL>
struct MixedShape {
  static constexpr int T0 = A, T1 = B, T2 = C, H = HH, NT = TH, COPIES = NC, R = RL;
};
template <int DIM>
struct MixedRunShape;
template <>
struct MixedRunShape<1> : MixedShape<16, 1, 1, 16, 256, 8, 8> {};
template <>
struct MixedRunShape<2> : MixedShape<16, 16, 1, 8, 512, 1, 16> {};
template <>
struct MixedRunShape<3> : MixedShape<8, 8, 8, 4, 512, 1, 16> {};

void mixed_runs_tile(int dim, int T[3]) {
  T[0] = dim == 3 ? 8 : 16;
  T[1] = dim == 1 ? 1 : dim == 2 ? 16 : 8;
  T[2] = dim == 3 ? 8 : 1;
}

// A workgroup clears and flushes a window whatever is in its tile, so on thin
// plasma the update of one HBM atomic per contribution is the faster one, unless
// there are so few tiles that either is a launch and little more.  The lines lie
// where the two meet (us per push, that one / this one): 1D, 62,500 tiles, 8
// slots a tile 105 / 229, 16 168 / 233, 32 333 / 237; 2D open, 4096 tiles, 13
// 62 / 88, 128 223 / 109; 3D open, 1728 tiles, 26 78 / 188, 256 328 / 213.
bool mixed_runs_pay(int dim, uint64_t kept, uint32_t items) {
  const uint64_t least = dim == 1 ? 24 : dim == 2 ? 64 : 192;
  return items <= (dim == 3 ? 256u : 1024u) || kept >= least * items;
}

// The mixed update of cell-sorted slots where the tiled push does not apply
// (1D, and open axes): one workgroup per tile (or share of a tile), the current
// and the charge of two species summed in an LDS window over the tile and a
// halo, flushed once per element; particles outside the window add to HBM.  A
// wave's lanes take 64 / R runs of R consecutive slots spread over the share
// and, in 1D, where a tile is a few cells wide, alternate between copies of the
// window, so that the wave's atomics fall on many addresses.  The same integer
// sums as one HBM atomic per contribution, which queued on a few elements: 1D,
// 10,000 cells at 80 per cell 220 -> 20 us per push.
template <int DIM>
__global__ void __launch_bounds__(MixedRunShape<DIM>::NT)
    k_push_deposit_mixed_runs(Mesh m, Species sp, float dt, float scale, PtcF32 p, FieldsF32 f,
                              AccMixed a, CellRuns cr, unsigned long long *__restrict__ counters) {
  using S = MixedRunShape<DIM>;
  constexpr int NT = S::NT, HW = S::H, R = S::R, NC = S::COPIES;
  constexpr int W0 = S::T0 + 2 * HW, W1 = DIM > 1 ? S::T1 + 2 * HW : 1;
  constexpr int W2 = DIM > 2 ? S::T2 + 2 * HW : 1, WN = W0 * W1 * W2;
  constexpr int NQ = DIM < 3 ? 5 : 3;  // 3D: Rho goes to HBM
  static_assert(64 % R == 0 && 64 % NC == 0, "lane runs and copies divide the wave");
  __shared__ unsigned long long win[NC * NQ * WN];
  __shared__ RunWalk<S::T1 * S::T2> walk;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  uint32_t tile, part, parts;
  if (!run_item(cr, blockIdx.x, tile, part, parts)) return;  // uniform
  for (int e = tid; e < NC * NQ * WN; e += NT) win[e] = 0;
  int org[3];
  uint32_t lo, hi;
  walk.open(m, cr, tile, part, parts, org, lo, hi);
  if (lo == hi) return;  // uniform
  const int w0 = org[0] - HW, w1 = DIM > 1 ? org[1] - HW : org[1];
  const int w2 = DIM > 2 ? org[2] - HW : org[2];
  const uint32_t cnt = hi - lo;
  constexpr uint32_t G = 64 / R;
  const uint32_t seg = ((cnt + G - 1) / G + R - 1) / R * R;
  unsigned long long *const mine = win + (lane & (NC - 1)) * NQ * WN;
#pragma unroll 1
  for (uint32_t k = wv * R; k < seg; k += (NT / 64) * R) {
    const uint32_t kk = k + (uint32_t)(lane % R), q = (uint32_t)(lane / R) * seg + kk;
    if (kk >= seg || q >= cnt) continue;
    const uint64_t idx = walk.slot(lo + q);
    const uint32_t c = p.cell[idx];
    if (c == MAX_CELL) continue;
    int c1, c2, c3;
    m.split(c, c1, c2, c3);
    if (!m.in_bulk(c1, c2, c3)) {
      p.cell[idx] = MAX_CELL;
      continue;
    }
    const int l0 = window_coord<W0>(c1, w0, m.N[0], m.periodic[0]);
    const int l1 = DIM > 1 ? window_coord<W1>(c2, w1, m.N[1], m.periodic[1]) : 0;
    const int l2 = DIM > 2 ? window_coord<W2>(c3, w2, m.N[2], m.periodic[2]) : 0;
    bool in = l0 >= 2 && l0 <= W0 - 3;
    if (DIM > 1) in = in && l1 >= 2 && l1 <= W1 - 3;
    if (DIM > 2) in = in && l2 >= 2 && l2 <= W2 - 3;
    unsigned long long *const e0 = mine + (in ? l0 + W0 * (l1 + W1 * l2) : 0);
    push_deposit_mixed<DIM>(
        m, sp, dt, a.rho, p, f, counters, idx, c1, c2, c3,
        [&](int q, int di, int dj, int dk, float v) {
          if (in && q < NQ)
            __hip_atomic_fetch_add(e0 + q * WN + di + W0 * (dj + W1 * dk),
                                   (unsigned long long)(long long)__float2int_rn(v * scale),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          else
            acc_fx(q < 3 ? a.J[q] : a.R[q - 3], m.widx(c1 + di, c2 + dj, c3 + dk), v, scale);
        });
  }
  __syncthreads();
  for (int e = tid; e < NQ * WN; e += NT) {
    unsigned long long v = 0;
#pragma unroll
    for (int cpy = 0; cpy < NC; cpy++) v += win[cpy * NQ * WN + e];
    if (v == 0) continue;
    const int q = e / WN, cc = e - q * WN;
    const int u0 = fold_axis(m, 0, w0 + cc % W0);
    const int u1 = DIM > 1 ? fold_axis(m, 1, w1 + cc / W0 % W1) : w1;
    const int u2 = DIM > 2 ? fold_axis(m, 2, w2 + cc / (W0 * W1)) : w2;
    __hip_atomic_fetch_add((unsigned long long *)(q < 3 ? a.J[q] : a.R[q - 3]) + m.idx(u0, u1, u2),
                           v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// The slots that a sort left in guard rows, which belong to no tile (see
// k_push_guard_rows_f64).
template <int DIM>
__global__ void __launch_bounds__(64)
    k_push_guard_rows_mixed(Mesh m, Species sp, float dt, float scale, PtcF32 p, FieldsF32 f,
                            AccMixed a, CellRuns cr, unsigned long long *__restrict__ counters) {
  for_guard_row_slots(m, cr, [&](uint32_t idx) {
    const uint32_t c = p.cell[idx];
    if (c == MAX_CELL) return;
    int c1, c2, c3;
    m.split(c, c1, c2, c3);
    if (!m.in_bulk(c1, c2, c3)) {
      p.cell[idx] = MAX_CELL;
      return;
    }
    push_deposit_mixed<DIM>(m, sp, dt, a.rho, p, f, counters, idx, c1, c2, c3,
                            [&](int q, int di, int dj, int dk, float v) {
                              acc_fx(q < 3 ? a.J[q] : a.R[q - 3],
                                     m.widx(c1 + di, c2 + dj, c3 + dk), v, scale);
                            });
  });
}

hipError_t launch_push_deposit_mixed_runs(const Mesh &m, const Species &sp, float dt, int S,
                                          const PtcF32 &p, const FieldsF32 &f, const AccMixed &a,
                                          const CellRuns &cr, unsigned long long *counters,
                                          hipStream_t st) {
  if (cr.end == 0) return hipSuccess;
  const float scale = ldexpf(1.0f, S);
  auto go = [&](auto kern, int NT) {
    kern<<<cr.items, NT, 0, st>>>(m, sp, dt, scale, p, f, a, cr, counters);
    return hipGetLastError();
  };
  if (cr.guard_slots > 0 && m.dim > 1) {
    if (m.dim == 2)
      k_push_guard_rows_mixed<2><<<guard_row_blocks(m), 64, 0, st>>>(m, sp, dt, scale, p, f, a, cr,
                                                                     counters);
    else
      k_push_guard_rows_mixed<3><<<guard_row_blocks(m), 64, 0, st>>>(m, sp, dt, scale, p, f, a, cr,
                                                                     counters);
  }
  if (m.dim == 1) return go(k_push_deposit_mixed_runs<1>, MixedRunShape<1>::NT);
  if (m.dim == 2) return go(k_push_deposit_mixed_runs<2>, MixedRunShape<2>::NT);
  return go(k_push_deposit_mixed_runs<3>, MixedRunShape<3>::NT);
}

hipError_t launch_push_deposit_mixed_range(const Mesh &m, const Species &sp,
                                           float dt, int S, const PtcF32 &p,
                                           const FieldsF32 &f,
                                           const AccMixed &a,
                                           unsigned long long *counters,
                                           uint64_t first, uint64_t n,
                                           hipStream_t st) {
  if (n == 0) return hipSuccess;
  float scale = ldexpf(1.0f, S);
  dim3 block(256), grid((unsigned)((n + 255) / 256));
  if (m.dim == 1)
    k_push_deposit_mixed<1><<<grid, block, 0, st>>>(m, sp, dt, scale, p, f, a,
                                                    counters, first, n);
  else if (m.dim == 2)
    k_push_deposit_mixed<2><<<grid, block, 0, st>>>(m, sp, dt, scale, p, f, a,
                                                    counters, first, n);
  else
    k_push_deposit_mixed<3><<<grid, block, 0, st>>>(m, sp, dt, scale, p, f, a,
                                                    counters, first, n);
  return hipGetLastError();
}

hipError_t launch_push_deposit_mixed(const Mesh &m, const Species &sp,
                                     float dt, int S, const PtcF32 &p,
                                     const FieldsF32 &f, const AccMixed &a,
                                     const TileInfo &tiles,
                                     unsigned long long *counters,
                                     uint64_t n, hipStream_t st, uint64_t first) {
  if (tiles.tile_off == nullptr || tiles.ntiles == 0)
    return launch_push_deposit_mixed_range(m, sp, dt, S, p, f, a, counters, first, n - first, st);
  hipError_t e = launch_push_deposit_tiled(m, sp, dt, S, p, f, a, tiles,
                                           counters, st);
  if (e != hipSuccess) return e;
  // slots past the tiled range (appended since the last sort)
  if (n > tiles.tiled_end)
    e = launch_push_deposit_mixed_range(m, sp, dt, S, p, f, a, counters,
                                        tiles.tiled_end, n - tiles.tiled_end,
                                        st);
  return e;
}

}  // namespace apt
