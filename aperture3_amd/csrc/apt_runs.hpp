// apt_runs.hpp -- tiles over cell-ordered slots.  After a sort by cell the
// slots of the cells (i0 .. i1, j, k) of one mesh row are contiguous, so a tile
// of T0 x T1 x T2 cells is T1 T2 runs of consecutive slots.  A table of run
// starts, built from the sorted keys at the sort, lets one workgroup take one
// tile's particles (or a share of them) and sum their current in an LDS window
// over the tile plus a halo for the drift until the next sort -- without
// moving the particles out of the order the sort gave them.
#pragma once
#include "apt_common.hpp"
#include "apt_kernels.hpp"

namespace apt {

// blockIdx -> work item: workgroups are dispatched round-robin over the 8
// XCDs, so giving XCD x the contiguous range [x n/8, (x+1) n/8) keeps
// neighbouring tiles' halos in one L2.
__device__ __forceinline__ uint32_t xcd_tile(uint32_t b, uint32_t ntiles) {
  if ((ntiles & 7u) != 0) return b;
  uint32_t per = ntiles >> 3;
  return (b & 7u) * per + (b >> 3);
}

// Window coordinate of mesh coordinate c: the periodic image that lies in the
// window's usable range [2, W - 3], if there is one (with an axis shorter
// than the window, the image on the tile itself).
template <int W>
__device__ __forceinline__ int window_coord(int c, int w, int N, bool periodic = true) {
  int l = c - w;
  if (periodic) {
    if (l < 2) l += N;
    else if (l > W - 3) l -= N;
  }
  return l;
}

// a window coordinate back on the mesh: any number of periods on a
// periodic axis, unchanged on the others
__device__ __forceinline__ int fold_axis(const Mesh &m, int ax, int i) {
  if (!m.periodic[ax]) return i;
  const int g = m.guard[ax], N = m.N[ax];
  int r = (i - g) % N;
  if (r < 0) r += N;
  return g + r;
}

// f(slot) for every slot that the table holds in guard rows, a row a workgroup
// at a time, a slot a lane.
template <class F>
__device__ __forceinline__ void for_guard_row_slots(const Mesh &m, const CellRuns &cr, const F &f) {
  const uint32_t rows = (uint32_t)m.dims[1] * (uint32_t)m.dims[2];
  for (uint32_t r = blockIdx.x; r < rows; r += gridDim.x) {
    const int j = (int)(r % (uint32_t)m.dims[1]), k = (int)(r / (uint32_t)m.dims[1]);
    if (m.in_bulk(m.guard[0], j, k)) continue;
    const uint64_t e = (uint64_t)r * (uint64_t)cr.nt[0];
    const uint32_t end = cr.off[e + (uint64_t)cr.nt[0]];
    for (uint32_t i = cr.off[e] + threadIdx.x; i < end; i += blockDim.x) f(i);
  }
}
inline unsigned guard_row_blocks(const Mesh &m) {
  const uint64_t rows = (uint64_t)m.dims[1] * m.dims[2];
  return (unsigned)(rows < 4096 ? rows : 4096);
}

// Work item of workgroup b: the items in use are spread over the XCDs as in
// xcd_tile.  False: there is none.
__device__ __forceinline__ bool run_item(const CellRuns &cr, uint32_t b, uint32_t &tile,
                                         uint32_t &part, uint32_t &parts) {
  const uint32_t n = cr.work[0], per = (n + 7u) >> 3, i = (b & 7u) * per + (b >> 3);
  if ((b >> 3) >= per || i >= n) return false;
  tile = cr.work[2 + 2 * i];
  part = cr.work[3 + 2 * i] & 0xffffu;
  parts = cr.work[3 + 2 * i] >> 16;
  return true;
}

// One workgroup's share of a tile's slots.  ROWS: the most rows of a tile.
template <int ROWS>
struct RunWalk {
  uint32_t first[ROWS];      // first slot of each row's run
  uint32_t pref[ROWS + 1];   // particles before each row
  // fills the table (all threads; ends with a barrier); returns the share's
  // range [lo, hi) of the tile's particles
  __device__ __forceinline__ void open(const Mesh &m, const CellRuns &cr, uint32_t tile,
                                       uint32_t part, uint32_t split, int org[3], uint32_t &lo,
                                       uint32_t &hi) {
    const int tx = (int)(tile % (uint32_t)cr.nt[0]);
    const int ty = (int)((tile / (uint32_t)cr.nt[0]) % (uint32_t)cr.nt[1]);
    const int tz = (int)(tile / ((uint32_t)cr.nt[0] * (uint32_t)cr.nt[1]));
    org[0] = m.guard[0] + cr.ax[0].origin(tx);
    org[1] = m.guard[1] + cr.ax[1].origin(ty);
    org[2] = m.guard[2] + cr.ax[2].origin(tz);
    const int e1 = cr.ax[1].origin(ty + 1) - cr.ax[1].origin(ty);
    const int e2 = cr.ax[2].origin(tz + 1) - cr.ax[2].origin(tz);
    const int nr = e1 * e2;
    // exclusive scan of the run lengths by the first wave
    if (threadIdx.x < 64) {
      const int lane = (int)threadIdx.x;
      uint32_t carry = 0;
      for (int b = 0; b < nr; b += 64) {
        const int r = b + lane;
        uint32_t f = 0, n = 0;
        if (r < nr) {
          const int jj = r % e1, kk = r / e1;
          const uint64_t row = (uint64_t)(org[1] + jj) + (uint64_t)m.dims[1] * (org[2] + kk);
          const uint64_t e = row * (uint64_t)cr.nt[0] + (uint64_t)tx;
          f = cr.off[e];
          n = cr.off[e + 1] - f;
        }
        uint32_t s = n;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
          const uint32_t u = __shfl_up(s, d);
          if (lane >= d) s += u;
        }
        if (r < nr) {
          first[r] = f;
          pref[r] = carry + s - n;
        }
        carry += __shfl(s, 63);
      }
      for (int r = nr + lane; r <= ROWS; r += 64) pref[r] = carry;
    }
    __syncthreads();
    const uint64_t total = pref[nr];
    lo = (uint32_t)(total * part / split);
    hi = (uint32_t)(total * (part + 1) / split);
  }
  // slot of the tile's q-th particle
  __device__ __forceinline__ uint32_t slot(uint32_t q) const {
    int a = 0;
    if (ROWS > 1) {
      int b = ROWS;  // pref[a] <= q < pref[b]
#pragma unroll
      for (int s = ROWS; s > 1; s = (s + 1) / 2) {
        const int mid = (a + b) >> 1;
        const bool up = pref[mid] <= q;
        a = up && mid > a ? mid : a;
        b = up ? b : mid;
      }
    }
    return first[a] + (q - pref[a]);
  }
};

}  // namespace apt
