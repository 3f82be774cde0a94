// kern_sort.hip -- particle sort by cell with compaction
// (particle_base::sort_by_cell, cuda/core/particle_base_impl.cu:435-464,
// and its CPU twin core/particle_base_impl.hpp:250-305): a stable sort on
// the key cell (empty slots keyed past the last cell), a gather of every
// SoA field, and number := count of non-empty slots.  The radix pass is
// rocPRIM's stable LSD sort through hipCUB; the key width is trimmed to
// the cell count, so a 2048^2 grid takes 23 bits.  Stability makes the
// order within a cell the arrival order, exactly like the reference's
// counting sort.
#include <hipcub/hipcub.hpp>

#include "apt_common.hpp"
#include "apt_kernels.hpp"
#include "apt_sort.hpp"

namespace apt {

__global__ void k_make_keys(const uint32_t *__restrict__ cell, uint64_t n,
                            uint32_t empty_key, const uint32_t *tile_key_lut,
                            uint32_t *__restrict__ keys,
                            uint32_t *__restrict__ perm) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint32_t c = cell[i];
  uint32_t k;
  if (c == MAX_CELL)
    k = empty_key;
  else
    k = tile_key_lut ? tile_key_lut[c] : c;
  keys[i] = k;
  perm[i] = (uint32_t)i;
}

// number of keys below empty_key in a sorted key array
__global__ void k_count_valid(const uint32_t *__restrict__ keys, uint64_t n,
                              uint32_t empty_key,
                              unsigned long long *__restrict__ out) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  bool here = keys[i] < empty_key;
  bool next = (i + 1 < n) ? keys[i + 1] < empty_key : false;
  if (i == 0 && !here) *out = 0;
  if (here && !next) *out = i + 1;
}

// All arrays of a particle set in one pass: the permutation is read once, and a
// slot's loads, which depend on nothing but it, are in flight together.  With a
// launch per array the loads of one array waited for the last one's grid to
// drain: eight 1D boxes, 26 M particles and their photons, 19 launches of 62-67 us
// on average, 1.2 ms a sort; 0.75 ms in two; a pass of 20 steps with one sort 11.4
// -> 10.9 ms.  638 M particles take as long as before (9 x 1.5 ms), as do 17 M in
// random order (9 x 295 us): the gathered lines are the bound there.
template <int N4, int N8>
__global__ void k_gather_set(GatherSet g, const uint32_t *__restrict__ perm, uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t p = perm[i];
  uint32_t a[N4 > 0 ? N4 : 1];
  uint64_t b[N8 > 0 ? N8 : 1];
#pragma unroll
  for (int k = 0; k < N4; k++) a[k] = g.src4[k][p];
#pragma unroll
  for (int k = 0; k < N8; k++) b[k] = g.src8[k][p];
#pragma unroll
  for (int k = 0; k < N4; k++) g.dst4[k][i] = a[k];
#pragma unroll
  for (int k = 0; k < N8; k++) g.dst8[k][i] = b[k];
}

// Run starts by tile (CellRuns): entry e is the first of the n sorted keys not
// below its tile row's first cell, found by bisection (one table per sort:
// rows x tiles in x entries of ~25 probes, most of them in L2).
__global__ void k_cell_runs(Mesh m, CellRuns cr, const uint32_t *__restrict__ keys, uint64_t n,
                            uint32_t *__restrict__ off, uint64_t entries) {
  const uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= entries) return;
  if (e == 0) off[entries] = off[entries + 1] = 0;  // counts of k_cell_work
  uint64_t key = m.size();
  if (e + 1 < entries) {
    const uint64_t row = e / (uint64_t)cr.nt[0];
    const int tx = (int)(e - row * (uint64_t)cr.nt[0]);
    key = row * (uint64_t)m.dims[0] + (tx == 0 ? 0 : m.guard[0] + cr.ax[0].origin(tx));
  }
  uint64_t lo = 0, hi = n;
  while (lo < hi) {
    const uint64_t mid = (lo + hi) >> 1;
    if (keys[mid] < key) lo = mid + 1;
    else hi = mid;
  }
  off[e] = (uint32_t)lo;
}

// Work items of the tiles (CellRuns): a tile's particles in parts of about `per`
// (1.4 per still is one part), no item for an empty tile.  256 tiles a workgroup,
// whose items are in tile order; workgroups append theirs as they come (sums of
// integers do not depend on the order).  One workgroup over all tiles took 80 us
// for 62,500 tiles of a 1D mesh of 10^6 cells and 700 us for the 131,072 of a 3D
// one of 256^3, a serial stretch at every sort.
__global__ void __launch_bounds__(256)
    k_cell_work(Mesh m, CellRuns cr, uint64_t per, uint32_t *__restrict__ work) {
  __shared__ uint32_t s_w[4], s_n[4], s_base;
  __shared__ uint32_t s_many, s_list[256][3];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  if (tid == 0) s_many = 0;
  const uint32_t t = blockIdx.x * 256 + (uint32_t)tid;
  uint32_t parts = 0, slots = 0;
  if (t < cr.ntiles) {
    const uint32_t tx = t % (uint32_t)cr.nt[0], r = t / (uint32_t)cr.nt[0];
    const int ty = (int)(r % (uint32_t)cr.nt[1]), tz = (int)(r / (uint32_t)cr.nt[1]);
    for (int k = cr.ax[2].origin(tz); k < cr.ax[2].origin(tz + 1); k++)
      for (int j = cr.ax[1].origin(ty); j < cr.ax[1].origin(ty + 1); j++) {
        const uint64_t row = (uint64_t)(m.guard[1] + j) + (uint64_t)m.dims[1] * (m.guard[2] + k);
        const uint64_t e = row * (uint64_t)cr.nt[0] + tx;
        slots += cr.off[e + 1] - cr.off[e];
      }
    const uint64_t q = (5 * (uint64_t)slots + 3 * per) / (5 * per);
    parts = slots == 0 ? 0u : q < 1 ? 1u : q > 0xffff ? 0xffffu : (uint32_t)q;
  }
  uint32_t s = parts, n = slots;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t u = __shfl_up(s, d), v = __shfl_up(n, d);
    if (lane >= d) {
      s += u;
      n += v;
    }
  }
  if (lane == 63) {
    s_w[wv] = s;
    s_n[wv] = n;
  }
  __syncthreads();
  if (tid == 0) {
    s_base = atomicAdd(&work[0], s_w[0] + s_w[1] + s_w[2] + s_w[3]);
    atomicAdd(&work[1], s_n[0] + s_n[1] + s_n[2] + s_n[3]);
  }
  __syncthreads();
  uint32_t at = s_base + s - parts;
  for (int k = 0; k < wv; k++) at += s_w[k];
  auto put = [&](uint32_t tile, uint32_t first, uint32_t k, uint32_t of) {
    work[2 + 2 * (first + k)] = tile;
    work[3 + 2 * (first + k)] = k | of << 16;
  };
  // a tile of many parts (a cluster) is written by the whole workgroup: by one
  // thread, 1000 parts took 40 us
  if (parts > 4) {
    const uint32_t b = atomicAdd(&s_many, 1u);
    s_list[b][0] = t;
    s_list[b][1] = at;
    s_list[b][2] = parts;
  } else {
    for (uint32_t k = 0; k < parts; k++) put(t, at, k, parts);
  }
  __syncthreads();
  for (uint32_t b = 0; b < s_many; b++)
    for (uint32_t k = tid; k < s_list[b][2]; k += 256)
      put(s_list[b][0], s_list[b][1], k, s_list[b][2]);
}

// particles of a part: enough parts for about four workgroups per CU where
// there are few tiles, and a tile that holds several times the average (dense
// plasma in a corner of the mesh) shared by as many workgroups, while each
// keeps `least` (512; 1D mixed, 10,000 cells at 80: 21 us a push, with 1024 or
// 2048 24; FP64 2D and 3D equal).  Parts then number at most n / per + ntiles <=
// items.
constexpr uint32_t RUN_WGS = 1024;

void cell_runs_shape(const Mesh &m, const int T[3], uint32_t least, CellRuns &cr) {
  cr.least = least;
  cr.ntiles = 1;
  for (int d = 0; d < 3; d++) {
    cr.nt[d] = d < m.dim ? (m.N[d] + T[d] - 1) / T[d] : 1;
    cr.ax[d] = make_tile_axis(m.N[d], cr.nt[d]);
    cr.ntiles *= (uint32_t)cr.nt[d];
  }
  cr.items = (cr.ntiles + (cr.ntiles > RUN_WGS ? cr.ntiles : RUN_WGS) + 7u) / 8u * 8u;
  cr.end = cr.guard_slots = 0;
}

static inline unsigned blocks_for(uint64_t n) {
  return (unsigned)((n + 255) / 256);
}

int key_bits(uint32_t max_key) {
  int b = 1;
  while (b < 32 && (1ull << b) <= (uint64_t)max_key) b++;
  return b;
}

// room for a growing count, as RtWork::ensure
hipError_t SortWork::ensure(uint64_t n) {
  if (n <= cap) return hipSuccess;
  const uint64_t slack = room_for(n, most);
  if (slack > n && slack <= 0x7fffffffull) {
    if (alloc(slack) == hipSuccess) return hipSuccess;
    (void)hipGetLastError();
  }
  return alloc(n);
}

hipError_t SortWork::alloc(uint64_t n) {
  release();
  hipError_t e;
  if ((e = hipMalloc(&keys_in, n * 4)) != hipSuccess) return e;
  if ((e = hipMalloc(&keys_out, n * 4)) != hipSuccess) return e;
  if ((e = hipMalloc(&perm_in, n * 4)) != hipSuccess) return e;
  if ((e = hipMalloc(&perm_out, n * 4)) != hipSuccess) return e;
  if ((e = hipMalloc(&count, sizeof(unsigned long long))) != hipSuccess)
    return e;
  size_t bytes = 0;
  e = hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, keys_in, keys_out,
                                         perm_in, perm_out, (int)n, 0, 32);
  if (e != hipSuccess) return e;
  if ((e = hipMalloc(&temp, bytes)) != hipSuccess) return e;
  temp_bytes = bytes;
  cap = n;
  return hipSuccess;
}

void SortWork::release() {
  (void)hipFree(keys_in);
  (void)hipFree(keys_out);
  (void)hipFree(perm_in);
  (void)hipFree(perm_out);
  (void)hipFree(count);
  (void)hipFree(temp);
  keys_in = keys_out = perm_in = perm_out = nullptr;
  count = nullptr;
  temp = nullptr;
  temp_bytes = 0;
  cap = 0;
}

hipError_t sort_keys(SortWork &w, const uint32_t *cell, uint64_t n,
                     uint32_t empty_key, const uint32_t *tile_key_lut,
                     hipStream_t st) {
  hipError_t e = w.ensure(n);
  if (e != hipSuccess) return e;
  k_make_keys<<<blocks_for(n), 256, 0, st>>>(cell, n, empty_key, tile_key_lut,
                                             w.keys_in, w.perm_in);
  size_t bytes = w.temp_bytes;
  e = hipcub::DeviceRadixSort::SortPairs(w.temp, bytes, w.keys_in,
                                         w.keys_out, w.perm_in, w.perm_out,
                                         (int)n, 0, key_bits(empty_key), st);
  if (e != hipSuccess) return e;
  k_count_valid<<<blocks_for(n), 256, 0, st>>>(w.keys_out, n, empty_key,
                                               w.count);
  return hipGetLastError();
}

hipError_t build_cell_runs(const Mesh &m, const CellRuns &cr, const uint32_t *keys, uint64_t n,
                           uint32_t *table, hipStream_t st) {
  const uint64_t entries = cell_runs_size(m, cr);
  k_cell_runs<<<blocks_for(entries), 256, 0, st>>>(m, cr, keys, n, table, entries);
  const uint64_t w = cr.ntiles > RUN_WGS ? cr.ntiles : RUN_WGS, per = (n + w - 1) / w;
  k_cell_work<<<(cr.ntiles + 255) / 256, 256, 0, st>>>(m, cr, per > cr.least ? per : cr.least,
                                                       table + entries);
  return hipGetLastError();
}

hipError_t hipcub_sort_pairs(SortWork &w, uint64_t n, int bits,
                             hipStream_t st) {
  size_t bytes = w.temp_bytes;
  return hipcub::DeviceRadixSort::SortPairs(w.temp, bytes, w.keys_in,
                                            w.keys_out, w.perm_in,
                                            w.perm_out, (int)n, 0, bits, st);
}

// particles and photons of the mixed form (9, 10 arrays of 4 bytes), of the
// FP64 form (2 of 4 bytes, 9 or 10 of 8 with the id)
hipError_t gather_set(SortWork &w, const GatherSet &g, uint64_t n, hipStream_t st) {
  const unsigned grid = blocks_for(n);
  auto is = [&](int n4, int n8) { return g.n4 == n4 && g.n8 == n8; };
  if (is(9, 0)) k_gather_set<9, 0><<<grid, 256, 0, st>>>(g, w.perm_out, n);
  else if (is(10, 0)) k_gather_set<10, 0><<<grid, 256, 0, st>>>(g, w.perm_out, n);
  else if (is(2, 9)) k_gather_set<2, 9><<<grid, 256, 0, st>>>(g, w.perm_out, n);
  else if (is(2, 10)) k_gather_set<2, 10><<<grid, 256, 0, st>>>(g, w.perm_out, n);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace apt
