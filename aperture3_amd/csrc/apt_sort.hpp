// apt_sort.hpp -- scratch and entry points of the particle sort.
#pragma once
#include "apt_common.hpp"

namespace apt {

// Slots to have room for when n are needed now: half as much again for a count
// that grows, but no more than there can ever be (a set that fills its capacity
// takes what it needs and no more).
inline uint64_t room_for(uint64_t n, uint64_t most) {
  const uint64_t s = n + n / 2;
  return s < most ? s : n > most ? n : most;
}

struct SortWork {
  uint32_t *keys_in = nullptr, *keys_out = nullptr;
  uint32_t *perm_in = nullptr, *perm_out = nullptr;
  unsigned long long *count = nullptr;  // non-empty slots after the sort
  void *temp = nullptr;
  size_t temp_bytes = 0;
  uint64_t cap = 0;
  uint64_t most = 0;  // slots its owner can ever have: no room beyond
  hipError_t ensure(uint64_t n);
  hipError_t alloc(uint64_t n);
  void release();
};

int key_bits(uint32_t max_key);

// Sort slot indices by key (cell, or tile_key_lut[cell] when given);
// empty slots take empty_key and sort last.  Leaves the permutation in
// w.perm_out and the non-empty count in *w.count (device).
hipError_t sort_keys(SortWork &w, const uint32_t *cell, uint64_t n,
                     uint32_t empty_key, const uint32_t *tile_key_lut,
                     hipStream_t st);

// radix sort of (keys_in, perm_in) -> (keys_out, perm_out) on `bits` bits
hipError_t hipcub_sort_pairs(SortWork &w, uint64_t n, int bits,
                             hipStream_t st);

// The arrays of a particle set, gathered into sorted order together.
struct GatherSet {
  static constexpr int MAX4 = 12, MAX8 = 12;
  const uint32_t *src4[MAX4];  // of 4-byte elements
  uint32_t *dst4[MAX4];
  const uint64_t *src8[MAX8];  // of 8-byte elements
  uint64_t *dst8[MAX8];
  int n4 = 0, n8 = 0;
  template <typename T>
  void add(const T *src, T *dst) {
    static_assert(sizeof(T) == 4 || sizeof(T) == 8, "4- or 8-byte elements");
    if constexpr (sizeof(T) == 4) {
      src4[n4] = reinterpret_cast<const uint32_t *>(src);
      dst4[n4++] = reinterpret_cast<uint32_t *>(dst);
    } else {
      src8[n8] = reinterpret_cast<const uint64_t *>(src);
      dst8[n8++] = reinterpret_cast<uint64_t *>(dst);
    }
  }
};
// dst[i] = src[w.perm_out[i]], i < n, of every array
hipError_t gather_set(SortWork &w, const GatherSet &g, uint64_t n, hipStream_t st);

}  // namespace apt
