// tfs_faces.hpp -- the cells' face lists (tfs_layout.hpp) on the device.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

#include "tfs_layout.hpp"

namespace tfs {

// What a kernel reads; a cell is addressed by its position k in the lists' order.
struct FaceSlots {
  int n;
  const long long *__restrict__ off;
  const unsigned *__restrict__ inc;
  const int *__restrict__ tptr;   // null if no cell has a tail
  const unsigned *__restrict__ tail;
  const int *__restrict__ orig;   // caller's cell at a position; null: the same
  __device__ int cell(int k) const { return orig ? orig[k] : k; }
};

// The entries of the cell at position k in ascending face order: get(i, e)
// loads what entry e needs (i: the entry's place, slots first, then the tails),
// put(e, value) takes them in order.  Up to eight entries are under way at a
// time; a wavefront's 64 cells are one slice.  The lanes past the last cell
// (k >= n) have no entries.
template <typename V, typename Get, typename Put>
__device__ __forceinline__ void each_face(const FaceSlots &L, int k, Get get, Put put) {
  constexpr int kBatch = 8;
  const int s = __builtin_amdgcn_readfirstlane(k / 64);
  const long long e0 = L.off[s];
  const int wd = (int)((L.off[s + 1] - e0) / 64);
  const long long base = e0 + k % 64;
  for (int j0 = 0; j0 < wd; j0 += kBatch) {
    unsigned e[kBatch];
    V v[kBatch];
#pragma unroll
    for (int j = 0; j < kBatch; ++j)
      if (j0 + j < wd) e[j] = L.inc[base + 64LL * (j0 + j)];
#pragma unroll
    for (int j = 0; j < kBatch; ++j)
      if (j0 + j < wd && e[j] != kNoFace) v[j] = get(base + 64LL * (j0 + j), e[j]);
#pragma unroll
    for (int j = 0; j < kBatch; ++j)
      if (j0 + j < wd && e[j] != kNoFace) put(e[j], v[j]);
  }
  if (L.tptr && k < L.n) {
    const long long t0 = L.off[(L.n + 63) / 64];
    for (int t = L.tptr[k]; t < L.tptr[k + 1]; ++t) put(L.tail[t], get(t0 + t, L.tail[t]));
  }
}

// The lists in device memory.
struct DevFaceLists {
  FaceSlots at{};
  int *of = nullptr;              // position of each caller cell, if reordered
  long long entries = 0;          // slots and tails
  void *mem[6] = {};
  // Threads for one lane per position, whole slices.
  long long lanes() const { return 64LL * ((at.n + 63) / 64); }
  bool upload(const FaceLists &F) {
    at.n = F.n;
    entries = F.off.back() + (long long)F.tail.size();
    auto up = [&](int k, const void *src, size_t bytes) -> void * {
      if (bytes == 0) return nullptr;
      if (hipMalloc(&mem[k], bytes) != hipSuccess) return nullptr;
      return hipMemcpy(mem[k], src, bytes, hipMemcpyHostToDevice) == hipSuccess ? mem[k] : nullptr;
    };
    at.off = (const long long *)up(0, F.off.data(), sizeof(long long) * F.off.size());
    at.inc = (const unsigned *)up(1, F.inc.data(), sizeof(unsigned) * F.inc.size());
    at.tptr = (const int *)up(2, F.tptr.data(), sizeof(int) * F.tptr.size());
    at.tail = (const unsigned *)up(3, F.tail.data(), sizeof(unsigned) * F.tail.size());
    at.orig = (const int *)up(4, F.orig.data(), sizeof(int) * F.orig.size());
    of = (int *)up(5, F.of.data(), sizeof(int) * F.of.size());
    return at.off && (F.inc.empty() || at.inc) && (F.tptr.empty() || at.tptr) &&
           (F.tail.empty() || at.tail) && (!F.reordered || (at.orig && of));
  }
  void release() {
    for (void *&p : mem) {
      if (p) (void)hipFree(p);
      p = nullptr;
    }
  }
};

}  // namespace tfs
