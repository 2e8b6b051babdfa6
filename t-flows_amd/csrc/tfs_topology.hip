// tfs_topology.hip -- the CRS topology of a face list, built on the device.
//
// Sources/Process/Matrix_Mod/Topology.f90 forms the matrix structure from the
// faces in four sequential loops: stencil widths (:34-41), row starts with the
// diagonal first (:54-59), off-diagonal columns appended in face order
// (:62-71), each row sorted ascending with its diagonal located (:75-82), and
// the two entries of every interior face located (:106-121).  Here:
//
//   k_width   one thread per face, atomic width counts per cell; the count an
//             atomic returns is the face's place in that row, kept per face;
//   k_scan_*  row starts: per-block sums, one scan of the block sums, per-block
//             rescan (an exclusive scan of width + 1 with 64-bit totals);
//   k_fill    one thread per face, no atomics: each face's two entries go to
//             the places k_width returned, each carrying a tag naming its face
//             and side (2 s + side);
//   k_sort    one thread per cell: insertion sort of its row's (column, tag)
//             pairs by column, the diagonal's position (the last entry equal
//             to the cell, as the reference's loop leaves it), and pos: every
//             tag in a run of equal columns gets the run's last position (the
//             reference's search keeps the last match).
//
// Atomics make the fill order nondeterministic, but a row holds a multiset of
// columns and sorting it fixes the order, so the result is bitwise the
// sequential one; tags only travel with their columns.  Everything is integer
// traffic; on a random numbering these kernels are bound by accesses of a memory
// line each, which meshes of more than a few cells avoid by buckets (below).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdint>

#include "tfs_solver.h"

namespace {

constexpr int kThreads = 256;
constexpr int kScanItems = 4;                       // per thread
constexpr int kScanTile = kThreads * kScanItems;    // cells per scan block

#define TFS_T_HIP(expr)        \
  do {                         \
    if ((expr) != hipSuccess) { \
      (void)hipGetLastError(); \
      rc = TFS_ERR_DEVICE;     \
      goto done;               \
    }                          \
  } while (0)

int grid_of(long long m) {
  long long g = (m + kThreads - 1) / kThreads;
  return (int)(g < 1 ? 1 : (g > 8192 ? 8192 : g));
}

__global__ void __launch_bounds__(kThreads) k_fill_int(long long m, int v, int *__restrict__ a) {
  for (long long i = blockIdx.x * (long long)kThreads + threadIdx.x; i < m;
       i += (long long)gridDim.x * kThreads)
    a[i] = v;
}

// widths of the off-diagonal part; err gets 1 for c1 outside 1..n or c2 > n
// (c2 <= 0 is a boundary face, as the reference's test c2 > 0 has it)
__global__ void __launch_bounds__(kThreads)
k_width(int n, long long nf, const int *__restrict__ faces, int *__restrict__ width,
        int2 *__restrict__ slot, int *__restrict__ err) {
  for (long long s = blockIdx.x * (long long)kThreads + threadIdx.x; s < nf;
       s += (long long)gridDim.x * kThreads) {
    const int2 f = reinterpret_cast<const int2 *>(faces)[s];
    if (f.x < 1 || f.x > n || f.y > n) {
      atomicOr(err, 1);
      continue;
    }
    if (f.y > 0) {
      // the count before this face is the face's place in each row, after
      // the diagonal
      const int k1 = atomicAdd(&width[f.x - 1], 1);
      const int k2 = atomicAdd(&width[f.y - 1], 1);
      slot[s] = make_int2(k1 + 1, k2 + 1);
    }
  }
}

// block sums of (width + 1) over tiles of kScanTile cells
__global__ void __launch_bounds__(kThreads)
k_scan_sums(int n, const int *__restrict__ width, long long *__restrict__ bsum) {
  __shared__ long long part[kThreads / 64];
  const long long base = (long long)blockIdx.x * kScanTile;
  long long t = 0;
  for (int k = 0; k < kScanItems; ++k) {
    const long long c = base + (long long)k * kThreads + threadIdx.x;
    if (c < n) t += width[c] + 1;
  }
  for (int o = 32; o > 0; o >>= 1) t += __shfl_down(t, o, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = t;
  __syncthreads();
  if (threadIdx.x == 0) {
    long long s = 0;
    for (int w = 0; w < kThreads / 64; ++w) s += part[w];
    bsum[blockIdx.x] = s;
  }
}

// exclusive scan of the block sums in place (one workgroup); total -> *total
__global__ void __launch_bounds__(kThreads)
k_scan_top(int nb, long long *__restrict__ bsum, long long *__restrict__ total) {
  __shared__ long long buf[kThreads];
  long long carry = 0;
  for (int b0 = 0; b0 < nb; b0 += kThreads) {
    const int b = b0 + threadIdx.x;
    const long long v = b < nb ? bsum[b] : 0;
    buf[threadIdx.x] = v;
    __syncthreads();
    for (int o = 1; o < kThreads; o <<= 1) {     // Hillis-Steele inclusive scan
      const long long add = threadIdx.x >= o ? buf[threadIdx.x - o] : 0;
      __syncthreads();
      buf[threadIdx.x] += add;
      __syncthreads();
    }
    if (b < nb) bsum[b] = carry + buf[threadIdx.x] - v;
    carry += buf[kThreads - 1];
    __syncthreads();
  }
  if (threadIdx.x == 0) *total = carry;
}

// row(c) = base + exclusive prefix of (width + 1); the diagonal goes first in
// its row (Topology.f90:54-59)
__global__ void __launch_bounds__(kThreads)
k_scan_rows(int n, int base, const long long *__restrict__ bsum, const int *__restrict__ width,
            int *__restrict__ row, int *__restrict__ col) {
  __shared__ int wsum[kThreads / 64];
  const long long t0 = (long long)blockIdx.x * kScanTile;
  // a thread's kScanItems consecutive cells
  int v[kScanItems], acc = 0;
  for (int k = 0; k < kScanItems; ++k) {
    const long long c = t0 + (long long)threadIdx.x * kScanItems + k;
    v[k] = c < n ? width[c] + 1 : 0;
    acc += v[k];
  }
  // exclusive scan of the per-thread totals: within the wave, then waves
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int inc = acc;
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(inc, o, 64);
    if (lane >= o) inc += y;
  }
  if (lane == 63) wsum[wv] = inc;
  __syncthreads();
  int before = 0;
  for (int w = 0; w < wv; ++w) before += wsum[w];
  long long off = bsum[blockIdx.x] + base + before + inc - acc;
  for (int k = 0; k < kScanItems; ++k) {
    const long long c = t0 + (long long)threadIdx.x * kScanItems + k;
    if (c < n) {
      row[c] = (int)off;
      col[off - base] = (int)c + base;
      if (c == n - 1) row[n] = (int)(off + v[k]);
    }
    off += v[k];
  }
}

// off-diagonal columns at the places k_width gave the face in its two rows
// (Topology.f90:62-71); the entry's tag 2 s + side locates pos(side + 1, s)
// after the sort; boundary faces get pos = base - 1 here
__global__ void __launch_bounds__(kThreads)
k_fill(long long nf, int base, const int *__restrict__ faces, const int *__restrict__ row,
       const int2 *__restrict__ slot, int *__restrict__ col, long long *__restrict__ tag,
       int *__restrict__ pos) {
  for (long long s = blockIdx.x * (long long)kThreads + threadIdx.x; s < nf;
       s += (long long)gridDim.x * kThreads) {
    const int2 f = reinterpret_cast<const int2 *>(faces)[s];
    if (f.y > 0) {
      const int c1 = f.x - 1, c2 = f.y - 1;
      const int2 k = slot[s];
      const long long q1 = row[c1] - base + k.x;
      const long long q2 = row[c2] - base + k.y;
      col[q1] = c2 + base;
      col[q2] = c1 + base;
      if (tag) {
        tag[q1] = 2 * s;
        tag[q2] = 2 * s + 1;
      }
    } else if (pos) {
      reinterpret_cast<int2 *>(pos)[s] = make_int2(base - 1, base - 1);
    }
  }
}

constexpr int kRegRow = 16;   // rows up to this long are sorted in registers

// One row of at most kRegRow entries: loaded once, sorted by an odd-even
// transposition network (stable: only strictly greater keys move down, so the
// padding keys stay behind every real entry), written back once.
__device__ __forceinline__ void sort_row_regs(int c, long long b, int w, int base,
                                              int *__restrict__ col, long long *__restrict__ tag,
                                              int *__restrict__ dia, int *__restrict__ pos) {
  int k[kRegRow];
  long long t[kRegRow];
#pragma unroll
  for (int i = 0; i < kRegRow; ++i) {
    k[i] = i < w ? col[b + i] : INT_MAX;
    t[i] = (tag && i < w) ? tag[b + i] : -1;
  }
#pragma unroll
  for (int pass = 0; pass < kRegRow; ++pass) {
#pragma unroll
    for (int i = pass & 1; i + 1 < kRegRow; i += 2) {
      if (k[i] > k[i + 1]) {
        const int kk = k[i];
        k[i] = k[i + 1];
        k[i + 1] = kk;
        const long long tt = t[i];
        t[i] = t[i + 1];
        t[i + 1] = tt;
      }
    }
  }
  int d = 0;
#pragma unroll
  for (int i = 0; i < kRegRow; ++i) {
    if (i < w) {
      col[b + i] = k[i];
      if (k[i] == c + base) d = i;
    }
  }
  dia[c] = (int)(b + d + base);
  if (!tag) return;
  // from the end: `last` is the end of the current run of equal columns
  int last = kRegRow - 1;
#pragma unroll
  for (int i = kRegRow - 1; i >= 0; --i) {
    if (i < w) {
      if (i == w - 1 || k[i] != k[last]) last = i;
      if (t[i] >= 0) pos[t[i]] = (int)(b + last + base);
    }
  }
}

// ascending columns per row with their tags, the diagonal's position
// (Topology.f90:75-82), and the face positions (:106-121)
__global__ void __launch_bounds__(kThreads)
k_sort(int n, int base, const int *__restrict__ row, int *__restrict__ col,
       long long *__restrict__ tag, int *__restrict__ dia, int *__restrict__ pos) {
  for (int c = blockIdx.x * kThreads + threadIdx.x; c < n; c += gridDim.x * kThreads) {
    const long long b = row[c] - base, e = row[c + 1] - base;
    if (e - b <= kRegRow) {
      sort_row_regs(c, b, (int)(e - b), base, col, tag, dia, pos);
      continue;
    }
    // longer rows: insertion sort in place
    for (long long q = b + 1; q < e; ++q) {
      const int key = col[q];
      const long long t = tag ? tag[q] : 0;
      long long r = q;
      while (r > b && col[r - 1] > key) {
        col[r] = col[r - 1];
        if (tag) tag[r] = tag[r - 1];
        --r;
      }
      col[r] = key;
      if (tag) tag[r] = t;
    }
    long long d = b;
    for (long long q = b; q < e; ++q)
      if (col[q] == c + base) d = q;
    dia[c] = (int)(d + base);
    if (!tag) continue;
    // walk down the row: `last` is the end of the current run of equal columns
    long long last = e - 1;
    for (long long q = e - 1; q >= b; --q) {
      if (col[q] != col[last]) last = q;
      const long long t = tag[q];
      if (t >= 0) pos[t] = (int)(last + base);
    }
  }
}

// ---- by buckets of cells ------------------------------------------------------------
// On a mesh numbered at random every access above is a memory line of its own:
// two atomics, two row starts, two columns, two tags and two positions a face
// (128^3: 505 us of k_width, 616 of k_fill, 279 of k_sort).  Here the entries
// first go to buckets of consecutive cells whose rows fit in LDS:
//
//   k_bucket_count  entries per bucket, counted per workgroup in LDS;
//   k_bucket_scan   where each bucket's rows start;
//   k_bucket_fill   each workgroup reserves a run in every bucket and writes its
//                   faces' entries there (column, cell within the bucket) --
//                   runs of several entries, which meet in the caches -- and
//                   notes each entry's place with its face;
//   k_bucket_rows   one workgroup per bucket: row starts, the rows in LDS, sorted
//                   one lane a row, written in runs; the entries' final places
//                   go back to where the entries stood;
//   k_bucket_pos    per face, the places of its two entries, again in runs.
//
// A bucket's entries stand in its own part of col until its rows replace them.
// Same results: a row is a multiset of columns, and pos is the last place of its
// column whatever the order of equal ones.  Whole calls on
// MI355X: 128^3 numbered at random 2016 -> 695 us (k_bucket_fill 283, k_bucket_pos
// 142, k_bucket_rows 128, k_bucket_count 26), in order 891 -> 426; 64^3 334 -> 212;
// 32^3 144 -> 107; below that the same.
constexpr int kBucketEntries = 10000;   // entries and diagonals of a bucket: 60 KB of LDS
constexpr int kBucketMax = 16384;       // buckets: as many LDS counters
constexpr int kBucketFrom = 1 << 15;    // cells from which buckets are used
constexpr int kCountThreads = 1024;

struct BucketInfo { long long total; int widest, err; };

__global__ void __launch_bounds__(kCountThreads)
k_bucket_count(int n, long long nf, long long per, int shift, int nb,
               const int2 *__restrict__ faces, int *__restrict__ count, BucketInfo *info) {
  extern __shared__ int hist[];
  for (int b = threadIdx.x; b < nb; b += kCountThreads) hist[b] = 0;
  __syncthreads();
  const long long s0 = blockIdx.x * per, s1 = s0 + per < nf ? s0 + per : nf;
  for (long long s = s0 + threadIdx.x; s < s1; s += kCountThreads) {
    const int2 f = faces[s];
    if (f.x < 1 || f.x > n || f.y > n) {
      atomicOr(&info->err, 1);
    } else if (f.y > 0) {
      atomicAdd(&hist[(f.x - 1) >> shift], 1);
      atomicAdd(&hist[(f.y - 1) >> shift], 1);
    }
  }
  __syncthreads();
  for (int b = threadIdx.x; b < nb; b += kCountThreads)
    if (hist[b]) atomicAdd(&count[b], hist[b]);
}

// first[b]: where bucket b's rows start (its entries before, and a diagonal a
// cell); cursor the same, for k_bucket_fill.  One workgroup.
__global__ void __launch_bounds__(kCountThreads)
k_bucket_scan(int n, int shift, int nb, const int *__restrict__ count, int *__restrict__ first,
              int *__restrict__ cursor, BucketInfo *info) {
  __shared__ long long wsum[kCountThreads / 64];
  __shared__ int wmax[kCountThreads / 64];
  const int per = (nb + kCountThreads - 1) / kCountThreads;
  const int b0 = min(nb, (int)threadIdx.x * per), b1 = min(nb, b0 + per);
  const auto rows = [&](int b) {   // entries and diagonals
    return (long long)count[b] + min(n - (b << shift), 1 << shift);
  };
  long long acc = 0;
  int widest = 0;
  for (int b = b0; b < b1; ++b) {
    const long long r = rows(b);
    acc += r;
    widest = max(widest, (int)(r < INT_MAX ? r : INT_MAX));
  }
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  long long inc = acc;
  for (int o = 1; o < 64; o <<= 1) {
    const long long y = __shfl_up(inc, o, 64);
    if (lane >= o) inc += y;
  }
  for (int o = 32; o > 0; o >>= 1) widest = max(widest, __shfl_xor(widest, o, 64));
  if (lane == 63) wsum[wv] = inc;
  if (lane == 0) wmax[wv] = widest;
  __syncthreads();
  long long at = inc - acc, total = 0;
  for (int w = 0; w < kCountThreads / 64; ++w) {
    if (w < wv) at += wsum[w];
    total += wsum[w];
    widest = max(widest, wmax[w]);
  }
  for (int b = b0; b < b1; ++b) {   // a total past 2^31 ends the call before these are used
    first[b] = cursor[b] = (int)at;
    at += rows(b);
  }
  if (threadIdx.x == 0) {
    first[nb] = (int)total;
    info->total = total;
    info->widest = widest;
  }
}

__global__ void __launch_bounds__(kCountThreads)
k_bucket_fill(long long nf, long long per, int shift, int nb, int base,
              const int2 *__restrict__ faces, int *__restrict__ cursor, int *__restrict__ col,
              int *__restrict__ local, int2 *__restrict__ pos) {
  extern __shared__ int hist[];
  for (int b = threadIdx.x; b < nb; b += kCountThreads) hist[b] = 0;
  __syncthreads();
  const long long s0 = blockIdx.x * per, s1 = s0 + per < nf ? s0 + per : nf;
  for (long long s = s0 + threadIdx.x; s < s1; s += kCountThreads) {
    const int2 f = faces[s];
    if (f.y > 0) {
      atomicAdd(&hist[(f.x - 1) >> shift], 1);
      atomicAdd(&hist[(f.y - 1) >> shift], 1);
    }
  }
  __syncthreads();
  for (int b = threadIdx.x; b < nb; b += kCountThreads)
    if (hist[b]) hist[b] = atomicAdd(&cursor[b], hist[b]);   // this workgroup's run
  __syncthreads();
  const int mask = (1 << shift) - 1;
  for (long long s = s0 + threadIdx.x; s < s1; s += kCountThreads) {
    const int2 f = faces[s];
    if (f.y <= 0) continue;
    const int c1 = f.x - 1, c2 = f.y - 1;
    const int q1 = atomicAdd(&hist[c1 >> shift], 1), q2 = atomicAdd(&hist[c2 >> shift], 1);
    col[q1] = c2 + base;
    col[q2] = c1 + base;
    local[q1] = c1 & mask;
    local[q2] = c2 & mask;
    if (pos) pos[s] = make_int2(q1, q2);
  }
}

// One row of w entries in LDS, sorted by column (the entry's number breaks ties);
// returns the place of the last entry equal to `self`, and puts each numbered
// entry's final place -- the last of its column -- into place[].
template <int W>
__device__ __forceinline__ int sort_row_lds(int *colb, unsigned short *tagb, int w, int self,
                                            int at, int *place) {
  unsigned long long k[W];
#pragma unroll
  for (int i = 0; i < W; ++i)   // columns are not negative
    k[i] = i < w ? (unsigned long long)(unsigned)colb[i] << 16 | tagb[i] : ~0ull;
#pragma unroll
  for (int pass = 0; pass < W; ++pass) {
#pragma unroll
    for (int i = pass & 1; i + 1 < W; i += 2) {
      const unsigned long long a = k[i], b = k[i + 1];
      k[i] = a < b ? a : b;
      k[i + 1] = a < b ? b : a;
    }
  }
  int d = 0, last = 0;
#pragma unroll
  for (int i = W - 1; i >= 0; --i) {
    if (i < w) {
      const int c = (int)(k[i] >> 16), t = (int)(k[i] & 0xffffu);
      if (i == w - 1 || c != (int)(k[i + 1 < W ? i + 1 : i] >> 16)) last = i;
      if (c == self && d < i) d = i;
      colb[i] = c;
      if (place && t != 0xffff) place[t] = at + last;
    }
  }
  return d;
}

__device__ int sort_row_long(int *colb, unsigned short *tagb, int w, int self, int at,
                             int *place) {
  for (int q = 1; q < w; ++q) {
    const int c = colb[q];
    const unsigned short t = tagb[q];
    int r = q;
    for (; r > 0 && colb[r - 1] > c; --r) {
      colb[r] = colb[r - 1];
      tagb[r] = tagb[r - 1];
    }
    colb[r] = c;
    tagb[r] = t;
  }
  int d = 0, last = w - 1;
  for (int i = w - 1; i >= 0; --i) {
    if (colb[i] != colb[last]) last = i;
    if (colb[i] == self && d < i) d = i;
    if (place && tagb[i] != 0xffff) place[tagb[i]] = at + last;
  }
  return d;
}

// local: the entries' cells within the bucket on entry; with `places`, their
// final places on return.
__global__ void __launch_bounds__(kThreads)
k_bucket_rows(int n, int shift, int nb, int base, const int *__restrict__ first,
              int *__restrict__ row, int *__restrict__ col, int *__restrict__ local,
              int *__restrict__ dia, int places) {
  extern __shared__ int lds[];
  const int cells_max = 1 << shift;
  int *const start = lds;                  // each row's start, then its cursor
  int *const colb = lds + cells_max;
  __shared__ int wsum[kThreads / 64];
  const int b = blockIdx.x, c0 = b << shift, cells = min(n - c0, cells_max);
  const int q0 = first[b], rows = first[b + 1] - q0, m = rows - cells;
  unsigned short *const tagb = reinterpret_cast<unsigned short *>(colb + rows);
  for (int c = threadIdx.x; c < cells_max; c += kThreads) start[c] = 0;
  __syncthreads();
  for (int e = threadIdx.x; e < m; e += kThreads) atomicAdd(&start[local[q0 + e]], 1);
  __syncthreads();
  // exclusive scan of width + 1, a run of cells per thread
  const int per = (cells_max + kThreads - 1) / kThreads;
  const int lo = min(cells, (int)threadIdx.x * per), hi = min(cells, lo + per);
  int acc = 0;
  for (int c = lo; c < hi; ++c) acc += start[c] + 1;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int inc = acc;
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(inc, o, 64);
    if (lane >= o) inc += y;
  }
  if (lane == 63) wsum[wv] = inc;
  __syncthreads();
  int off = inc - acc;
  for (int w = 0; w < wv; ++w) off += wsum[w];
  for (int c = lo; c < hi; ++c) {
    const int w = start[c] + 1;
    row[c0 + c] = q0 + off + base;
    colb[off] = c0 + c + base;   // the diagonal goes first (Topology.f90:54-59)
    tagb[off] = 0xffff;
    start[c] = off + 1;
    off += w;
  }
  if (b == nb - 1 && threadIdx.x == 0) row[n] = q0 + rows + base;
  __syncthreads();
  for (int e = threadIdx.x; e < m; e += kThreads) {
    const int k = atomicAdd(&start[local[q0 + e]], 1);
    colb[k] = col[q0 + e];
    tagb[k] = (unsigned short)e;
  }
  __syncthreads();
  // start[c] is now the end of row c
  int *const place = places ? local + q0 : nullptr;
  for (int c = threadIdx.x; c < cells; c += kThreads) {
    const int r0 = c ? start[c - 1] : 0, w = start[c] - r0, self = c0 + c + base;
    const int at = q0 + r0 + base;
    const int d = w <= 8 ? sort_row_lds<8>(colb + r0, tagb + r0, w, self, at, place)
                  : w <= kRegRow ? sort_row_lds<kRegRow>(colb + r0, tagb + r0, w, self, at, place)
                                 : sort_row_long(colb + r0, tagb + r0, w, self, at, place);
    dia[c0 + c] = at + d;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < rows; i += kThreads) col[q0 + i] = colb[i];
}

__global__ void __launch_bounds__(kThreads)
k_bucket_pos(long long nf, int base, const int2 *__restrict__ faces,
             const int *__restrict__ place, int2 *__restrict__ pos) {
  for (long long s = blockIdx.x * (long long)kThreads + threadIdx.x; s < nf;
       s += (long long)gridDim.x * kThreads) {
    const int2 q = pos[s];
    pos[s] = faces[s].y > 0 ? make_int2(place[q.x], place[q.y]) : make_int2(base - 1, base - 1);
  }
}

// The log2 of the cells per bucket for this mesh, -1 where the kernels above
// are used: too many buckets, or so few cells that launches are all there is
// to save.
int bucket_shift(int n, long long nf) {
  if (nf == 0) return -1;
  const double entries = 2.0 * (double)nf / n + 1.0;   // per cell, at most
  for (int shift = 10; shift >= 6; --shift)
    if (1.25 * entries * (1 << shift) <= kBucketEntries)
      return n >= kBucketFrom && (n - 1) / (1 << shift) < kBucketMax ? shift : -1;
  return -1;
}

// The topology by buckets; false, with nothing written but scratch, where a
// bucket does not fit (some cells have very many faces).
bool bucket_topology(int n, long long nf, const int *d_faces, int base, long long col_cap,
                     int *d_row, int *d_col, int *d_dia, int *d_pos, int shift, int *result,
                     long long *nnz) {
  const hipStream_t st = nullptr;
  const int nb = (n - 1) / (1 << shift) + 1;
  const int2 *const faces = reinterpret_cast<const int2 *>(d_faces);
  int2 *const pos = reinterpret_cast<int2 *>(d_pos);
  // faces per workgroup: eight entries a bucket make runs worth it (sixteen
  // measured no faster), and smaller meshes are spread over the chip
  const long long per = std::max(4LL * nb, std::min(8192LL, std::max(1024LL, nf / 512)));
  const int grid = (int)((nf + per - 1) / per);
  const size_t hist = sizeof(int) * (size_t)nb;
  char *mem = nullptr;   // info, counts, starts, cursors, the entries' cells
  const size_t head = sizeof(BucketInfo) + sizeof(int) * (3 * (size_t)nb + 1);
  BucketInfo h{};
  bool mine = true;
  int rc = TFS_OK;
  if (hipMallocAsync((void **)&mem, head + sizeof(int) * (size_t)(n + 2 * nf), st) != hipSuccess) {
    (void)hipGetLastError();
    *result = TFS_ERR_NOMEM;
    return true;
  }
  BucketInfo *const info = reinterpret_cast<BucketInfo *>(mem);
  int *const count = reinterpret_cast<int *>(info + 1);
  int *const first = count + nb, *const cursor = first + nb + 1, *const local = cursor + nb;
  hipLaunchKernelGGL(k_fill_int, dim3(grid_of(nb)), dim3(kThreads), 0, st,
                     (long long)(sizeof(BucketInfo) / sizeof(int)) + nb, 0,
                     reinterpret_cast<int *>(info));
  hipLaunchKernelGGL(k_bucket_count, dim3(grid), dim3(kCountThreads), hist, st, n, nf, per, shift,
                     nb, faces, count, info);
  hipLaunchKernelGGL(k_bucket_scan, dim3(1), dim3(kCountThreads), 0, st, n, shift, nb, count,
                     first, cursor, info);
  TFS_T_HIP(hipGetLastError());
  TFS_T_HIP(hipMemcpy(&h, info, sizeof(h), hipMemcpyDeviceToHost));
  if (h.err) {
    rc = TFS_ERR_INVALID;
    goto done;
  }
  if (h.total > INT_MAX - 1 || h.total > col_cap) {
    rc = TFS_ERR_INVALID;
    if (nnz) *nnz = h.total;
    goto done;
  }
  if (h.widest > kBucketEntries) {
    mine = false;
    goto done;
  }
  hipLaunchKernelGGL(k_bucket_fill, dim3(grid), dim3(kCountThreads), hist, st, nf, per, shift, nb,
                     base, faces, cursor, d_col, local, pos);
  hipLaunchKernelGGL(k_bucket_rows, dim3(nb), dim3(kThreads),
                     sizeof(int) * ((size_t)1 << shift) + (sizeof(int) + sizeof(short)) *
                                                             (size_t)h.widest,
                     st, n, shift, nb, base, first, d_row, d_col, local, d_dia, pos ? 1 : 0);
  if (pos)
    hipLaunchKernelGGL(k_bucket_pos, dim3(grid_of(nf)), dim3(kThreads), 0, st, nf, base, faces,
                       local, pos);
  TFS_T_HIP(hipGetLastError());
  TFS_T_HIP(hipStreamSynchronize(st));
  if (nnz) *nnz = h.total;
done:
  (void)hipFreeAsync(mem, st);
  *result = rc;
  return mine;
}

}  // namespace

extern "C" int tfs_topology_build_device(int n_cells, long long n_faces, const int *d_faces_c,
                                         int base, long long col_cap, int *d_row, int *d_col,
                                         int *d_dia, int *d_pos, long long *nnz) {
  if (n_cells < 1 || n_faces < 0 || (base != 0 && base != 1) || !d_row || !d_col || !d_dia ||
      (n_faces > 0 && !d_faces_c) || col_cap < n_cells)
    return TFS_ERR_INVALID;
  // faces and pos are read and written as (c1, c2) / (pos1, pos2) pairs
  if ((reinterpret_cast<uintptr_t>(d_faces_c) | reinterpret_cast<uintptr_t>(d_pos)) % 8 != 0)
    return TFS_ERR_INVALID;
  if (nnz) *nnz = 0;
  int rc = TFS_OK;
  const int shift = bucket_shift(n_cells, n_faces);
  if (shift >= 0 && bucket_topology(n_cells, n_faces, d_faces_c, base, col_cap, d_row, d_col,
                                    d_dia, d_pos, shift, &rc, nnz))
    return rc;
  const int nb = (int)((n_cells + (long long)kScanTile - 1) / kScanTile);
  int *width = nullptr, *err = nullptr;
  int2 *slot = nullptr;
  long long *bsum = nullptr, *total = nullptr, *tag = nullptr;
  int h_err = 0;
  long long h_total = 0;
  const hipStream_t st = nullptr;    // the calling thread's default stream
  // scratch from the stream-ordered pool: no device-wide synchronisation on
  // allocation or release
  if (hipMallocAsync((void **)&width, sizeof(int) * (size_t)n_cells, st) != hipSuccess ||
      hipMallocAsync((void **)&bsum, sizeof(long long) * (size_t)nb + 2 * sizeof(long long), st) !=
          hipSuccess ||
      hipMallocAsync((void **)&slot, sizeof(int2) * (size_t)(n_faces > 0 ? n_faces : 1), st) !=
          hipSuccess) {
    (void)hipGetLastError();
    rc = TFS_ERR_NOMEM;
    goto done;
  }
  total = bsum + nb;
  err = reinterpret_cast<int *>(bsum + nb + 1);
  hipLaunchKernelGGL(k_fill_int, dim3(grid_of(n_cells)), dim3(kThreads), 0, st,
                     (long long)n_cells, 0, width);
  hipLaunchKernelGGL(k_fill_int, dim3(1), dim3(kThreads), 0, st, 1LL, 0, err);
  if (n_faces > 0)
    hipLaunchKernelGGL(k_width, dim3(grid_of(n_faces)), dim3(kThreads), 0, st, n_cells, n_faces,
                       d_faces_c, width, slot, err);
  hipLaunchKernelGGL(k_scan_sums, dim3(nb), dim3(kThreads), 0, st, n_cells, width, bsum);
  hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(kThreads), 0, st, nb, bsum, total);
  TFS_T_HIP(hipGetLastError());
  TFS_T_HIP(hipMemcpy(&h_total, total, sizeof(long long), hipMemcpyDeviceToHost));
  TFS_T_HIP(hipMemcpy(&h_err, err, sizeof(int), hipMemcpyDeviceToHost));
  if (h_err) {
    rc = TFS_ERR_INVALID;
    goto done;
  }
  if (h_total > INT_MAX - 1 || h_total > col_cap) {
    rc = TFS_ERR_INVALID;
    if (nnz) *nnz = h_total;
    goto done;
  }
  if (d_pos) {
    if (hipMallocAsync((void **)&tag, sizeof(long long) * (size_t)h_total, st) != hipSuccess) {
      (void)hipGetLastError();
      rc = TFS_ERR_NOMEM;
      goto done;
    }
    // the diagonal entries keep tag -1 (k_scan_rows writes only their column)
    hipLaunchKernelGGL(k_fill_int, dim3(grid_of(2 * h_total)), dim3(kThreads), 0, st,
                       2 * h_total, -1, reinterpret_cast<int *>(tag));
  }
  hipLaunchKernelGGL(k_scan_rows, dim3(nb), dim3(kThreads), 0, st, n_cells, base, bsum, width,
                     d_row, d_col);
  if (n_faces > 0)
    hipLaunchKernelGGL(k_fill, dim3(grid_of(n_faces)), dim3(kThreads), 0, st, n_faces, base,
                       d_faces_c, d_row, slot, d_col, tag, d_pos);
  hipLaunchKernelGGL(k_sort, dim3(grid_of(n_cells)), dim3(kThreads), 0, st, n_cells, base, d_row,
                     d_col, tag, d_dia, d_pos);
  TFS_T_HIP(hipGetLastError());
  TFS_T_HIP(hipStreamSynchronize(st));
  if (nnz) *nnz = h_total;
done:
  for (void *p : {(void *)width, (void *)bsum, (void *)slot, (void *)tag})
    if (p) (void)hipFreeAsync(p, st);
  return rc;
}
