// tfs_layout_capi.cpp -- the solver's host-side layout builders behind a C
// ABI in the CPU library (libtfs_mesh.so), so that the permutations and level
// structures the device code relies on can be checked without a GPU.
#include <cstddef>
#include <vector>

#include "tfs_layout.hpp"
#include "tfs_mesh.h"

extern "C" int tfs_layout_block_colour(int n, const int *row, const int *col, int block,
                                       int *perm, int *colour) {
  if (n < 0 || block < 1 || (n > 0 && (!row || !col || !perm || !colour))) return -1;
  std::vector<int> p, c;
  const int ncol = tfs::colour_order(n, row, col, p, &c, block);
  for (int i = 0; i < n; ++i) {
    perm[i] = p[i];
    colour[i] = c[i];
  }
  return ncol;
}

extern "C" int tfs_layout_colour(int n, const int *row, const int *col, int *perm, int *colour) {
  if (n < 0 || (n > 0 && (!row || !col || !perm || !colour))) return -1;
  std::vector<int> p, c;
  const int ncol = tfs::colour_order(n, row, col, p, &c);
  for (int i = 0; i < n; ++i) {
    perm[i] = p[i];
    colour[i] = c[i];
  }
  return ncol;
}

extern "C" int tfs_layout_summary(int n, const int *row, const int *col, const int *dia,
                                  int *s_orig, int *level_lower, int *level_upper,
                                  int *bandwidth) {
  if (n < 1 || !row || !col || !dia || !s_orig || !level_lower || !level_upper || !bandwidth)
    return -1;
  tfs::Layout L;
  tfs::build_layout(n, row, col, dia, 64, 512, 2048, L);
  for (int i = 0; i < n; ++i) s_orig[i] = L.s_orig[i];
  for (const tfs::SweepLayout *S : {&L.L, &L.U}) {
    int *lev = S == &L.L ? level_lower : level_upper;
    for (int l = 0; l < S->nlev; ++l)
      for (int q = S->lev_ptr[l]; q < S->lev_ptr[l + 1]; ++q) lev[S->orig[q]] = l;
  }
  *bandwidth = L.bandwidth;
  return 0;
}

extern "C" int tfs_layout_block_colour_bfs(int n, const int *row, const int *col, int block,
                                           int *perm, int *colour, int *block_of) {
  if (n < 0 || block < 1 || (n > 0 && (!row || !col || !perm || !colour || !block_of)))
    return -1;
  std::vector<int> p, c, b;
  const int ncol = tfs::block_colour_order(n, row, col, block, p, &c, &b);
  for (int i = 0; i < n; ++i) {
    perm[i] = p[i];
    colour[i] = c[i];
    block_of[i] = b[i];
  }
  return ncol;
}

extern "C" int tfs_layout_brick_colour(int n, const int *row, const int *col, const int *dia,
                                       int edge, int cap, int *perm, int *colour,
                                       int *block_of) {
  if (n < 0 || edge < 1 || cap < 1 ||
      (n > 0 && (!row || !col || !dia || !perm || !colour || !block_of)))
    return -1;
  std::vector<int> p, bstart, bcolour;
  const int ncol = tfs::brick_colour_order(n, row, col, dia, edge, cap, p, bstart, bcolour);
  for (std::size_t b = 0; b + 1 < bstart.size(); ++b)
    for (int k = bstart[b]; k < bstart[b + 1]; ++k) {
      perm[k] = p[(size_t)k];
      colour[p[(size_t)k]] = bcolour[b];
      block_of[p[(size_t)k]] = (int)b;
    }
  return ncol;
}

extern "C" int tfs_layout_blocks(int n, const int *row, const int *col, const int *dia, int *order,
                                 int *block_of, int *step_of) {
  if (n < 1 || !row || !col || !dia || !order || !block_of || !step_of) return -1;
  tfs::Layout L;
  tfs::build_layout(n, row, col, dia, 64, 512, 2048, L);
  tfs::BlockLayout B;
  tfs::build_blocks(n, row, col, dia, L.s_of_orig, L.L.nlev, B);
  if (!B.ok) return 0;
  for (int b = 0; b < B.nblk; ++b) {
    const tfs::Block &K = B.L.blk[(std::size_t)b];
    for (int t = 0; t < K.steps; ++t)
      for (int p = B.L.step[(std::size_t)(K.step0 + t)];
           p < B.L.step[(std::size_t)(K.step0 + t + 1)]; ++p) {
        const int i = B.orig[(std::size_t)(K.row0 + p)];
        order[K.row0 + p] = i;
        block_of[i] = b;
        step_of[i] = t;
      }
  }
  return B.nblk;
}

extern "C" int tfs_layout_faces(int n, long long nf, const int *faces, int base, int from,
                                int *order, int *first, unsigned *entry) {
  if (n < 1 || nf < 0 || (nf > 0 && !faces) || !order || !first || !entry) return -1;
  tfs::FaceLists F;
  tfs::build_face_lists(n, nf, faces, base, from, F);
  int at = 0;
  for (int c = 0; c < n; ++c) {
    const int k = F.at(c), s = k / 64;
    const int wd = (int)((F.off[(std::size_t)s + 1] - F.off[(std::size_t)s]) / 64);
    order[k] = c;
    first[c] = at;
    for (int j = 0; j < wd; ++j) {
      const unsigned e = F.inc[(std::size_t)(F.off[(std::size_t)s] + 64LL * j + k % 64)];
      if (e != tfs::kNoFace) entry[at++] = e;
    }
    if (!F.tptr.empty())
      for (int t = F.tptr[(std::size_t)k]; t < F.tptr[(std::size_t)k + 1]; ++t)
        entry[at++] = F.tail[(std::size_t)t];
  }
  first[n] = at;
  return F.reordered ? 1 : 0;
}

extern "C" int tfs_layout_short_columns(int nslice, const long long *off, const int *col,
                                        int *out) {
  if (nslice < 0 || !off || (off[nslice] > 0 && (!col || !out))) return -1;
  tfs::ShortColumns S;
  tfs::short_columns(std::vector<long long>(off, off + nslice + 1),
                     std::vector<int>(col, col + off[nslice]), S);
  if (!S.ok) return 0;
  for (int s = 0; s < nslice; ++s)
    for (long long i = off[s]; i < off[s + 1]; ++i) {
      const long long slot = (i - off[s]) / 64, lane = (i - off[s]) % 64;
      const unsigned h = S.code[(std::size_t)(S.off[(std::size_t)s] + 64 * (slot / 2) + lane)] >>
                             (slot % 2 ? 16 : 0) & 0xffffu;
      out[i] = S.window[(std::size_t)s * tfs::kWindows + (h >> 12)] + (int)(h & 0xfffu);
    }
  return 1;
}
