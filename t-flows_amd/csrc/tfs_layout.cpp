// tfs_layout.cpp -- host-side construction of the S / L / U layouts.
#include "tfs_layout.hpp"

#include <algorithm>
#include <atomic>
#include <climits>
#include <cstdint>
#include <future>
#include <unordered_map>
#include <cstdlib>

namespace tfs {
namespace {

// The upper layout is the lower one backwards (see build_sweep).
constexpr bool kMirrorUpper = true;

// How parts of a layout of n rows are built beside one another: on a thread of
// their own (where one can be had) or, where that would cost as much, in turn.
// ms of a box's layout and blocks on eight cores, in turn / beside one another:
// 26^3 5.0 / 5.4, 32^3 9.7 / 6.9, 48^3 37.5 / 25.7.
inline std::launch beside(int n) {
  return n < 1 << 15 ? std::launch::deferred : std::launch::async | std::launch::deferred;
}

// Breadth-first search from `start` over nodes whose mark differs from
// `stamp` (marking them); neighbours are taken in ascending degree, ties by
// number (Cuthill-McKee).  Appends the visit order to `out`, returns the
// number of BFS levels and, if asked, the nodes of the last level.
int cm_bfs(int start, int stamp, const std::vector<int> &row, const std::vector<int> &adj,
           const std::vector<int> &deg, std::vector<int> &mark, std::vector<int> &out,
           std::vector<int> *last_level) {
  size_t head = out.size(), level_begin = head, level_end = head + 1;
  out.push_back(start);
  mark[start] = stamp;
  int levels = 1;
  std::vector<int> nb;
  while (head < out.size()) {
    if (head == level_end) {
      level_begin = level_end;
      level_end = out.size();
      ++levels;
    }
    const int v = out[head++];
    nb.clear();
    for (int e = row[v]; e < row[v + 1]; ++e)
      if (mark[adj[e]] != stamp) {
        mark[adj[e]] = stamp;
        nb.push_back(adj[e]);
      }
    std::sort(nb.begin(), nb.end(), [&](int a, int b) {
      return deg[a] != deg[b] ? deg[a] < deg[b] : a < b;
    });
    out.insert(out.end(), nb.begin(), nb.end());
  }
  if (last_level) last_level->assign(out.begin() + (long)level_begin, out.end());
  return levels;
}

// Whether every entry has its mirror (columns ascend, as they do in a matrix).
bool symmetric_structure(int n, const int *row, const int *col) {
  std::vector<int> next(row, row + n);  // per row, the first lower entry not yet mirrored
  for (int i = 0; i < n; ++i) {
    int lower = 0;
    for (int e = row[i]; e < row[i + 1]; ++e) {
      const int k = col[e];
      if (e > row[i] && k <= col[e - 1]) return false;
      lower += k < i;
      if (k <= i) continue;
      // row k's lower columns ascend, so their mirrors come in order
      if (next[(size_t)k] >= row[k + 1] || col[next[(size_t)k]] != i) return false;
      ++next[(size_t)k];
    }
    if (next[(size_t)i] != row[i] + lower) return false;
  }
  return true;
}

// Reverse Cuthill-McKee (Cuthill & McKee 1969; George 1971), starting each
// connected component from a pseudo-peripheral node (George & Liu 1979).
std::vector<int> rcm(int n, const int *row, const int *col) {
  // symmetric adjacency without the diagonal
  std::vector<int> arow(n + 1, 0), a2;
  if (symmetric_structure(n, row, col)) {
    a2.reserve((size_t)row[n]);
    for (int i = 0; i < n; ++i) {
      for (int e = row[i]; e < row[i + 1]; ++e)
        if (col[e] != i) a2.push_back(col[e]);
      arow[i + 1] = (int)a2.size();
    }
  } else {
    std::vector<int> cnt(n + 1, 0);
    for (int i = 0; i < n; ++i)
      for (int e = row[i]; e < row[i + 1]; ++e)
        if (col[e] != i) {
          cnt[i + 1]++;
          cnt[col[e] + 1]++;
        }
    for (int i = 0; i < n; ++i) cnt[i + 1] += cnt[i];
    std::vector<int> adj(cnt[n]), fill(cnt.begin(), cnt.end() - 1);
    for (int i = 0; i < n; ++i)
      for (int e = row[i]; e < row[i + 1]; ++e)
        if (col[e] != i) {
          adj[fill[i]++] = col[e];
          adj[fill[col[e]]++] = i;
        }
    // drop duplicates (a pair that has its mirror is listed twice)
    a2.reserve(adj.size() / 2 + 1);
    for (int i = 0; i < n; ++i) {
      std::sort(adj.begin() + cnt[i], adj.begin() + cnt[i + 1]);
      int prev = -1;
      for (int e = cnt[i]; e < cnt[i + 1]; ++e)
        if (adj[e] != prev) a2.push_back(prev = adj[e]);
      arow[i + 1] = (int)a2.size();
    }
  }
  std::vector<int> deg(n);
  for (int i = 0; i < n; ++i) deg[i] = arow[i + 1] - arow[i];

  // mark: 0 = unvisited; 1 = placed in `order`; >= 2 = probe stamps
  std::vector<int> mark(n, 0), order, tmp, last;
  order.reserve(n);
  int stamp = 2;
  for (int s0 = 0; s0 < n; ++s0) {
    if (mark[s0] == 1) continue;
    int r = s0, ecc = -1;
    for (int it = 0; it < 4; ++it) {
      tmp.clear();
      // probe BFS inside the component (placed nodes carry mark 1 and are
      // in other components, so they are never reached)
      const int levels = cm_bfs(r, stamp++, arow, a2, deg, mark, tmp, &last);
      if (levels <= ecc) break;
      ecc = levels;
      int best = last[0];
      for (int v : last)
        if (deg[v] < deg[best] || (deg[v] == deg[best] && v < best)) best = v;
      r = best;
    }
    cm_bfs(r, 1, arow, a2, deg, mark, order, nullptr);
  }
  std::reverse(order.begin(), order.end());
  return order;  // order[k] = caller row placed at position k
}

// With `mirror` (the lower layout, for the upper triangle) the levels are
// the lower levels counted from the deepest one, ties in reverse S order: the
// upper order is then the lower order backwards.  That is a valid order for
// the backward sweep (a row's upper dependencies have larger caller numbers,
// hence deeper lower levels, hence earlier mirrored positions), has the same
// number of levels as its own level order, and lets the backward sweep read
// the forward sweep's output and re-arm it in contiguous runs.
void build_sweep(int n, const int *row, const int *col, const int *dia, bool lower,
                 const std::vector<int> &s_of_orig, int small_level, SweepLayout &S,
                 const SweepLayout *mirror = nullptr) {
  std::vector<int> lev(n, 0);
  int nlev = 0;
  if (mirror) {
    nlev = mirror->nlev;
    for (int l = 0; l < nlev; ++l)
      for (int p = mirror->lev_ptr[l]; p < mirror->lev_ptr[l + 1]; ++p)
        lev[mirror->orig[p]] = nlev - 1 - l;
  } else if (lower) {
    for (int i = 0; i < n; ++i) {
      int l = 0;
      for (int j = row[i]; j < dia[i]; ++j) l = std::max(l, lev[col[j]] + 1);
      lev[i] = l;
      nlev = std::max(nlev, l + 1);
    }
  } else {
    for (int i = n - 1; i >= 0; --i) {
      int l = 0;
      for (int j = dia[i] + 1; j < row[i + 1]; ++j) l = std::max(l, lev[col[j]] + 1);
      lev[i] = l;
      nlev = std::max(nlev, l + 1);
    }
  }
  S.nlev = nlev;
  S.lev_ptr.assign(nlev + 1, 0);
  for (int i = 0; i < n; ++i) S.lev_ptr[lev[i] + 1]++;
  for (int l = 0; l < nlev; ++l) S.lev_ptr[l + 1] += S.lev_ptr[l];
  // order: by level, ties in S order (walk caller rows in S order), or in
  // reverse S order for a mirrored layout
  std::vector<int> s_orig(n);
  for (int i = 0; i < n; ++i) s_orig[s_of_orig[i]] = i;
  std::vector<int> fill(S.lev_ptr.begin(), S.lev_ptr.end() - 1);
  S.orig.assign(n, 0);
  S.of_orig.assign(n, 0);
  for (int k = 0; k < n; ++k) {
    const int i = s_orig[mirror ? n - 1 - k : k];
    const int p = fill[lev[i]]++;
    S.orig[p] = i;
    S.of_orig[i] = p;
  }
  S.ptr.assign(n + 1, 0);
  for (int p = 0; p < n; ++p) {
    const int i = S.orig[p];
    S.ptr[p + 1] = S.ptr[p] + (lower ? dia[i] - row[i] : row[i + 1] - dia[i] - 1);
  }
  S.col.assign(S.ptr[n], 0);
  S.src.assign(S.ptr[n], 0);
  S.diag_src.assign(n, 0);
  for (int p = 0; p < n; ++p) {
    const int i = S.orig[p];
    const int j0 = lower ? row[i] : dia[i] + 1, j1 = lower ? dia[i] : row[i + 1];
    int e = S.ptr[p];
    for (int j = j0; j < j1; ++j, ++e) {
      S.col[e] = S.of_orig[col[j]];
      S.src[e] = j;
    }
    S.diag_src[p] = dia[i];
  }
  S.segs.clear();
  for (int l = 0; l < nlev; ++l) {
    const int rows = S.lev_ptr[l + 1] - S.lev_ptr[l];
    const bool small = rows <= small_level;
    if (small && !S.segs.empty() && S.segs.back().small) {
      S.segs.back().l1 = l + 1;
      S.segs.back().rows += rows;
    } else {
      S.segs.push_back({l, l + 1, rows, small});
    }
  }
}

// The brick blocks of rows [r0, r1), which no entry couples to other rows:
// blk[i] for each of them (numbered from 0 in order of the groups' first rows);
// returns their number.  See brick_colour_order.  With `split`, index steps of
// at most three binary orders are a class each, whatever their counts (a box
// whose shorter sides come first merges two of them otherwise).
int brick_blocks(int r0, int r1, const int *row, const int *col, const int *dia, int edge, int cap,
                 bool split, int *blk) {
  const int n = r1 - r0;
  // classes of the dependencies j -> i by the binary order of i - j
  constexpr int kClasses = 3;
  std::vector<long long> hist(32, 0);
  auto order_of = [](unsigned d) { return 31 - __builtin_clz(d); };
  long long ntri = 0;
  for (int i = r0; i < r1; ++i)
    for (int e = row[i]; e < dia[i]; ++e) {
      hist[order_of((unsigned)(i - col[e]))]++;
      ++ntri;
    }
  std::vector<int> cls(32, 0);
  {
    int c = 0;
    long long acc = 0;
    bool any = false;
    int orders = 0;
    for (int o = 0; o < 32; ++o) orders += hist[o] > 0;
    const bool own = split && orders <= kClasses;
    for (int o = 0; o < 32; ++o) {
      if (!hist[o]) continue;
      if (any && c < kClasses - 1 && (own || acc * kClasses >= (long long)(c + 1) * ntri)) ++c;
      cls[o] = c;
      acc += hist[o];
      any = true;
    }
  }
  // potentials, row by row in caller order (dependencies come first)
  std::vector<int> phi((size_t)n * kClasses, 0);
  for (int i = r0; i < r1; ++i) {
    int *f = &phi[(size_t)(i - r0) * kClasses];
    for (int e = row[i]; e < dia[i]; ++e) {
      const int j = col[e], c = cls[order_of((unsigned)(i - j))];
      const int *g = &phi[(size_t)(j - r0) * kClasses];
      for (int k = 0; k < kClasses; ++k) f[k] = std::max(f[k], g[k] + (k == c ? 1 : 0));
    }
  }
  // groups: one id per distinct brick key, in order of their first row; a
  // group's rows in caller order, split into blocks of at most cap rows
  long long span = 1;
  for (size_t i = 0; i < phi.size(); ++i) span = std::max<long long>(span, phi[i] / edge + 1);
  std::unordered_map<long long, int> gid;
  gid.reserve((size_t)n / (size_t)std::max(1, edge * edge * edge) + 16);
  std::vector<int> grp(n);
  std::vector<int> gcount;
  long long last = -1;  // the row before mostly has the same key
  for (int i = 0; i < n; ++i) {
    const int *f = &phi[(size_t)i * kClasses];
    const long long key = (f[0] / edge) + span * ((f[1] / edge) + span * (long long)(f[2] / edge));
    if (key == last) {
      grp[i] = grp[i - 1];
    } else {
      auto it = gid.find(key);
      if (it == gid.end()) {
        it = gid.emplace(key, (int)gcount.size()).first;
        gcount.push_back(0);
      }
      grp[i] = it->second;
      last = key;
    }
    gcount[(size_t)grp[i]]++;
  }
  std::vector<int>().swap(phi);
  const int ng = (int)gcount.size();
  std::vector<int> gfirst((size_t)ng + 1, 0);  // blocks of each group
  for (int g = 0; g < ng; ++g) gfirst[(size_t)g + 1] = gfirst[(size_t)g] + (gcount[(size_t)g] + cap - 1) / cap;
  const int nb = gfirst[(size_t)ng];
  std::vector<int> seen_in_group((size_t)ng, 0);
  for (int i = 0; i < n; ++i) {
    const int g = grp[i];
    blk[r0 + i] = gfirst[(size_t)g] + seen_in_group[(size_t)g]++ / cap;
  }
  return nb;
}

}  // namespace

int colour_order(int n, const int *row, const int *col, std::vector<int> &perm,
                 std::vector<int> *colour_out, int block) {
  // symmetrised adjacency: the pattern may be unsymmetric
  std::vector<int> deg(n + 1, 0);
  for (int i = 0; i < n; ++i)
    for (int k = row[i]; k < row[i + 1]; ++k)
      if (col[k] != i) {
        deg[i + 1]++;
        deg[col[k] + 1]++;
      }
  for (int i = 0; i < n; ++i) deg[i + 1] += deg[i];
  std::vector<int> adj(deg[n]), fill(deg.begin(), deg.end() - 1);
  for (int i = 0; i < n; ++i)
    for (int k = row[i]; k < row[i + 1]; ++k)
      if (col[k] != i) {
        adj[fill[i]++] = col[k];
        adj[fill[col[k]]++] = i;
      }
  // blocks of `block` consecutive rows are coloured as units: a block takes
  // the smallest colour that no neighbouring block has
  block = std::max(1, block);
  const int nb = (n + block - 1) / block;
  std::vector<int> bcol(nb, -1), seen;  // seen[c] == B: colour c taken by a neighbour of B
  int ncol = 0;
  for (int B = 0; B < nb; ++B) {
    const int i0 = B * block, i1 = std::min(n, i0 + block);
    for (int i = i0; i < i1; ++i)
      for (int k = deg[i]; k < deg[i + 1]; ++k) {
        const int Bj = adj[k] / block;
        if (Bj != B && bcol[Bj] >= 0) seen[bcol[Bj]] = B;
      }
    int c = 0;
    while (c < ncol && seen[c] == B) ++c;
    if (c == ncol) {
      ++ncol;
      seen.push_back(-1);
    }
    bcol[B] = c;
  }
  std::vector<int> colour(n);
  for (int i = 0; i < n; ++i) colour[i] = bcol[i / block];
  std::vector<int> start(ncol + 1, 0);
  for (int i = 0; i < n; ++i) start[colour[i] + 1]++;
  for (int c = 0; c < ncol; ++c) start[c + 1] += start[c];
  perm.assign(n, 0);
  for (int i = 0; i < n; ++i) perm[start[colour[i]]++] = i;
  if (colour_out) *colour_out = std::move(colour);
  return ncol;
}

int block_colour_order(int n, const int *row, const int *col, int block, std::vector<int> &perm,
                       std::vector<int> *colour_out, std::vector<int> *block_out) {
  // symmetrised adjacency, each row's neighbours ascending and distinct
  std::vector<int> deg(n + 1, 0);
  for (int i = 0; i < n; ++i)
    for (int k = row[i]; k < row[i + 1]; ++k)
      if (col[k] != i) {
        deg[i + 1]++;
        deg[col[k] + 1]++;
      }
  for (int i = 0; i < n; ++i) deg[i + 1] += deg[i];
  std::vector<int> adj(deg[n]), fill(deg.begin(), deg.end() - 1);
  for (int i = 0; i < n; ++i)
    for (int k = row[i]; k < row[i + 1]; ++k)
      if (col[k] != i) {
        adj[fill[i]++] = col[k];
        adj[fill[col[k]]++] = i;
      }
  for (int i = 0; i < n; ++i) std::sort(adj.begin() + deg[i], adj.begin() + deg[i + 1]);
  block = std::max(1, block);
  // blocks grown breadth-first from the lowest unassigned vertex
  std::vector<int> blk(n, -1), order;  // order: vertices block by block, discovery order
  std::vector<int> bstart(1, 0);
  order.reserve(n);
  for (int s = 0; s < n; ++s) {
    if (blk[s] >= 0) continue;
    const int b = (int)bstart.size() - 1;
    size_t head = order.size();
    const size_t first = head;
    blk[s] = b;
    order.push_back(s);
    while (head < order.size() && (int)(order.size() - first) < block) {
      const int v = order[head++];
      for (int e = deg[v]; e < deg[v + 1] && (int)(order.size() - first) < block; ++e) {
        const int w = adj[e];
        if (blk[w] < 0) {
          blk[w] = b;
          order.push_back(w);
        }
      }
    }
    bstart.push_back((int)order.size());
  }
  const int nb = (int)bstart.size() - 1;
  // greedy colouring of the block graph, blocks in growth order
  std::vector<int> bcol(nb, -1), seen;
  int ncol = 0;
  for (int B = 0; B < nb; ++B) {
    for (int k = bstart[B]; k < bstart[B + 1]; ++k) {
      const int v = order[k];
      for (int e = deg[v]; e < deg[v + 1]; ++e) {
        const int Bj = blk[adj[e]];
        if (Bj != B && bcol[Bj] >= 0) seen[bcol[Bj]] = B;
      }
    }
    int c = 0;
    while (c < ncol && seen[c] == B) ++c;
    if (c == ncol) {
      ++ncol;
      seen.push_back(-1);
    }
    bcol[B] = c;
  }
  // colour, then block, then discovery order
  std::vector<int> cstart(ncol + 1, 0);
  for (int B = 0; B < nb; ++B) cstart[bcol[B] + 1] += bstart[B + 1] - bstart[B];
  for (int c = 0; c < ncol; ++c) cstart[c + 1] += cstart[c];
  perm.assign(n, 0);
  for (int B = 0; B < nb; ++B)
    for (int k = bstart[B]; k < bstart[B + 1]; ++k) perm[cstart[bcol[B]]++] = order[k];
  if (colour_out) {
    colour_out->assign(n, 0);
    for (int i = 0; i < n; ++i) (*colour_out)[i] = bcol[blk[i]];
  }
  if (block_out) *block_out = std::move(blk);
  return ncol;
}

int brick_colour_order(int n, const int *row, const int *col, const int *dia, int edge, int cap,
                       std::vector<int> &perm, std::vector<int> &bstart,
                       std::vector<int> &bcolour) {
  perm.clear();
  bstart.assign(1, 0);
  bcolour.clear();
  if (n <= 0) return 0;
  edge = std::max(1, edge);
  cap = std::max(1, cap);
  std::vector<int> blk(n);
  const int nb = brick_blocks(0, n, row, col, dia, edge, cap, false, blk.data());
  // greedy colouring of the block graph (symmetrised pattern), blocks in id order
  std::vector<int> bstart_c((size_t)nb + 1, 0);
  for (int i = 0; i < n; ++i) bstart_c[(size_t)blk[i] + 1]++;
  for (int b = 0; b < nb; ++b) bstart_c[(size_t)b + 1] += bstart_c[(size_t)b];
  std::vector<int> rows_of((size_t)n), fill(bstart_c.begin(), bstart_c.end() - 1);
  for (int i = 0; i < n; ++i) rows_of[(size_t)fill[(size_t)blk[i]]++] = i;  // caller order within
  // upper neighbours too: a block must differ from every adjacent block
  std::vector<int> deg(n + 1, 0);
  for (int i = 0; i < n; ++i)
    for (int e = row[i]; e < row[i + 1]; ++e)
      if (col[e] != i) {
        deg[i + 1]++;
        deg[col[e] + 1]++;
      }
  for (int i = 0; i < n; ++i) deg[i + 1] += deg[i];
  std::vector<int> adj((size_t)deg[n]);
  {
    std::vector<int> f2(deg.begin(), deg.end() - 1);
    for (int i = 0; i < n; ++i)
      for (int e = row[i]; e < row[i + 1]; ++e)
        if (col[e] != i) {
          adj[(size_t)f2[i]++] = col[e];
          adj[(size_t)f2[col[e]]++] = i;
        }
  }
  std::vector<int> bcol((size_t)nb, -1), taken;
  int ncol = 0;
  for (int b = 0; b < nb; ++b) {
    for (int k = bstart_c[(size_t)b]; k < bstart_c[(size_t)b + 1]; ++k) {
      const int v = rows_of[(size_t)k];
      for (int e = deg[v]; e < deg[v + 1]; ++e) {
        const int bb = blk[(size_t)adj[(size_t)e]];
        if (bb != b && bcol[(size_t)bb] >= 0) taken[(size_t)bcol[(size_t)bb]] = b;
      }
    }
    int c = 0;
    while (c < ncol && taken[(size_t)c] == b) ++c;
    if (c == ncol) {
      ++ncol;
      taken.push_back(-1);
    }
    bcol[(size_t)b] = c;
  }
  // order: colour, block, caller order
  std::vector<int> cstart((size_t)ncol + 1, 0);
  for (int b = 0; b < nb; ++b) cstart[(size_t)bcol[(size_t)b] + 1]++;
  for (int c = 0; c < ncol; ++c) cstart[(size_t)c + 1] += cstart[(size_t)c];
  std::vector<int> border((size_t)nb);
  {
    std::vector<int> f3(cstart.begin(), cstart.end() - 1);
    for (int b = 0; b < nb; ++b) border[(size_t)f3[(size_t)bcol[(size_t)b]]++] = b;
  }
  perm.reserve(n);
  bstart.reserve((size_t)nb + 1);
  bcolour.reserve(nb);
  for (int k = 0; k < nb; ++k) {
    const int b = border[(size_t)k];
    for (int q = bstart_c[(size_t)b]; q < bstart_c[(size_t)b + 1]; ++q) perm.push_back(rows_of[(size_t)q]);
    bstart.push_back((int)perm.size());
    bcolour.push_back(bcol[(size_t)b]);
  }
  return ncol;
}

namespace {

// One triangle of the blocks in block order: `of_orig` the position of each caller
// row, blocks [bstart[b], bstart[b + 1]), per position its block and its level in it;
// the upper triangle has everything backwards.  False if a limit is exceeded.
// The entries go to their rows' places in one pass over the caller's rows, whose
// neighbours' positions then come in runs; the halo is numbered from there.
bool build_block_triangle(int n, const int *row, const int *col, const int *dia, bool lower,
                          const std::vector<int> &of_orig, const std::vector<int> &bstart,
                          const std::vector<int> &block_at, const std::vector<int> &lstep,
                          int width, int places, BlockTriangle &T) {
  const int nb = (int)bstart.size() - 1;
  auto start = [&](int b) { return lower ? bstart[(size_t)b] : n - bstart[(size_t)(nb - b)]; };
  auto mirror = [&](int p) { return lower ? p : n - 1 - p; };   // position <-> lower position
  auto level = [&](int p) { return lower ? lstep[(size_t)p] : -lstep[(size_t)(n - 1 - p)]; };
  T.blk.resize((size_t)nb);
  size_t padded = 0;
  for (int b = 0; b < nb; ++b) {
    Block &B = T.blk[(size_t)b];
    B.row0 = start(b);
    B.rows = start(b + 1) - B.row0;
    B.rpad = (B.rows + 7) & ~7;
    if ((size_t)width * (padded + (size_t)B.rpad) > 0x7fffffffu) return false;
    B.ent0 = (int)((size_t)width * padded);
    B.idx0 = (int)padded;
    padded += (size_t)B.rpad;
  }
  T.src.assign((size_t)width * padded, -1);
  T.idx.assign((size_t)places * padded, 0);
  std::vector<int> dep((size_t)width * (size_t)n, -1);   // positions of each row's entries
  for (int i = 0; i < n; ++i) {
    const int at = mirror(of_orig[(size_t)i]);
    const int b = block_at[(size_t)of_orig[(size_t)i]];
    const Block &B = T.blk[(size_t)(lower ? b : nb - 1 - b)];
    const int j0 = lower ? row[i] : dia[i] + 1, j1 = lower ? dia[i] : row[i + 1];
    int *const from = &T.src[(size_t)B.ent0 + (size_t)(at - B.row0)];
    for (int j = j0; j < j1; ++j) {
      dep[(size_t)width * (size_t)at + (size_t)(j - j0)] = mirror(of_orig[(size_t)col[j]]);
      from[(size_t)(j - j0) * (size_t)B.rpad] = j;
    }
  }
  // halo number of a position in this block: a table that stays in the caches
  constexpr unsigned kTable = 1024;
  static_assert(kTable > 2 * kBlockHalo, "entries of the halo table");
  struct Slot { int block = -1, q = 0, h = 0; };
  std::vector<Slot> table(kTable);
  for (int b = 0; b < nb; ++b) {
    Block &B = T.blk[(size_t)b];
    B.halo0 = (int)T.halo.size();
    B.step0 = (int)T.step.size();
    B.halo = 0;
    for (int p = 0; p < B.rows; ++p) {
      const int lev = level(B.row0 + p);
      const int *const d = &dep[(size_t)width * (size_t)(B.row0 + p)];
      unsigned short *const at = &T.idx[(size_t)(B.idx0 + p) * (size_t)places];
      for (int k = 0; k < width && d[k] >= 0; ++k) {
        const int q = d[k];
        int slot;
        if (q >= B.row0 && q < B.row0 + B.rows) {
          if (level(q) >= lev) return false;
          slot = 1 + q - B.row0;
        } else {
          if (q > B.row0) return false;  // only earlier blocks
          unsigned t = (unsigned)q * 2654435761u >> 22;
          while (table[t].block == b && table[t].q != q) t = (t + 1) % kTable;
          if (table[t].block != b) {
            if (B.halo == kBlockHalo) return false;
            table[t].block = b;
            table[t].q = q;
            table[t].h = B.halo++;
            T.halo.push_back(q);
          }
          slot = 1 + B.rows + table[t].h;
        }
        at[k] = (unsigned short)(slot * sizeof(double));
      }
      // a step: one lane per row, so at most a wavefront of one level's rows
      if (p == 0 || lev != level(B.row0 + p - 1) || p - T.step.back() == kBlockLanes)
        T.step.push_back((unsigned short)p);
    }
    B.steps = (int)T.step.size() - B.step0;
    T.step.push_back((unsigned short)B.rows);
    if (B.steps > kBlockSteps) return false;
    T.halo_max = std::max(T.halo_max, B.halo);
  }
  return true;
}

}  // namespace

void build_blocks(int n, const int *row, const int *col, const int *dia,
                  const std::vector<int> &s_of_orig, int nlev, BlockLayout &out) {
  out = BlockLayout();
  if (n <= 0 || nlev < kBlockLevels) return;
  // the triangles: at most kBlockWide entries a row, and structurally
  // symmetric (the upper sweep runs the lower order backwards, which needs
  // every upper entry to mirror a lower one)
  int width = 0;
  for (int i = 0; i < n; ++i)
    width = std::max({width, dia[i] - row[i], row[i + 1] - dia[i] - 1});
  if (width > kBlockWide || !symmetric_structure(n, row, col)) return;
  out.width = width <= 3 ? 3 : kBlockWide;
  // blocks per range of rows that no entry leaves (the systems of a batch)
  std::vector<int> blk((size_t)n);
  int nb = 0;
  for (int r0 = 0, reach = 0, i = 0; i < n; ++i) {
    reach = std::max(reach, col[row[i + 1] - 1]);
    if (reach > i) continue;
    const int m = brick_blocks(r0, i + 1, row, col, dia, kBlockEdge, kBlockRows, true, blk.data());
    for (int k = r0; k <= i; ++k) blk[(size_t)k] += nb;
    nb += m;
    r0 = i + 1;
  }
  // depth of each block in the block graph (its edges, sorted and distinct)
  std::vector<long long> edges;
  for (int i = 0; i < n; ++i)
    for (int j = row[i]; j < dia[i]; ++j) {
      const int from = blk[(size_t)col[j]], to = blk[(size_t)i];
      if (from == to) continue;
      const long long e = (long long)from * nb + to;
      if (edges.empty() || edges.back() != e) edges.push_back(e);
    }
  std::sort(edges.begin(), edges.end());
  edges.erase(std::unique(edges.begin(), edges.end()), edges.end());
  std::vector<int> indeg((size_t)nb, 0), lev((size_t)nb, 0), order;
  std::vector<size_t> first((size_t)nb + 1, 0);
  for (long long e : edges) {
    indeg[(size_t)(e % nb)]++;
    first[(size_t)(e / nb) + 1]++;
  }
  for (int b = 0; b < nb; ++b) first[(size_t)b + 1] += first[(size_t)b];
  order.reserve((size_t)nb);
  for (int b = 0; b < nb; ++b)
    if (!indeg[(size_t)b]) order.push_back(b);
  int depth = 0;
  for (size_t k = 0; k < order.size(); ++k) {
    const int b = order[k];
    depth = std::max(depth, lev[(size_t)b] + 1);
    for (size_t e = first[(size_t)b]; e < first[(size_t)b + 1]; ++e) {
      const int to = (int)(edges[e] % nb);
      lev[(size_t)to] = std::max(lev[(size_t)to], lev[(size_t)b] + 1);
      if (--indeg[(size_t)to] == 0) order.push_back(to);
    }
  }
  if ((int)order.size() != nb || (long long)depth * kBlockGain > nlev) return;
  // blocks by depth (then number), rows of a block by their level inside it,
  // ties in S order (whose right-hand side they gather)
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
    return lev[(size_t)a] != lev[(size_t)b] ? lev[(size_t)a] < lev[(size_t)b] : a < b;
  });
  std::vector<int> place((size_t)nb);
  for (int k = 0; k < nb; ++k) place[(size_t)order[(size_t)k]] = k;
  std::vector<int> rlev((size_t)n, 0), bstart((size_t)nb + 1, 0);
  for (int i = 0; i < n; ++i) {
    for (int j = row[i]; j < dia[i]; ++j)
      if (blk[(size_t)col[j]] == blk[(size_t)i])
        rlev[(size_t)i] = std::max(rlev[(size_t)i], rlev[(size_t)col[j]] + 1);
    bstart[(size_t)place[(size_t)blk[(size_t)i]] + 1]++;
  }
  for (int k = 0; k < nb; ++k) bstart[(size_t)k + 1] += bstart[(size_t)k];
  out.orig.resize((size_t)n);
  {
    std::vector<int> fill(bstart.begin(), bstart.end() - 1);
    for (int i = 0; i < n; ++i)
      out.orig[(size_t)fill[(size_t)place[(size_t)blk[(size_t)i]]]++] = i;
  }
  for (int k = 0; k < nb; ++k)
    std::sort(out.orig.begin() + bstart[(size_t)k], out.orig.begin() + bstart[(size_t)k + 1],
              [&](int a, int b) {
                return rlev[(size_t)a] != rlev[(size_t)b]
                           ? rlev[(size_t)a] < rlev[(size_t)b]
                           : s_of_orig[(size_t)a] < s_of_orig[(size_t)b];
              });
  out.of_orig.resize((size_t)n);
  for (int p = 0; p < n; ++p) out.of_orig[(size_t)out.orig[(size_t)p]] = p;
  std::vector<int> lstep((size_t)n);
  for (int p = 0; p < n; ++p) lstep[(size_t)p] = rlev[(size_t)out.orig[(size_t)p]];
  long long steps = 0;
  for (int k = 0; k < nb; ++k)
    for (int p = bstart[(size_t)k], first = p; p < bstart[(size_t)k + 1]; ++p)
      if (p == bstart[(size_t)k] || lstep[(size_t)p] != lstep[(size_t)p - 1] ||
          p - first == kBlockLanes) {
        first = p;
        ++steps;
      }
  if ((out.width > 3 ? 2.0 : 1.0) * (kBlockNs * nb + kBlockStepNs * (double)steps) >
      kLevelNs * nlev + kRowNs * n)
    return;
  std::vector<int> block_at((size_t)n);
  for (int k = 0; k < nb; ++k)
    std::fill(block_at.begin() + bstart[(size_t)k], block_at.begin() + bstart[(size_t)k + 1], k);
  auto triangle = [&](bool lower) {
    return build_block_triangle(n, row, col, dia, lower, out.of_orig, bstart, block_at, lstep,
                                out.width, out.places(), lower ? out.L : out.U);
  };
  std::future<bool> upper = std::async(beside(n), triangle, false);
  const bool fits = triangle(true);
  if (!upper.get() || !fits) return;
  out.nblk = nb;
  out.depth = depth;
  out.ok = true;
}

void build_bricks(int n, const int *row, const int *col, const int *dia,
                  const std::vector<int> &blk, const std::vector<int> &colour,
                  const std::vector<int> &s_of, BrickLayout &out) {
  out = BrickLayout();
  if (n <= 0 || n > 0x07ffffff) return;  // 32-bit byte offsets of 16-byte records
  const int nb = (int)colour.size();
  int ncol = 0;
  for (int c : colour) ncol = std::max(ncol, c + 1);
  // units: blocks by colour, then number, merged up to kUnitFull rows
  std::vector<int> unit_of((size_t)nb), brows((size_t)nb, 0), count;
  for (int i = 0; i < n; ++i) brows[(size_t)blk[(size_t)i]]++;
  out.colour0.assign(1, 0);
  for (int c = 0; c < ncol; ++c) {
    bool open = false;
    for (int b = 0; b < nb; ++b) {
      if (colour[(size_t)b] != c) continue;
      if (!open || count.back() + brows[(size_t)b] > kUnitFull) count.push_back(0);
      open = true;
      unit_of[(size_t)b] = (int)count.size() - 1;
      count.back() += brows[(size_t)b];
    }
    out.colour0.push_back((int)count.size());
  }
  const int nu = (int)count.size();
  std::vector<int> first((size_t)nu + 1, 0);
  for (int k = 0; k < nu; ++k) first[(size_t)k + 1] = first[(size_t)k] + count[(size_t)k];
  out.row.resize((size_t)n);
  {
    std::vector<int> fill(first.begin(), first.end() - 1);
    for (int i = 0; i < n; ++i)
      out.row[(size_t)fill[(size_t)unit_of[(size_t)blk[(size_t)i]]]++] = i;
  }
  auto nlow = [&](int i) { return dia[i] - row[i]; };
  auto nup = [&](int i) { return row[i + 1] - dia[i] - 1; };
  // per row its level in its block, its step in the unit, then (per triangle) its slot
  std::vector<int> lev((size_t)n, 0), step_of((size_t)n), slot((size_t)n, -1);
  out.unit.resize((size_t)nu);
  // Units go in parts beside one another, each with its own steps, second records
  // and halos, which are joined after.
  struct Joined {
    std::vector<BrickStep> step;
    std::vector<int> halo;
    std::vector<BrickPlaces> more_idx;
    std::vector<BrickSource> more_src;
    int slots = 0;
  };
  struct Part {
    Joined of[2];   // lower, upper
    int first = 0, last = 0, steps = 0;
    bool ok = true;
  };
  std::vector<Part> part((size_t)kBeside);
  for (BrickTriangle *T : {&out.L, &out.U}) {
    T->idx.resize((size_t)n);
    T->src.resize((size_t)n);
  }
  in_parts(nu, 64, [&](int which, int k0, int k1) {
    Part &P = part[(size_t)which];
    P.first = k0;
    P.last = k1;
    P.ok = false;
    // the halo number of a row in this unit and triangle
    constexpr unsigned kTable = 1 << 15;
    constexpr size_t kHaloMost = 0x3ffe;   // more leave no slot for a row (16-bit offsets)
    struct Entry { int when = -1, y = 0, h = 0; };
    std::vector<Entry> table(kTable);
    auto halo_at = [&](int stamp, int y) -> Entry & {
      unsigned t = (unsigned)y * 2654435761u >> 17;
      while (table[t].when == stamp && table[t].y != y) t = (t + 1) % kTable;
      return table[t];
    };
    std::vector<int> halo, hlast, last, start, unused;   // start: first row of each step
    std::vector<std::pair<uint64_t, int>> keys;
    std::vector<std::vector<int>> dies;           // slots whose last reader is in a step
    for (int k = k0; k < k1; ++k) {
      BrickUnit &B = out.unit[(size_t)k];
      B.row0 = first[(size_t)k];
      B.rows = count[(size_t)k];
      B.step0 = (int)P.of[0].step.size();
      if (B.rows > kUnitRows) return;
      int *const r = out.row.data() + B.row0;
      // levels inside the blocks, and the couplings between them
      int wl = 0, wu = 0;
      for (int p = 0; p < B.rows; ++p) {
        const int i = r[p], b = blk[(size_t)i];
        wl = std::max(wl, nlow(i));
        wu = std::max(wu, nup(i));
        for (int e = row[i]; e < row[i + 1]; ++e) {
          const int j = col[e], bj = blk[(size_t)j];
          if (bj != b) {
            if ((j < i) != (colour[(size_t)bj] < colour[(size_t)b]) ||
                colour[(size_t)bj] == colour[(size_t)b])
              return;
          } else if (j < i) {
            lev[(size_t)i] = std::max(lev[(size_t)i], lev[(size_t)j] + 1);
          }
        }
      }
      if (wl > kBrickWide || wu > kBrickWide) return;
      // a block's upper couplings must climb in level (they do where the pattern is
      // structurally symmetric)
      for (int p = 0; p < B.rows; ++p)
        for (int e = dia[r[p]] + 1; e < row[r[p] + 1]; ++e)
          if (blk[(size_t)col[e]] == blk[(size_t)r[p]] &&
              lev[(size_t)col[e]] <= lev[(size_t)r[p]])
            return;
      auto more = [&](int i) { return (wl > wu ? nlow(i) : nup(i)) > 3; };
      // by level, rows with second records first, then S position
      keys.clear();
      for (int p = 0; p < B.rows; ++p)
        keys.push_back({(uint64_t)lev[(size_t)r[p]] << 33 | (uint64_t)!more(r[p]) << 32 |
                            (uint32_t)s_of[(size_t)r[p]],
                        r[p]});
      std::sort(keys.begin(), keys.end());
      for (int p = 0; p < B.rows; ++p) r[p] = keys[(size_t)p].second;
      start.clear();
      for (int p = 0; p < B.rows; ++p) {
        if (p == 0 || lev[(size_t)r[p]] != lev[(size_t)r[p - 1]] || p - start.back() == kBrickLanes)
          start.push_back(p);
        step_of[(size_t)r[p]] = (int)start.size() - 1;
      }
      B.steps = (int)start.size();
      start.push_back(B.rows);
      P.steps = std::max(P.steps, B.steps);
      for (int t = 0; t < 2; ++t) {
        BrickTriangle &T = t == 0 ? out.L : out.U;
        Joined &J = P.of[t];
        const int stamp = 2 * k + t;
        auto when = [&](int x) {  // sweep order of a row's step
          return t == 0 ? step_of[(size_t)x] : B.steps - 1 - step_of[(size_t)x];
        };
        auto entries = [&](int x, auto &&f) {
          const int e0 = t == 0 ? row[x] : dia[x] + 1, w = t == 0 ? nlow(x) : nup(x);
          for (int j = 0; j < w; ++j) f(j, e0 + j, col[e0 + j]);
        };
        // the last step that reads each value of the unit and its halo
        halo.clear();
        hlast.clear();
        last.assign((size_t)B.rows, -1);
        for (int p = 0; p < B.rows; ++p) slot[(size_t)r[p]] = p;  // (for now its row in the unit)
        for (int p = 0; p < B.rows; ++p)
          entries(r[p], [&](int, int, int y) {
            if (blk[(size_t)y] == blk[(size_t)r[p]]) {
              int &l = last[(size_t)slot[(size_t)y]];
              l = std::max(l, when(r[p]));
            } else if (halo.size() <= kHaloMost) {
              Entry &E = halo_at(stamp, y);
              if (E.when != stamp) {
                E = {stamp, y, (int)halo.size()};
                halo.push_back(y);
                hlast.push_back(0);
              }
              int &l = hlast[(size_t)E.h];
              l = std::max(l, when(r[p]));
            }
          });
        if (halo.size() > kHaloMost) return;
        // slots in sweep order
        if ((int)dies.size() < B.steps) dies.resize((size_t)B.steps);
        for (int q = 0; q < B.steps; ++q) dies[(size_t)q].clear();
        int slots = 1 + (int)halo.size();
        for (size_t h = 0; h < halo.size(); ++h) dies[(size_t)hlast[h]].push_back(1 + (int)h);
        unused.clear();
        const size_t step0 = J.step.size();
        J.step.resize(step0 + (size_t)B.steps);
        for (int q = 0; q < B.steps; ++q) {
          const int at_step = t == 0 ? q : B.steps - 1 - q;
          const int c = start[(size_t)at_step], m = start[(size_t)at_step + 1] - c;
          if (q > 0)
            for (int s : dies[(size_t)q - 1]) unused.push_back(s);
          for (int i = 0; i < m; ++i) {
            const int x = r[c + i];
            const int l = last[(size_t)(c + i)];
            int s;
            if (!unused.empty()) {
              s = unused.back();
              unused.pop_back();
            } else {
              s = slots++;
            }
            dies[(size_t)std::max(l, q)].push_back(s);
            slot[(size_t)x] = s;
            if (s > 0x3fff) return;  // 16-bit byte offsets
          }
          int more_rows = 0;
          for (int i = 0; i < m; ++i)
            if ((t == 0 ? nlow(r[c + i]) : nup(r[c + i])) > 3) more_rows = i + 1;
          J.step[step0 + (size_t)at_step] = {(int)J.more_idx.size(),
                                             (unsigned)(c | m << 12 | more_rows << 20)};
          for (int i = 0; i < m; ++i) {
            const int x = r[c + i];
            BrickPlaces at[2] = {{{0, 0, 0, 0}}, {{0, 0, 0, 0}}};
            BrickSource from[2] = {{{-1, -1, -1, x}}, {{-1, -1, -1, -1}}};
            entries(x, [&](int j, int e, int y) {
              const int s = blk[(size_t)y] == blk[(size_t)x] ? slot[(size_t)y]
                                                             : 1 + halo_at(stamp, y).h;
              at[j / 3].at[j % 3] = (unsigned short)(s * sizeof(float));
              from[j / 3].e[j % 3] = e;
            });
            at[0].at[3] = (unsigned short)(slot[(size_t)x] * sizeof(float));
            T.idx[(size_t)(B.row0 + c + i)] = at[0];
            T.src[(size_t)(B.row0 + c + i)] = from[0];
            if (i < more_rows) {
              J.more_idx.push_back(at[1]);
              J.more_src.push_back(from[1]);
            }
          }
        }
        (t == 0 ? B.lh0 : B.uh0) = (int)J.halo.size();
        (t == 0 ? B.lh : B.uh) = (int)halo.size();
        for (int y : halo) J.halo.push_back(s_of[(size_t)y]);
        J.slots = std::max(J.slots, slots);
      }
    }
    P.ok = true;
  });
  for (const Part &P : part)
    if (!P.ok) return;
  for (int t = 0; t < 2; ++t) {
    BrickTriangle &T = t == 0 ? out.L : out.U;
    for (const Part &P : part) {
      const Joined &J = P.of[t];
      const int more0 = (int)T.idx.size();   // the first records are all there
      for (int k = P.first; k < P.last; ++k) {
        BrickUnit &B = out.unit[(size_t)k];
        if (t == 0) B.step0 += (int)T.step.size();
        (t == 0 ? B.lh0 : B.uh0) += (int)T.halo.size();
      }
      for (BrickStep K : J.step) {
        K.x0 += more0;
        T.step.push_back(K);
      }
      T.halo.insert(T.halo.end(), J.halo.begin(), J.halo.end());
      T.idx.insert(T.idx.end(), J.more_idx.begin(), J.more_idx.end());
      T.src.insert(T.src.end(), J.more_src.begin(), J.more_src.end());
      out.slots[t] = std::max(out.slots[t], J.slots);
      out.steps = std::max(out.steps, P.steps);
    }
    // one spare record: a step without second ones reads the record at its x0
    T.idx.push_back(BrickPlaces{{0, 0, 0, 0}});
    T.src.push_back(BrickSource{{-1, -1, -1, -1}});
  }
  out.pos.resize((size_t)n);
  for (int p = 0; p < n; ++p) out.pos[(size_t)p] = s_of[(size_t)out.row[(size_t)p]];
  out.ok = true;
}

void short_columns(const std::vector<long long> &off, const std::vector<int> &col,
                   ShortColumns &out) {
  out = ShortColumns();
  const size_t ns = off.size() - 1;
  out.window.assign(ns * kWindows, 0);
  out.off.assign(ns + 1, 0);
  for (size_t s = 0; s < ns; ++s) {
    const long long w = (off[s + 1] - off[s]) / 64;
    out.off[s + 1] = out.off[s] + 64 * ((w + 1) / 2);
  }
  out.code.assign((size_t)out.off[ns], 0);
  std::atomic<bool> fits{true};
  in_parts((int)ns, 1 << 9, [&](int, int s0, int s1) {
    for (int s = s0; s < s1 && fits; ++s) {
      const int *const c = col.data() + off[(size_t)s];
      const int slots = (int)(off[(size_t)s + 1] - off[(size_t)s]);
      // each window starts at the smallest column that none before it holds
      int *const first = &out.window[(size_t)s * kWindows];
      int nw = 0;
      for (long long bound = 0;;) {
        int next = INT_MAX;
        for (int i = 0; i < slots; ++i) next = c[i] >= bound && c[i] < next ? c[i] : next;
        if (next == INT_MAX) break;
        if (nw == kWindows) {
          fits = false;
          return;
        }
        first[nw++] = next;
        bound = (long long)next + kWindow;
      }
      unsigned *const code = out.code.data() + out.off[(size_t)s];
      for (int i = 0; i < slots; ++i) {
        int k = 0;
        while (k + 1 < nw && first[k + 1] <= c[i]) ++k;
        const int slot = i / 64, lane = i % 64;
        code[64 * (slot / 2) + lane] |= ((unsigned)k << 12 | (unsigned)(c[i] - first[k]))
                                        << (slot % 2 ? 16 : 0);
      }
    }
  });
  out.ok = fits;
}

double gather_lines(int n, const int *row, const int *col) {
  const int ngroup = (n + 63) / 64, step = std::max(1, ngroup / 256);
  long long lines = 0;
  int taken = 0;
  std::vector<int> last((size_t)n / 16 + 1, -1);   // the last group that touched each line
  for (int g = 0; g < ngroup; g += step, ++taken)
    for (int e = row[64 * g]; e < row[std::min(n, 64 * g + 64)]; ++e) {
      int &l = last[(size_t)(col[e] / 16)];
      lines += l != g;
      l = g;
    }
  return taken ? (double)lines / taken : 0.0;
}

void build_layout(int n, const int *row, const int *col, const int *dia, int spmv_rows,
                  int spmv_cap, int small_level, Layout &out, bool identity_s, BlockLayout *blocks) {
  out.n = n;
  out.nnz = n > 0 ? row[n] : 0;
  if (identity_s) {
    out.s_orig.resize(n);
    for (int i = 0; i < n; ++i) out.s_orig[i] = i;
  } else {
    out.s_orig = rcm(n, row, col);
  }
  out.s_of_orig.assign(n, 0);
  for (int k = 0; k < n; ++k) out.s_of_orig[out.s_orig[k]] = k;
  // the S copy, beside the sweeps' orders
  std::future<void> s_copy = std::async(beside(n), [&] {
    out.s_row.assign(n + 1, 0);
    for (int k = 0; k < n; ++k) {
      const int i = out.s_orig[k];
      out.s_row[k + 1] = out.s_row[k] + row[i + 1] - row[i];
    }
    out.s_col.assign(out.nnz, 0);
    out.s_src.assign(out.nnz, 0);
    out.s_diag_src.assign(n, 0);
    int bw = 0;
    for (int k = 0; k < n; ++k) {
      const int i = out.s_orig[k];
      int e = out.s_row[k];
      for (int j = row[i]; j < row[i + 1]; ++j, ++e) {
        out.s_col[e] = out.s_of_orig[col[j]];
        out.s_src[e] = j;
        bw = std::max(bw, std::abs(out.s_col[e] - k));
      }
      out.s_diag_src[k] = dia[i];
    }
    out.bandwidth = bw;
    // SpMV row blocks: <= spmv_rows rows and <= spmv_cap entries each
    out.s_rblk.assign(1, 0);
    for (int r = 0; r < n;) {
      int e = r + 1;
      while (e < n && e - r < spmv_rows && out.s_row[e + 1] - out.s_row[r] <= spmv_cap) ++e;
      out.s_rblk.push_back(e);
      r = e;
    }
  });
  build_sweep(n, row, col, dia, true, out.s_of_orig, small_level, out.L);
  std::future<void> block_sweeps;
  if (blocks)
    block_sweeps = std::async(beside(n), [&] {
      build_blocks(n, row, col, dia, out.s_of_orig, out.L.nlev, *blocks);
    });
  build_sweep(n, row, col, dia, false, out.s_of_orig, small_level, out.U,
              kMirrorUpper ? &out.L : nullptr);
  out.l_to_s.assign(n, 0);
  out.u_to_l.assign(n, 0);
  out.s_to_u.assign(n, 0);
  for (int p = 0; p < n; ++p) out.l_to_s[p] = out.s_of_orig[out.L.orig[p]];
  for (int q = 0; q < n; ++q) out.u_to_l[q] = out.L.of_orig[out.U.orig[q]];
  for (int k = 0; k < n; ++k) out.s_to_u[k] = out.U.of_orig[out.s_orig[k]];
  s_copy.get();
  if (blocks) block_sweeps.get();
}

namespace {

// 128-byte lines of a cell field and of a face field that the slices of an
// order touch, summed over up to 256 slices spread over the mesh.  Lists and
// pairs are by position in the order of first naming: that order's lines or, with
// `orig` and `of`, the caller's.
long long lines_touched(int n, const std::vector<int> &pair, const std::vector<int> &ptr,
                        const std::vector<unsigned> &inc, const std::vector<int> *orig,
                        const std::vector<int> *of) {
  const int nslice = (n + 63) / 64, step = std::max(1, nslice / 256);
  long long lines = 0;
  // the last slice that touched each line of the cell and of the face field
  std::vector<int> cell_line((size_t)n / 16 + 1, -1), face_line(pair.size() / 32 + 1, -1);
  for (int s = 0; s < nslice; s += step) {
    auto touch = [&](int &line) {
      lines += line != s;
      line = s;
    };
    for (int k = 64 * s; k < std::min(n, 64 * s + 64); ++k) {
      const int p = of ? (*of)[(size_t)k] : k;
      touch(cell_line[(size_t)(k / 16)]);
      for (int e = ptr[(size_t)p]; e < ptr[(size_t)p + 1]; ++e) {
        const long long f = inc[(size_t)e] >> 1;
        const int o = pair[(size_t)(2 * f + ((inc[(size_t)e] & 1) ? 0 : 1))];
        touch(face_line[(size_t)(f / 16)]);
        if (o >= 0) touch(cell_line[(size_t)((orig ? (*orig)[(size_t)o] : o) / 16)]);
      }
    }
  }
  return lines;
}

}  // namespace

void build_face_lists(int n, long long nf, const int *faces, int base, int from, FaceLists &out) {
  out = FaceLists();
  out.n = n;
  // Both cells of each face (boundary: -1), from `from` cells on by position in the
  // order of first naming (cells of no face last): whatever is done per cell below
  // then goes through memory in runs, the one random access a face's cell being its
  // position.
  const bool named = n >= from;
  std::vector<int> orig, of, pair((size_t)(2 * nf));
  if (named) {
    of.assign((size_t)n, -1);
    orig.reserve((size_t)n);
  }
  auto name = [&](int c) {
    if (c < 0) return -1;
    if (!named) return c;
    int &p = of[(size_t)c];
    if (p < 0) {
      p = (int)orig.size();
      orig.push_back(c);
    }
    return p;
  };
  for (long long k = 0; k < 2 * nf; ++k) pair[(size_t)k] = name(faces[k] - base);
  for (int c = 0; c < n && named; ++c) name(c);
  // per cell, its faces in ascending order (a counting sort over the faces)
  std::vector<int> ptr((size_t)n + 1, 0);
  for (const int p : pair)
    if (p >= 0) ptr[(size_t)p + 1]++;
  for (int c = 0; c < n; ++c) ptr[(size_t)c + 1] += ptr[(size_t)c];
  std::vector<unsigned> inc((size_t)ptr[(size_t)n]);
  {
    std::vector<int> fill(ptr.begin(), ptr.end() - 1);
    for (long long k = 0; k < 2 * nf; ++k)
      if (pair[(size_t)k] >= 0) inc[(size_t)fill[(size_t)pair[(size_t)k]]++] = (unsigned)k;
  }
  if (named && lines_touched(n, pair, ptr, inc, &orig, &of) >
                   2 * lines_touched(n, pair, ptr, inc, nullptr, nullptr)) {
    out.reordered = true;
    out.orig = std::move(orig);
    out.of = std::move(of);
  }
  const int nslice = (n + 63) / 64;
  out.off.assign((size_t)nslice + 1, 0);
  bool tails = false;
  auto cell = [&](int k) { return named && !out.reordered ? of[(size_t)k] : k; };   // in ptr
  auto width = [&](int c) { return ptr[(size_t)c + 1] - ptr[(size_t)c]; };
  for (int s = 0; s < nslice; ++s) {
    int w = 0;
    for (int k = 64 * s; k < std::min(n, 64 * s + 64); ++k) w = std::max(w, width(cell(k)));
    tails = tails || w > kFaceSlots;
    out.off[(size_t)s + 1] = out.off[(size_t)s] + 64LL * std::min(w, kFaceSlots);
  }
  out.inc.assign((size_t)out.off[(size_t)nslice], kNoFace);
  if (tails) out.tptr.assign((size_t)n + 1, 0);
  for (int k = 0; k < n; ++k) {
    const int c = cell(k), w = width(c);
    for (int j = 0; j < std::min(w, kFaceSlots); ++j)
      out.inc[(size_t)(out.off[(size_t)(k / 64)] + 64LL * j + k % 64)] =
          inc[(size_t)(ptr[(size_t)c] + j)];
    for (int j = kFaceSlots; j < w; ++j) out.tail.push_back(inc[(size_t)(ptr[(size_t)c] + j)]);
    if (tails) out.tptr[(size_t)k + 1] = (int)out.tail.size();
  }
}

}  // namespace tfs
