// tfs_assembly.hip -- device-side assembly of A % val from face coefficients.
//
// T-FlowS forms its pressure and momentum matrices in a loop over faces that
// scatters through the topology's pos/dia arrays
// (Sources/Process/Pressure_Matrix_Fractional.f90:19-48,
//  Sources/Process/NewUVW.f90:349-384 for the faces, :500-506 for the
//  inertia term, :586-590 for under-relaxation; pos/dia from
//  Sources/Process/Matrix_Mod/Topology.f90:105-121):
//
//   val := 0
//   do s = 1, n_faces
//     if (c2 > 0) then  val(pos(1,s)) -= a12;  val(dia(c1)) += a12
//                       val(pos(2,s)) -= a21;  val(dia(c2)) += a21
//     else (boundary kinds that contribute)    val(dia(c1)) += a12
//   do c: val(dia(c)) += cell(c);  sav(c) = val(dia(c));  val(dia(c)) /= urf
//
// Every off-diagonal entry belongs to one face and side, so it is 0 - a12
// whatever the order.  A diagonal receives one addition per incident face, in
// face order; here each cell sums its own faces in ascending order (the face
// lists of tfs_layout.hpp), so the result is bitwise that of the sequential
// loop, with one lane per cell and no atomics.  The same pass writes the cell's
// off-diagonals: its entries are one row, so the stores of a lane meet in the
// caches, where a pass over faces scatters two values each.  The values then go
// through the solver's usual change path (layouts regathered, factor rebuilt on
// the next solve).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "tfs_faces.hpp"
#include "tfs_internal.hpp"
#include "tfs_solver.h"

using namespace tfs;

namespace {

constexpr int kThreads = 256;

#define TFS_A_HIP(expr)                        \
  do {                                         \
    if ((expr) != hipSuccess) {                \
      (void)hipGetLastError();                 \
      return TFS_ERR_DEVICE;                   \
    }                                          \
  } while (0)

// pos: per list entry, where the face's entry of this cell's side goes in `out`
// (kBoundary: the face is a boundary face; kDropped: the entry is a diagonal,
// which its cell writes), dia: where the diagonals go.  The reference's
// val(pos) = val(pos) - a on cleared values is 0 - a (which keeps the sign of a
// zero coefficient as it does).
// `out` is val itself where the lists keep the caller's cells.  Where they do
// not, a cell's row would be 56 bytes somewhere in val, less than a memory line
// and not aligned: the rows then go one after another into a buffer, which
// k_place brings into the caller's order, reading parts of lines and writing
// whole ones.  128^3 numbered at random: 577 us for passes over faces and cells
// in the caller's orders, 308 us with rows written in place, 198 us with both
// kernels here.
constexpr int kBoundary = -1, kDropped = -2;

__global__ void __launch_bounds__(kThreads)
k_assemble(FaceSlots L, const int *__restrict__ pos, const double *__restrict__ a12,
           const double *__restrict__ a21, const unsigned char *__restrict__ bnd_on,
           const double *__restrict__ cell, double urf, const int *__restrict__ dia,
           double *__restrict__ out, double *__restrict__ sav) {
  const int lanes = (L.n + 63) / 64 * 64;
  for (int k = blockIdx.x * kThreads + threadIdx.x; k < lanes; k += gridDim.x * kThreads) {
    struct Term { double a; int q; };
    double d = 0.0;
    each_face<Term>(
        L, k,
        [&](long long i, unsigned e) {
          const long long s = e >> 1;
          return Term{(e & 1u) && a21 ? a21[s] : a12[s], pos[i]};
        },
        [&](unsigned e, const Term &t) {
          if (t.q != kBoundary || !bnd_on || bnd_on[e >> 1]) d = d + t.a;
          if (t.q >= 0) out[t.q] = 0.0 - t.a;
        });
    if (k >= L.n) continue;
    const int c = L.cell(k);
    if (cell) d = d + cell[c];
    if (sav) sav[c] = d;
    if (urf != 1.0) d = d / urf;
    out[dia[k]] = d;
  }
}

// val from the rows in the lists' order; src < 0: an entry nothing writes.
__global__ void __launch_bounds__(kThreads)
k_place(long long m, const int *__restrict__ src, const double *__restrict__ rows,
        double *__restrict__ val) {
  for (long long i = blockIdx.x * (long long)kThreads + threadIdx.x; i < m;
       i += (long long)gridDim.x * kThreads)
    val[i] = src[i] >= 0 ? rows[src[i]] : 0.0;
}

__global__ void __launch_bounds__(kThreads) k_zero(long long m, double *__restrict__ v) {
  for (long long i = blockIdx.x * (long long)kThreads + threadIdx.x; i < m;
       i += (long long)gridDim.x * kThreads)
    v[i] = 0.0;
}

int grid_of(long long m) { return (int)std::max(1LL, std::min(4096LL, (m + kThreads - 1) / kThreads)); }

}  // namespace

struct tfs_assembly {
  tfs_matrix *A = nullptr;
  long long nf = 0, nnz = 0;
  DevFaceLists lists;
  int *pos = nullptr, *dia = nullptr;
  bool clear = false;   // val has entries that no face and no diagonal writes
  double *rows = nullptr;   // reordered cells: the rows in the lists' order
  int *src = nullptr;       // and each entry's place there
};

extern "C" int tfs_assembly_destroy(tfs_assembly *S) {
  if (!S) return TFS_OK;
  for (void *p : {(void *)S->pos, (void *)S->dia, (void *)S->rows, (void *)S->src})
    if (p) (void)hipFree(p);
  S->lists.release();
  delete S;
  return TFS_OK;
}

extern "C" int tfs_assembly_create(tfs_matrix *A, long long n_faces, const int *faces_c,
                                   const int *pos, const int *dia, int base, tfs_assembly **out) {
  if (!out) return TFS_ERR_INVALID;
  *out = nullptr;
  tfs_matrix_info info;
  if (!A || tfs_matrix_get_info(A, &info) != TFS_OK || n_faces < 0 ||
      (n_faces > 0 && (!faces_c || !pos)) || (info.n > 0 && !dia) || (base != 0 && base != 1))
    return TFS_ERR_INVALID;
  const int n = info.n;
  const long long nf = n_faces, nnz = info.nnz;
  std::vector<int> hdia((size_t)n);
  std::vector<bool> diagonal((size_t)nnz);   // bits: they are looked up in any order
  for (int c = 0; c < n; ++c) {
    hdia[(size_t)c] = dia[c] - base;
    if (hdia[(size_t)c] < 0 || hdia[(size_t)c] >= nnz) return TFS_ERR_INVALID;
    diagonal[(size_t)hdia[(size_t)c]] = true;
  }
  for (long long s = 0; s < nf; ++s) {
    const int c1 = faces_c[2 * s] - base, c2 = faces_c[2 * s + 1] - base;
    if (c1 < 0 || c1 >= n || c2 >= n || c2 == c1) return TFS_ERR_INVALID;
    for (int k = 0; k < 2 && c2 >= 0; ++k) {
      const long long q = (long long)pos[2 * s + k] - base;
      if (q < 0 || q >= nnz) return TFS_ERR_INVALID;
    }
  }
  FaceLists F;
  build_face_lists(n, nf, faces_c, base, kReorderAssembly, F);
  // where each entry goes, slice by slice, and how many of a slice go anywhere
  const int nslice = (n + 63) / 64;
  std::vector<int> hpos(F.inc.size() + F.tail.size(), kBoundary), first((size_t)nslice + 1, 0);
  auto place = [&](unsigned e) {
    const long long s = e >> 1;
    if (faces_c[2 * s + 1] < base) return kBoundary;
    const int q = pos[2 * s + (e & 1)] - base;
    return diagonal[(size_t)q] ? kDropped : q;
  };
  // the tail entries of a slice's cells
  auto tails = [&](int s, int k) {
    return F.tptr.empty() ? 0 : F.tptr[(size_t)std::min(n, 64 * s + k)];
  };
  in_parts(nslice, 1 << 12, [&](int, int s0, int s1) {
    for (int s = s0; s < s1; ++s) {
      int go = std::min(n, 64 * s + 64) - 64 * s;   // the diagonals
      for (size_t i = (size_t)F.off[(size_t)s]; i < (size_t)F.off[(size_t)s + 1]; ++i)
        if (F.inc[i] != kNoFace) go += (hpos[i] = place(F.inc[i])) >= 0;
      for (int t = tails(s, 0); t < tails(s, 64); ++t)
        go += (hpos[F.inc.size() + (size_t)t] = place(F.tail[(size_t)t])) >= 0;
      first[(size_t)s + 1] = go;
    }
  });
  // rows in the lists' order, each one's entries as they stand in val
  std::vector<int> src, to_dia((size_t)n);
  for (int s = 0; s < nslice; ++s) first[(size_t)s + 1] += first[(size_t)s];
  const int nrows = first[(size_t)nslice];
  bool clear = false;   // entries that nothing writes (k_place sets them itself)
  if (F.reordered) {
    src.assign((size_t)nnz, -1);
    in_parts(nslice, 1 << 12, [&](int, int s0, int s1) {
      std::vector<int *> mine;   // where this row's places are, by place
      auto add = [&](int *q) {
        mine.push_back(q);
        for (size_t j = mine.size() - 1; j > 0 && *mine[j - 1] > *mine[j]; --j)
          std::swap(mine[j - 1], mine[j]);
      };
      for (int k = 64 * s0, at = first[(size_t)s0]; k < std::min(n, 64 * s1); ++k) {
        const long long i0 = F.off[(size_t)(k / 64)] + k % 64, i1 = F.off[(size_t)(k / 64) + 1];
        mine.clear();
        for (long long i = i0; i < i1; i += 64)
          if (hpos[(size_t)i] >= 0) add(&hpos[(size_t)i]);
        if (!F.tptr.empty()) {
          for (int t = F.tptr[(size_t)k]; t < F.tptr[(size_t)k + 1]; ++t)
            if (hpos[F.inc.size() + (size_t)t] >= 0) mine.push_back(&hpos[F.inc.size() + (size_t)t]);
          std::stable_sort(mine.begin(), mine.end(), [](int *a, int *b) { return *a < *b; });
        }
        to_dia[(size_t)k] = hdia[(size_t)F.orig[(size_t)k]];
        add(&to_dia[(size_t)k]);
        for (int *q : mine) {
          src[(size_t)*q] = at;
          *q = at++;
        }
      }
    });
  } else {
    to_dia = hdia;
    std::vector<unsigned char> written((size_t)nnz, 0);
    for (const int q : hdia) written[(size_t)q] = 1;
    for (const int q : hpos)
      if (q >= 0) written[(size_t)q] = 1;
    clear = std::count(written.begin(), written.end(), (unsigned char)0) > 0;
  }
  auto *S = new tfs_assembly;
  S->A = A;
  S->nf = nf;
  S->nnz = nnz;
  S->clear = clear;
  auto up = [](void **dst, const void *src, size_t bytes) -> bool {
    if (hipMalloc(dst, std::max<size_t>(bytes, 8)) != hipSuccess) return false;
    return bytes == 0 || hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice) == hipSuccess;
  };
  if (!S->lists.upload(F) ||
      !up((void **)&S->pos, hpos.data(), sizeof(int) * hpos.size()) ||
      !up((void **)&S->dia, to_dia.data(), sizeof(int) * to_dia.size()) ||
      (F.reordered && (!up((void **)&S->src, src.data(), sizeof(int) * src.size()) ||
                       hipMalloc((void **)&S->rows, sizeof(double) * (size_t)nrows) !=
                           hipSuccess))) {
    (void)hipGetLastError();
    tfs_assembly_destroy(S);
    return TFS_ERR_NOMEM;
  }
  *out = S;
  return TFS_OK;
}

extern "C" int tfs_assemble_device(tfs_assembly *S, const double *d_a12, const double *d_a21,
                                   const unsigned char *d_bnd_on, const double *d_cell, double urf,
                                   double *d_sav) {
  if (!S || (S->nf > 0 && !d_a12) || !(urf > 0.0)) return TFS_ERR_INVALID;
  double *val = tfs_matrix_values_device(S->A);
  hipStream_t st = tfs::matrix_stream(S->A);
  if (S->clear)
    hipLaunchKernelGGL(k_zero, dim3(grid_of(S->nnz)), dim3(kThreads), 0, st, S->nnz, val);
  if (S->lists.at.n > 0)
    hipLaunchKernelGGL(k_assemble, dim3(grid_of(S->lists.lanes())), dim3(kThreads), 0, st,
                       S->lists.at, S->pos, d_a12, d_a21, d_bnd_on, d_cell, urf, S->dia,
                       S->rows ? S->rows : val, d_sav);
  if (S->rows)
    hipLaunchKernelGGL(k_place, dim3(grid_of(S->nnz)), dim3(kThreads), 0, st, S->nnz, S->src,
                       S->rows, val);
  TFS_A_HIP(hipGetLastError());
  TFS_A_HIP(hipStreamSynchronize(st));
  return tfs_matrix_values_changed(S->A);
}
