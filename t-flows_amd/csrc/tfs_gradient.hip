// tfs_gradient.hip -- least-squares cell gradients on the device.
//
// T-FlowS computes cell gradients by least squares over the face neighbours:
//   Compute_Gradient_Matrix  Sources/Process/Compute_Gradient_Matrix.f90:21-116
//     G(c) = inverse of sum over the faces of c of d d^T (d the centre-to-centre
//     vector of the face after Compute_Geometry), by cofactors over Jac + TINY;
//   GraPhi                   Sources/Process/GraPhi.f90:25-173
//     grad phi(c) = G(c) sum over the faces of c of (phi(c2) - phi(c1)) d,
//     zero difference across a SYMMETRY boundary;
//   GradP                    Sources/Process/GradP.f90:24-64
//     boundary cells (not BUFFER / PRESSURE) take the inside value, gradient,
//     boundary values extrapolated along it with factor 1.2, gradient again.
// All with Boundary = .TRUE., as every call site passes it: both cells of an
// interior face and the inside cell of a boundary face take the face's term.
//
// The reference accumulates in one sequential loop over faces.  Here every
// cell sums its own faces in ascending face order (the face lists of
// tfs_layout.hpp), so each sum has the reference's order and the result is
// bitwise the same, one lane per cell and no atomics.  The three components of
// a gradient are formed in one pass (the reference makes three passes over the
// same data, one per component; each component's sum is unchanged).  What a
// list entry needs of the mesh -- the other cell and G d, three numbers -- is
// laid out beside it at creation, so a wavefront reads contiguous runs and
// gathers one phi per entry.
//
// Where the lists take the cells in another order than the caller's (a random
// numbering), fields go into that order in one pass and results come back in
// another, as records of one cell (one line each way): the gathers in between
// then stay in the caches.  On MI355X at 128^3 numbered at random, grad phi and
// grad p together took 1523 us with cells in the caller's order (every gather a
// line of its own) and take 447 us; the flux sum of the face loops 285 and 23.
//
// The same mesh object serves Correct_Velocity
// (Sources/Process/Correct_Velocity.f90:34-135): velocities corrected by the
// pressure gradient, PRESSURE boundary cells given the inside velocity, face
// fluxes corrected by the pressure-correction difference, the mass error per
// cell (each cell sums its faces' fluxes in face order, as the reference's
// loop does) and the maxima of |mass error|, CFL and Peclet numbers (maxima
// are exact in any order).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "tfs_device.hpp"
#include "tfs_faces.hpp"
#include "tfs_solver.h"

using namespace tfs;

namespace {

constexpr int kThreads = 256;
#define TFS_G_HIP(expr)                        \
  do {                                         \
    if ((expr) != hipSuccess) {                \
      (void)hipGetLastError();                 \
      return TFS_ERR_DEVICE;                   \
    }                                          \
  } while (0)

int grid_of(long long m) {
  long long g = (m + kThreads - 1) / kThreads;
  return (int)(g < 1 ? 1 : (g > 8192 ? 8192 : g));
}

// One lane per cell of the face lists, whole slices.
#define TFS_CELL_LOOP(k, L)                                                      \
  for (int k = blockIdx.x * kThreads + threadIdx.x, k##_end = ((L).n + 63) / 64 * 64; \
       k < k##_end; k += gridDim.x * kThreads)

// What entry i of a face list holds for the gradients: the other cell's
// position (n and up: a boundary slot of the caller's array; -1: across a
// SYMMETRY boundary, whose difference is zero) and G d, signed so that the term
// is (phi(other) - phi(cell)) w whichever side the cell is on.
struct GradEntries {
  int *other;
  double *w;   // three runs of `entries`
  long long entries;
};

// G(c): the normal matrix summed over the cell's faces in face order, then its
// inverse (Compute_Gradient_Matrix.f90:30-70, :96-116), and what the entries
// hold.  g holds six blocks of n: G(1..6, c) at g[k n + c], the caller's cells.
__global__ void __launch_bounds__(kThreads)
k_gmatrix(FaceSlots L, long long nf, const int2 *__restrict__ pairs,
          const unsigned char *__restrict__ kind, const double *__restrict__ d,
          double *__restrict__ g, GradEntries E) {
  const int n = L.n;
  TFS_CELL_LOOP(k, L) {
    double G0 = 0.0, G1 = 0.0, G2 = 0.0, G3 = 0.0, G4 = 0.0, G5 = 0.0;
    struct V3 { double x, y, z; };
    const auto face_d = [&](long long, unsigned e) {
      const long long s = e >> 1;
      return V3{d[s], d[nf + s], d[2 * nf + s]};
    };
    each_face<V3>(L, k, face_d, [&](unsigned, const V3 &v) {
      G0 = G0 + v.x * v.x;
      G1 = G1 + v.y * v.y;
      G2 = G2 + v.z * v.z;
      G3 = G3 + v.x * v.y;
      G4 = G4 + v.x * v.z;
      G5 = G5 + v.y * v.z;
    });
    const double jac = G0 * G1 * G2 - G0 * G5 * G5 - G3 * G3 * G2 + 2.0 * G3 * G4 * G5 -
                       G4 * G4 * G1;
    const double g0 = +(G1 * G2 - G5 * G5) / (jac + kTiny);
    const double g1 = +(G0 * G2 - G4 * G4) / (jac + kTiny);
    const double g2 = +(G0 * G1 - G3 * G3) / (jac + kTiny);
    const double g3 = -(G3 * G2 - G4 * G5) / (jac + kTiny);
    const double g4 = +(G3 * G5 - G4 * G1) / (jac + kTiny);
    const double g5 = -(G0 * G5 - G3 * G4) / (jac + kTiny);
    if (k < n) {
      const long long c = L.cell(k);
      g[c] = g0;
      g[n + c] = g1;
      g[2LL * n + c] = g2;
      g[3LL * n + c] = g3;
      g[4LL * n + c] = g4;
      g[5LL * n + c] = g5;
    }
    struct At { long long i; };
    each_face<At>(L, k, [&](long long i, unsigned) { return At{i}; }, [&](unsigned e, At at) {
      const V3 v = face_d(0, e);
      const int2 f = pairs[e >> 1];
      const double sign = (e & 1u) ? -1.0 : 1.0;
      int o = (e & 1u) ? f.x : f.y;
      if (o >= n && kind[o - n] == TFS_BC_SYMMETRY) o = -1;
      E.other[at.i] = o;
      E.w[at.i] = sign * (g0 * v.x + g3 * v.y + g4 * v.z);
      E.w[E.entries + at.i] = sign * (g3 * v.x + g1 * v.y + g5 * v.z);
      E.w[2 * E.entries + at.i] = sign * (g4 * v.x + g5 * v.y + g2 * v.z);
    });
  }
}

// One cell's values side by side: 32-byte records, so that a cell in another
// order is one access.
struct Rec4 { double x, y, z, pad; };

// GraPhi for i = 1, 2, 3 at once (GraPhi.f90:25-73, :75-123, :125-173 with
// Boundary = .TRUE.).  phi: the cells in the lists' order; phib: the caller's
// array, for the boundary slots.  The gradient goes to px, py, pz or, where the
// cells are reordered, to rec.
// Bound by memory: 28 bytes an entry, 32 to 40 a cell.
__global__ void __launch_bounds__(kThreads)
k_graphi(FaceSlots L, GradEntries E, const double *__restrict__ phi,
         const double *__restrict__ phib, double *__restrict__ px, double *__restrict__ py,
         double *__restrict__ pz, Rec4 *__restrict__ rec) {
  const int n = L.n;
  TFS_CELL_LOOP(k, L) {
    const double pc = k < n ? phi[k] : 0.0;
    double ax = 0.0, ay = 0.0, az = 0.0;
    struct Term { double po, x, y, z; int o; };
    each_face<Term>(
        L, k,
        [&](long long i, unsigned) {
          Term t;
          t.o = E.other[i];
          t.x = E.w[i];
          t.y = E.w[E.entries + i];
          t.z = E.w[2 * E.entries + i];
          t.po = t.o < 0 ? 0.0 : t.o < n ? phi[t.o] : phib[t.o];
          return t;
        },
        [&](unsigned, const Term &t) {
          const double dphi = t.o < 0 ? 0.0 : t.po - pc;
          ax = ax + dphi * t.x;
          ay = ay + dphi * t.y;
          az = az + dphi * t.z;
        });
    if (k < n) {
      if (rec) {
        rec[k] = Rec4{ax, ay, az, 0.0};
      } else {
        px[k] = ax;
        py[k] = ay;
        pz[k] = az;
      }
    }
  }
}

// A field into the lists' order.
__global__ void __launch_bounds__(kThreads)
k_into_order(int n, const int *__restrict__ orig, const double *__restrict__ in,
             double *__restrict__ out) {
  for (int k = blockIdx.x * kThreads + threadIdx.x; k < n; k += gridDim.x * kThreads)
    out[k] = in[orig[k]];
}

// Gradients from the lists' order into the caller's.
__global__ void __launch_bounds__(kThreads)
k_from_order(int n, const int *__restrict__ of, const Rec4 *__restrict__ rec,
             double *__restrict__ px, double *__restrict__ py, double *__restrict__ pz) {
  for (int c = blockIdx.x * kThreads + threadIdx.x; c < n; c += gridDim.x * kThreads) {
    const Rec4 r = rec[of[c]];
    px[c] = r.x;
    py[c] = r.y;
    pz[c] = r.z;
  }
}

// Whether GradP.f90:32-40 extrapolates to boundary cells of this kind.
__device__ __forceinline__ bool extrapolated(unsigned char kind) {
  return kind != TFS_BC_BUFFER && kind != TFS_BC_PRESSURE;
}

// GradP.f90:32-58 for the cells (positions `at`) with extrapolated boundary
// faces: their gradient with the boundary cells at the inside value, and the
// boundary cells extrapolated along it.  Only these cells' gradients are used
// of GradP's first pass, and a boundary cell is read by its inside cell alone,
// so one lane does both for its cell.
__global__ void __launch_bounds__(kThreads)
k_bnd_extrap(int m, const int *__restrict__ at, FaceSlots L, GradEntries E,
             const int2 *__restrict__ pairs, const unsigned char *__restrict__ kind,
             const double *__restrict__ xc, long long na, double *__restrict__ phi) {
  const int n = L.n;
  for (int q = blockIdx.x * kThreads + threadIdx.x; q < m; q += gridDim.x * kThreads) {
    const int k = at[q], c1 = L.cell(k);
    const double pc = phi[c1];
    double ax = 0.0, ay = 0.0, az = 0.0;
    const long long i0 = L.off[k / 64] + k % 64;
    const int wd = (int)((L.off[k / 64 + 1] - L.off[k / 64]) / 64);
    const long long t0 = L.off[(n + 63) / 64];
    const int ta = L.tptr ? L.tptr[k] : 0, tb = L.tptr ? L.tptr[k + 1] : 0;
    auto all = [&](auto &&visit) {
      for (int j = 0; j < wd; ++j) {
        const unsigned e = L.inc[i0 + 64LL * j];
        if (e != kNoFace) visit(e, i0 + 64LL * j);
      }
      for (int t = ta; t < tb; ++t) visit(L.tail[t], t0 + t);
    };
    all([&](unsigned e, long long i) {
      const int o = E.other[i];
      double dphi = 0.0;
      if (o >= 0)
        dphi = (o < n ? phi[L.cell(o)] : extrapolated(kind[o - n]) ? pc : phi[o]) - pc;
      ax = ax + dphi * E.w[i];
      ay = ay + dphi * E.w[E.entries + i];
      az = az + dphi * E.w[2 * E.entries + i];
    });
    all([&](unsigned e, long long) {
      const int c2 = pairs[e >> 1].y;
      if ((e & 1u) == 0 && c2 >= n && extrapolated(kind[c2 - n]))
        phi[c2] = pc + 1.2 * (ax * (xc[c2] - xc[c1]) + ay * (xc[na + c2] - xc[na + c1]) +
                              az * (xc[2 * na + c2] - xc[2 * na + c1]));
    });
  }
}

// ---- Correct_Velocity -------------------------------------------------------

constexpr int kParts = 8192;   // the largest grid of grid_of(): one partial per block

// max over the workgroup of v, written by thread 0 to part[blockIdx.x]
__device__ void block_max(double v, double *__restrict__ part) {
  __shared__ double wmax[kThreads / 64];
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double m = wmax[0];
    for (int w = 1; w < kThreads / 64; ++w) m = fmax(m, wmax[w]);
    part[blockIdx.x] = m;
  }
  __syncthreads();
}

// Correct_Velocity.f90:34-46
__global__ void __launch_bounds__(kThreads)
k_cv_cells(int n, const double *__restrict__ vol, const double *__restrict__ sav,
           const double *__restrict__ px, const double *__restrict__ py,
           const double *__restrict__ pz, double *__restrict__ u, double *__restrict__ v,
           double *__restrict__ w) {
  for (int c = blockIdx.x * kThreads + threadIdx.x; c < n; c += gridDim.x * kThreads) {
    const double vc = vol[c], sc = sav[c];
    u[c] = u[c] - px[c] * vc / sc;
    v[c] = v[c] - py[c] * vc / sc;
    w[c] = w[c] - pz[c] * vc / sc;
  }
}

// Correct_Velocity.f90:48-59 (PRESSURE boundaries), :72-82 (flux correction),
// :117-135 (CFL and Peclet numbers of the corrected fluxes); per-block maxima
// to part_cfl / part_pe.  pp: the cells in the lists' order; ppb: the caller's
// array, for the boundary slots.
__global__ void __launch_bounds__(kThreads)
k_cv_faces(int n, long long nf, const int2 *__restrict__ pairs, const int *__restrict__ orig,
           const unsigned char *__restrict__ kind, const double *__restrict__ pp,
           const double *__restrict__ ppb, const double *__restrict__ coef,
           const double *__restrict__ bou, const unsigned char *__restrict__ in_m,
           const double *__restrict__ scoef, const double *__restrict__ d, double dt,
           double visc, double *__restrict__ flux, double *__restrict__ u,
           double *__restrict__ v, double *__restrict__ w, double *__restrict__ part_cfl,
           double *__restrict__ part_pe) {
  double cm = 0.0, pm = 0.0;
  for (long long s = blockIdx.x * (long long)kThreads + threadIdx.x; s < nf;
       s += (long long)gridDim.x * kThreads) {
    const int2 f = pairs[s];
    const bool inner = f.y < n;
    const int kd = inner ? TFS_BC_WALL : kind[f.y - n];
    if (!inner && kd == TFS_BC_PRESSURE) {
      const int c1 = orig ? orig[f.x] : f.x;
      u[f.y] = u[c1];
      v[f.y] = v[c1];
      w[f.y] = w[c1];
    }
    if (inner || kd == TFS_BC_BUFFER) {
      const double p2 = inner ? pp[f.y] : ppb[f.y];
      const double a = inner ? coef[s] : (bou ? bou[f.y - n] : 0.0);
      const double fl = flux[s] + (p2 - pp[f.x]) * a;
      flux[s] = fl;
      if (!in_m || in_m[s]) {
        const double x = d[s], y = d[nf + s], z = d[2 * nf + s];
        cm = fmax(cm, fabs(dt * fl / (scoef[s] * (x * x + y * y + z * z))));
        pm = fmax(pm, fabs(fl / scoef[s] / (visc + kTiny)));
      }
    }
  }
  block_max(cm, part_cfl);
  block_max(pm, part_pe);
}

// Per cell, in face order, inflow - outflow (Correct_Velocity.f90:88-100,
// Compute_Pressure_Fractional.f90:112-113, :126); `out` in the lists' order.
// Bound by memory: 4 bytes of list and the flux an entry, each flux line read
// once where the lists' order is the faces'.
__global__ void __launch_bounds__(kThreads)
k_flux_sum(FaceSlots L, const double *__restrict__ flux, double *__restrict__ out) {
  TFS_CELL_LOOP(k, L) {
    double m = 0.0;
    each_face<double>(
        L, k, [&](long long, unsigned e) { return flux[e >> 1]; },
        [&](unsigned e, double fl) { m = (e & 1u) ? m + fl : m - fl; });
    if (k < L.n) out[k] = m;
  }
}

// Correct_Velocity.f90:102-111: b(c) over vol * density, from the sums (in the
// lists' order, `of` null: the caller's, b itself); per-block maxima of |b|.
__global__ void __launch_bounds__(kThreads)
k_cv_mass(int n, const int *__restrict__ of, const double *sum, const double *__restrict__ vol,
          const double *__restrict__ den, double *b, double *__restrict__ part_err) {
  double em = 0.0;
  for (int c = blockIdx.x * kThreads + threadIdx.x; c < n; c += gridDim.x * kThreads) {
    const double m = sum[of ? of[c] : c] / (vol[c] * den[c]);
    b[c] = m;
    em = fmax(em, fabs(m));
  }
  block_max(em, part_err);
}

// the three maxima over the per-block partials
__global__ void __launch_bounds__(kThreads)
k_cv_final(int nf_parts, int n_parts, const double *__restrict__ part, double *__restrict__ out) {
  double e = 0.0, cm = 0.0, pm = 0.0;
  for (int i = threadIdx.x; i < n_parts; i += kThreads) e = fmax(e, part[i]);
  for (int i = threadIdx.x; i < nf_parts; i += kThreads) {
    cm = fmax(cm, part[kParts + i]);
    pm = fmax(pm, part[2 * kParts + i]);
  }
  block_max(e, out);
  block_max(cm, out + 1);
  block_max(pm, out + 2);
}

// ---- Compute_Pressure_Fractional's face loop -----------------------------------

// Per cell slot, once per call, what the faces gather: the velocity with the
// pressure-gradient term put back, u + p_x vol / sav (the raw velocity for a
// boundary cell, which the reference's boundary faces read), sav, p and the
// density -- six values side by side, so a face reads two records instead of
// twenty scattered arrays.  Each value is the one the reference's face
// expression forms, so the result stays bitwise.  Records go into the lists'
// order; reordered ones are 64 bytes apart (R 8), so that each is one aligned
// access, the others 48 (R 6), read in runs.  At 128^3 numbered at random the
// faces took 255 us with the records in the caller's order and take 153; writing
// them out of order costs 114 us here against 63.
template <int R>
__global__ void __launch_bounds__(kThreads)
k_pf_cells(int n, long long na, const int *__restrict__ of, const double *__restrict__ vol,
           const double *__restrict__ sav, const double *__restrict__ u,
           const double *__restrict__ v, const double *__restrict__ w,
           const double *__restrict__ px, const double *__restrict__ py,
           const double *__restrict__ pz, const double *__restrict__ p,
           const double *__restrict__ den, double *__restrict__ rec) {
  for (long long c = blockIdx.x * (long long)kThreads + threadIdx.x; c < na;
       c += (long long)gridDim.x * kThreads) {
    double r[R] = {u[c], v[c], w[c], 0.0, p[c], den[c]};
    if (c < n) {
      r[0] = u[c] + px[c] * vol[c] / sav[c];
      r[1] = v[c] + py[c] * vol[c] / sav[c];
      r[2] = w[c] + pz[c] * vol[c] / sav[c];
      r[3] = sav[c];
    }
    double2 *const to =
        reinterpret_cast<double2 *>(rec + R * (of && c < n ? (long long)of[c] : c));
#pragma unroll
    for (int j = 0; j < R / 2; ++j) to[j] = make_double2(r[2 * j], r[2 * j + 1]);
  }
}

// Compute_Pressure_Fractional.f90:50-131 for fluid materials without BUFFER
// faces: per face the f-weighted density, the face velocity rebuilt from the
// cells' velocities and pressure gradients (Rhie-Chow), the flux and A12;
// a boundary face takes its boundary cell's velocity and has A12 = 0.
template <int R>
__global__ void __launch_bounds__(kThreads)
k_pf_faces(int n, long long nf, const int2 *__restrict__ pairs, const double *__restrict__ f,
           const double *__restrict__ sv, const double *__restrict__ rec,
           double *__restrict__ flux, double *__restrict__ a12) {
  for (long long s = blockIdx.x * (long long)kThreads + threadIdx.x; s < nf;
       s += (long long)gridDim.x * kThreads) {
    const int2 fc = pairs[s];
    const double *r1 = rec + R * (long long)fc.x, *r2 = rec + R * (long long)fc.y;
    const double fs = f[s], sx = sv[s], sy = sv[nf + s], sz = sv[2 * nf + s];
    const double dens = fs * r1[5] + (1.0 - fs) * r2[5];
    if (fc.y < n) {
      const double sav1 = r1[3], sav2 = r2[3];
      double us = fs * r1[0] + (1.0 - fs) * r2[0];
      double vs = fs * r1[1] + (1.0 - fs) * r2[1];
      double ws = fs * r1[2] + (1.0 - fs) * r2[2];
      const double wsav = fs / sav1 + (1.0 - fs) / sav2;
      const double dp = r1[4] - r2[4];
      us = us + dp * sx * wsav;
      vs = vs + dp * sy * wsav;
      ws = ws + dp * sz * wsav;
      flux[s] = dens * (us * sx + vs * sy + ws * sz);
      const double a = dens * (sx * sx + sy * sy + sz * sz);
      a12[s] = a * wsav;
    } else {
      flux[s] = dens * (r2[0] * sx + r2[1] * sy + r2[2] * sz);
      a12[s] = 0.0;
    }
  }
}

// Compute_Pressure_Simple.f90:50-177 for fluid materials without BUFFER
// faces: per interior face SMDPN = |S|^2 / (S . d), A12 = 0.5 DENs SMDPN
// (vol1/sav1 + vol2/sav2), the interpolated velocity and pressure gradient and
// the face flux; per boundary face by the kind of its boundary cell: the flux
// from the boundary cell's velocity (inflow, outflow, convective) or the
// inside cell's (pressure), A12 = DENs SMDPN vol1/sav1 added to the diagonal
// (bnd_on) for outflow, convective and pressure boundaries, no flux on walls
// and symmetry planes.  Every expression in the reference's order.
__global__ void __launch_bounds__(kThreads)
k_ps_faces(int n, long long nf, const int2 *__restrict__ faces,
           const unsigned char *__restrict__ kind, const double *__restrict__ f,
           const double *__restrict__ sv, const double *__restrict__ dv,
           const double *__restrict__ vol, const double *__restrict__ sav,
           const double *__restrict__ u, const double *__restrict__ v,
           const double *__restrict__ w, const double *__restrict__ p,
           const double *__restrict__ px, const double *__restrict__ py,
           const double *__restrict__ pz, const double *__restrict__ den,
           double *__restrict__ flux, double *__restrict__ a12,
           unsigned char *__restrict__ bnd_on) {
  for (long long s = blockIdx.x * (long long)kThreads + threadIdx.x; s < nf;
       s += (long long)gridDim.x * kThreads) {
    const int2 fc = faces[s];
    const long long k1 = fc.x - 1;
    const long long k2 = fc.y > 0 ? (long long)(fc.y - 1) : (long long)n + (-fc.y - 1);
    const double fs = f[s], sx = sv[s], sy = sv[nf + s], sz = sv[2 * nf + s];
    const double dx = dv[s], dy = dv[nf + s], dz = dv[2 * nf + s];
    const double dens = fs * den[k1] + (1.0 - fs) * den[k2];
    double fl = 0.0, a = 0.0;
    unsigned char on = 0;
    if (fc.y > 0) {
      const double smdpn = (sx * sx + sy * sy + sz * sz) / (sx * dx + sy * dy + sz * dz);
      const double us = fs * u[k1] + (1.0 - fs) * u[k2];
      const double vs = fs * v[k1] + (1.0 - fs) * v[k2];
      const double ws = fs * w[k1] + (1.0 - fs) * w[k2];
      a = 0.5 * dens * smdpn * (vol[k1] / sav[k1] + vol[k2] / sav[k2]);
      const double dpxi = .5 * (px[k1] + px[k2]) * dx;
      const double dpyi = .5 * (py[k1] + py[k2]) * dy;
      const double dpzi = .5 * (pz[k1] + pz[k2]) * dz;
      fl = dens * (us * sx + vs * sy + ws * sz) + a * (p[k1] - p[k2]) + a * (dpxi + dpyi + dpzi);
    } else {
      const int kd = kind[-fc.y - 1];
      if (kd == TFS_BC_INFLOW || kd == TFS_BC_OUTFLOW || kd == TFS_BC_CONVECT ||
          kd == TFS_BC_PRESSURE) {
        const long long kv = kd == TFS_BC_PRESSURE ? k1 : k2;
        fl = dens * (u[kv] * sx + v[kv] * sy + w[kv] * sz);
        if (kd != TFS_BC_INFLOW) {
          const double smdpn = (sx * sx + sy * sy + sz * sz) / (sx * dx + sy * dy + sz * dz);
          a = dens * smdpn * vol[k1] / sav[k1];
          on = 1;
        }
      }
    }
    flux[s] = fl;
    a12[s] = a;
    bnd_on[s] = on;
  }
}

// A cell field out of the lists' order.
__global__ void __launch_bounds__(kThreads)
k_out_of_order(int n, const int *__restrict__ of, const double *__restrict__ in,
               double *__restrict__ out) {
  for (int c = blockIdx.x * kThreads + threadIdx.x; c < n; c += gridDim.x * kThreads)
    out[c] = in[of[c]];
}

}  // namespace

struct tfs_gradient {
  int n = 0, nb = 0;
  long long nf = 0;
  DevFaceLists lists;
  GradEntries ent{};
  int n_extrap = 0;           // cells (list positions) with extrapolated boundary faces
  int *extrap = nullptr;
  bool has_buffer = false;    // some boundary cell is of kind TFS_BC_BUFFER
  int2 *faces = nullptr;      // (c1, c2) as the caller numbers them
  int2 *pairs = nullptr;      // both cells' list positions (n and up: boundary slots)
  double *d = nullptr, *g = nullptr, *xc = nullptr;
  unsigned char *kind = nullptr;
  double *part = nullptr;     // 3 kParts partial maxima + 3 results
  double *field = nullptr;    // a cell field in the lists' order (reordered cells only)
  Rec4 *rec = nullptr;        // a gradient in that order
  double *prec = nullptr;     // the pressure face loop's cell records (lazy)
  // A call holds this from its first launch to its last: the arrays above are
  // the object's own, so another thread's calls on it must not come between.
  std::mutex mu;
};

extern "C" int tfs_gradient_destroy(tfs_gradient *S) {
  if (!S) return TFS_OK;
  for (void *p : {(void *)S->ent.other, (void *)S->ent.w, (void *)S->extrap, (void *)S->faces,
                  (void *)S->pairs, (void *)S->d, (void *)S->g, (void *)S->xc, (void *)S->kind,
                  (void *)S->part, (void *)S->field, (void *)S->rec, (void *)S->prec})
    if (p) (void)hipFree(p);
  S->lists.release();
  delete S;
  return TFS_OK;
}

extern "C" int tfs_gradient_create(int n_cells, int n_bnd_cells, long long n_faces,
                                   const int *faces_c, const double *d, const double *xc,
                                   const unsigned char *bc, tfs_gradient **out) {
  if (!out) return TFS_ERR_INVALID;
  *out = nullptr;
  if (n_cells < 1 || n_bnd_cells < 0 || n_faces < 0 || (n_faces > 0 && (!faces_c || !d)))
    return TFS_ERR_INVALID;
  const int n = n_cells, nb = n_bnd_cells;
  const long long nf = n_faces;
  std::vector<int> seen((size_t)nb, 0);
  std::vector<unsigned char> kinds((size_t)std::max(nb, 1), 0);
  bool any_buffer = false;
  std::vector<int> inside;    // cells with an extrapolated boundary face
  for (long long s = 0; s < nf; ++s) {
    const int c1 = faces_c[2 * s], c2 = faces_c[2 * s + 1];
    if (c1 < 1 || c1 > n || c2 == 0 || c2 > n || c2 < -nb) return TFS_ERR_INVALID;
    if (c2 < 0) {
      // a boundary cell belongs to one face: GradP writes it from that face
      if (seen[(size_t)(-c2 - 1)]++) return TFS_ERR_INVALID;
      const int kind = bc ? bc[-c2 - 1] : TFS_BC_WALL;
      if (kind > TFS_BC_CONVECT) return TFS_ERR_INVALID;
      kinds[(size_t)(-c2 - 1)] = (unsigned char)kind;
      any_buffer = any_buffer || kind == TFS_BC_BUFFER;
      if (kind != TFS_BC_BUFFER && kind != TFS_BC_PRESSURE) inside.push_back(c1 - 1);
    }
  }
  FaceLists F;
  build_face_lists(n, nf, faces_c, 1, kReorderGradient, F);
  std::vector<int2> pairs((size_t)nf);
  for (long long s = 0; s < nf; ++s) {
    const int c2 = faces_c[2 * s + 1];
    pairs[(size_t)s] = make_int2(F.at(faces_c[2 * s] - 1), c2 > 0 ? F.at(c2 - 1) : n + (-c2 - 1));
  }
  for (int &c : inside) c = F.at(c);
  std::sort(inside.begin(), inside.end());
  inside.erase(std::unique(inside.begin(), inside.end()), inside.end());
  auto *S = new tfs_gradient;
  S->n = n;
  S->nb = nb;
  S->nf = nf;
  S->has_buffer = any_buffer;
  S->n_extrap = (int)inside.size();
  auto up = [](void **dst, const void *src, size_t bytes) -> bool {
    if (hipMalloc(dst, std::max<size_t>(bytes, 8)) != hipSuccess) return false;
    return bytes == 0 || !src || hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice) == hipSuccess;
  };
  const size_t na = (size_t)n + (size_t)nb;
  bool ok = S->lists.upload(F);
  const size_t m = (size_t)S->lists.entries;
  S->ent.entries = (long long)m;
  ok = ok && up((void **)&S->ent.other, nullptr, sizeof(int) * m) &&
       up((void **)&S->ent.w, nullptr, 3 * sizeof(double) * m) &&
       up((void **)&S->extrap, inside.data(), sizeof(int) * inside.size()) &&
       up((void **)&S->faces, faces_c, sizeof(int2) * (size_t)nf) &&
       up((void **)&S->pairs, pairs.data(), sizeof(int2) * (size_t)nf) &&
       up((void **)&S->d, d, 3 * sizeof(double) * (size_t)nf) &&
       up((void **)&S->g, nullptr, 6 * sizeof(double) * (size_t)n) &&
       up((void **)&S->kind, kinds.data(), kinds.size()) &&
       up((void **)&S->part, nullptr, sizeof(double) * (3 * (size_t)kParts + 3)) &&
       (!F.reordered || (up((void **)&S->field, nullptr, sizeof(double) * (size_t)n) &&
                         up((void **)&S->rec, nullptr, sizeof(Rec4) * (size_t)n))) &&
       (!xc || up((void **)&S->xc, xc, 3 * sizeof(double) * na));
  if (!ok) {
    (void)hipGetLastError();
    tfs_gradient_destroy(S);
    return TFS_ERR_NOMEM;
  }
  hipLaunchKernelGGL(k_gmatrix, dim3(grid_of(S->lists.lanes())), dim3(kThreads), 0, nullptr,
                     S->lists.at, nf, S->pairs, S->kind, S->d, S->g, S->ent);
  if (hipGetLastError() != hipSuccess || hipStreamSynchronize(nullptr) != hipSuccess) {
    (void)hipGetLastError();
    tfs_gradient_destroy(S);
    return TFS_ERR_DEVICE;
  }
  *out = S;
  return TFS_OK;
}

namespace {

// The cells of a field in the lists' order.
const double *in_order(tfs_gradient *S, const double *phi) {
  if (!S->field) return phi;
  hipLaunchKernelGGL(k_into_order, dim3(grid_of(S->n)), dim3(kThreads), 0, nullptr, S->n,
                     S->lists.at.orig, phi, S->field);
  return S->field;
}

void gradient(tfs_gradient *S, const double *phi, double *px, double *py, double *pz) {
  const double *cells = in_order(S, phi);
  hipLaunchKernelGGL(k_graphi, dim3(grid_of(S->lists.lanes())), dim3(kThreads), 0, nullptr,
                     S->lists.at, S->ent, cells, phi, px, py, pz, S->rec);
  if (S->rec)
    hipLaunchKernelGGL(k_from_order, dim3(grid_of(S->n)), dim3(kThreads), 0, nullptr, S->n,
                       S->lists.of, S->rec, px, py, pz);
}

// The right-hand side of the pressure face loops: each cell's fluxes.
void flux_sum(tfs_gradient *S, const double *flux, double *out) {
  hipLaunchKernelGGL(k_flux_sum, dim3(grid_of(S->lists.lanes())), dim3(kThreads), 0, nullptr,
                     S->lists.at, flux, S->field ? S->field : out);
}

void flux_sum_in_cells(tfs_gradient *S, const double *flux, double *out) {
  flux_sum(S, flux, out);
  if (S->field)
    hipLaunchKernelGGL(k_out_of_order, dim3(grid_of(S->n)), dim3(kThreads), 0, nullptr, S->n,
                       S->lists.of, S->field, out);
}

}  // namespace

extern "C" int tfs_gradient_matrix_get(tfs_gradient *S, double *g) {
  if (!S || !g) return TFS_ERR_INVALID;
  std::vector<double> soa(6 * (size_t)S->n);
  TFS_G_HIP(hipMemcpy(soa.data(), S->g, sizeof(double) * soa.size(), hipMemcpyDeviceToHost));
  for (int c = 0; c < S->n; ++c)
    for (int k = 0; k < 6; ++k) g[6 * (size_t)c + k] = soa[(size_t)k * S->n + c];
  return TFS_OK;
}

extern "C" int tfs_grad_phi_device(tfs_gradient *S, const double *d_phi, double *d_px,
                                   double *d_py, double *d_pz) {
  if (!S || !d_phi || !d_px || !d_py || !d_pz) return TFS_ERR_INVALID;
  std::lock_guard<std::mutex> lk(S->mu);
  gradient(S, d_phi, d_px, d_py, d_pz);
  TFS_G_HIP(hipGetLastError());
  TFS_G_HIP(hipStreamSynchronize(nullptr));
  return TFS_OK;
}

extern "C" int tfs_grad_p_device(tfs_gradient *S, double *d_phi, double *d_px, double *d_py,
                                 double *d_pz) {
  if (!S || !d_phi || !d_px || !d_py || !d_pz || (S->n_extrap > 0 && !S->xc))
    return TFS_ERR_INVALID;
  std::lock_guard<std::mutex> lk(S->mu);
  if (S->n_extrap > 0)
    hipLaunchKernelGGL(k_bnd_extrap, dim3(grid_of(S->n_extrap)), dim3(kThreads), 0, nullptr,
                       S->n_extrap, S->extrap, S->lists.at, S->ent, S->pairs, S->kind, S->xc,
                       (long long)S->n + S->nb, d_phi);
  gradient(S, d_phi, d_px, d_py, d_pz);
  TFS_G_HIP(hipGetLastError());
  TFS_G_HIP(hipStreamSynchronize(nullptr));
  return TFS_OK;
}

extern "C" int tfs_correct_velocity_device(tfs_gradient *S, const double *d_vol,
                                           const double *d_sav, const double *d_px,
                                           const double *d_py, const double *d_pz, double *d_u,
                                           double *d_v, double *d_w, const double *d_pp,
                                           const double *d_coef, const double *d_bou,
                                           const double *d_den, const unsigned char *d_in_m,
                                           const double *d_scoef, double dt, double visc,
                                           double *d_flux, double *d_b, double *errmax,
                                           double *cfl_max, double *pe_max) {
  if (!S || !d_vol || !d_sav || !d_px || !d_py || !d_pz || !d_u || !d_v || !d_w || !d_pp ||
      !d_den || !d_b || (S->nf > 0 && (!d_coef || !d_scoef || !d_flux)))
    return TFS_ERR_INVALID;
  std::lock_guard<std::mutex> lk(S->mu);
  const int gc = grid_of(S->n), gf = grid_of(S->nf);
  double *part = S->part;
  hipLaunchKernelGGL(k_cv_cells, dim3(gc), dim3(kThreads), 0, nullptr, S->n, d_vol, d_sav, d_px,
                     d_py, d_pz, d_u, d_v, d_w);
  hipLaunchKernelGGL(k_cv_faces, dim3(gf), dim3(kThreads), 0, nullptr, S->n, S->nf, S->pairs,
                     S->lists.at.orig, S->kind, in_order(S, d_pp), d_pp, d_coef, d_bou, d_in_m, d_scoef, S->d, dt, visc, d_flux, d_u,
                     d_v, d_w, part + kParts, part + 2 * kParts);
  flux_sum(S, d_flux, d_b);
  hipLaunchKernelGGL(k_cv_mass, dim3(gc), dim3(kThreads), 0, nullptr, S->n, S->lists.of,
                     S->field ? S->field : d_b, d_vol, d_den, d_b, part);
  hipLaunchKernelGGL(k_cv_final, dim3(1), dim3(kThreads), 0, nullptr, gf, gc, part,
                     part + 3 * kParts);
  TFS_G_HIP(hipGetLastError());
  double out[3];
  TFS_G_HIP(hipMemcpy(out, part + 3 * kParts, sizeof(out), hipMemcpyDeviceToHost));
  if (errmax) *errmax = out[0];
  if (cfl_max) *cfl_max = out[1];
  if (pe_max) *pe_max = out[2];
  return TFS_OK;
}

extern "C" int tfs_pressure_fractional_device(tfs_gradient *S, const double *d_f,
                                              const double *d_s, const double *d_vol,
                                              const double *d_sav, const double *d_u,
                                              const double *d_v, const double *d_w,
                                              const double *d_px, const double *d_py,
                                              const double *d_pz, const double *d_p,
                                              const double *d_den, double *d_flux,
                                              double *d_a12, double *d_b) {
  if (!S || S->has_buffer || !d_vol || !d_sav || !d_u || !d_v || !d_w || !d_px || !d_py ||
      !d_pz || !d_p || !d_den || !d_b ||
      (S->nf > 0 && (!d_f || !d_s || !d_flux || !d_a12)))
    return TFS_ERR_INVALID;
  const long long na = (long long)S->n + S->nb;
  std::lock_guard<std::mutex> lk(S->mu);
  // the per-cell records (48 bytes per cell slot, 64 reordered) on the first
  // call only: meshes that never run this face loop do not hold them
  const bool far = S->field != nullptr;
  if (!S->prec && hipMalloc((void **)&S->prec, std::max<size_t>((far ? 8 : 6) * sizeof(double) *
                                                                (size_t)na, 8)) != hipSuccess) {
    (void)hipGetLastError();
    S->prec = nullptr;
    return TFS_ERR_NOMEM;
  }
  hipLaunchKernelGGL(far ? k_pf_cells<8> : k_pf_cells<6>, dim3(grid_of(na)), dim3(kThreads), 0,
                     nullptr, S->n, na, S->lists.of, d_vol, d_sav, d_u, d_v, d_w, d_px, d_py,
                     d_pz, d_p, d_den, S->prec);
  if (S->nf > 0)
    hipLaunchKernelGGL(far ? k_pf_faces<8> : k_pf_faces<6>, dim3(grid_of(S->nf)), dim3(kThreads),
                       0, nullptr, S->n, S->nf, S->pairs, d_f, d_s, S->prec, d_flux, d_a12);
  flux_sum_in_cells(S, d_flux, d_b);
  TFS_G_HIP(hipGetLastError());
  TFS_G_HIP(hipStreamSynchronize(nullptr));
  return TFS_OK;
}

extern "C" int tfs_pressure_simple_device(tfs_gradient *S, const double *d_f, const double *d_s,
                                          const double *d_vol, const double *d_sav,
                                          const double *d_u, const double *d_v,
                                          const double *d_w, const double *d_px,
                                          const double *d_py, const double *d_pz,
                                          const double *d_p, const double *d_den,
                                          double *d_flux, double *d_a12,
                                          unsigned char *d_bnd_on, double *d_b) {
  if (!S || S->has_buffer || !d_vol || !d_sav || !d_u || !d_v || !d_w || !d_px || !d_py ||
      !d_pz || !d_p || !d_den || !d_b ||
      (S->nf > 0 && (!d_f || !d_s || !d_flux || !d_a12 || !d_bnd_on)))
    return TFS_ERR_INVALID;
  std::lock_guard<std::mutex> lk(S->mu);
  if (S->nf > 0)
    hipLaunchKernelGGL(k_ps_faces, dim3(grid_of(S->nf)), dim3(kThreads), 0, nullptr, S->n, S->nf,
                       S->faces, S->kind, d_f, d_s, S->d, d_vol, d_sav, d_u, d_v, d_w, d_p, d_px,
                       d_py, d_pz, d_den, d_flux, d_a12, d_bnd_on);
  flux_sum_in_cells(S, d_flux, d_b);
  TFS_G_HIP(hipGetLastError());
  TFS_G_HIP(hipStreamSynchronize(nullptr));
  return TFS_OK;
}
