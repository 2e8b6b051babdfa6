// tfs_internal.hpp -- what the library's other translation units need of a
// tfs_matrix beyond the C ABI (C++ linkage, not exported by the headers).
#pragma once

#include <hip/hip_runtime.h>

#include "tfs_solver.h"

namespace tfs {
// The matrix's own stream: work queued on it is ordered with its solves.
hipStream_t matrix_stream(const tfs_matrix *A);
// Workgroups of the heaviest persistent sweep kernel that fit on the GPU at
// once, and a cap on one matrix's persistent sweep grid (at least 1).
int sweep_capacity(const tfs_matrix *A);
void set_sweep_grid(tfs_matrix *A, int groups);
// tfs_matrix_create for a matrix whose solves run beside other matrices'
// (the server): without the block sweeps, so that the sweep grids' shares of
// one kernel's occupancy hold, and with the sweeps' triangles allocated from the
// start, so that a later request with another preconditioner takes no memory
// that was not accounted for when the case came in.
int matrix_create_shared(int n, long long nnz, const int *row, const int *col, const int *dia,
                         int base, tfs_matrix **out);
}  // namespace tfs
