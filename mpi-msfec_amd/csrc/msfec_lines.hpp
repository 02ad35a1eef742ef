// Direct solve of 9-point systems on refined boxes by lines of nodes
// (msfec_lines.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace msfec_detail {

// 2^l fine cells per direction, 2^l - 1 inner nodes.  Whether there is a kernel.
inline bool lines_has(int l) { return l == 4 || l == 5; }
// Scratch per cell in doubles.
size_t lines_doubles(int l);
// K X = R for a batch of symmetric positive definite systems.  rows
// [cells][n][24]: the diagonal, the present ones of the lower entries left,
// below-right, below, below-left in this order; from 16 on 8 right-hand sides.
// X [cells][n][8].  status: MSFEC_CELL_OK, or MSFEC_CELL_NOT_SPD where a pivot
// is not positive and finite (X is then of no use).
hipError_t lines_solve(int l, int n_cells, const double* rows, double* work, double* X,
                       int* status, hipStream_t s);

}  // namespace msfec_detail
