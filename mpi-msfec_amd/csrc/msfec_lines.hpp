// Direct solve of 9-point systems on refined boxes by lines of nodes
// (msfec_lines.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace msfec_detail {

// 2^l fine cells per direction, 2^l - 1 inner nodes.  Whether there is a kernel
// and it is the faster one: below l = 4 a line is less than a tile, and many
// cells fill the card with the band factorisation's one wave each, which takes
// fewer operations.  A pass of 2-D RT_DQ, band and this: l = 4 1 cell 108 and 50
// us, 1024 159 and 125, 2025 236 and 238, 4096 473 and 493; l = 5 1 cell 497 and
// 172, 400 569 and 399, 625 619 and 593, 784 667 and 779.
inline bool lines_has(int l, int n_cells) {
  return (l == 4 && n_cells <= 1536) || (l == 5 && n_cells <= 640);
}
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
