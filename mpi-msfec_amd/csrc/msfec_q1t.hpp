// Q1 problems with a tensor coefficient on the 2^l-refined box of one coarse
// cell (3-D): the assembled 27-point rows of the interior nodes, and
// conjugate gradients on them.  Host entry points of msfec_q1t.hip.
//
// Nodes are stored flat, (k M + j) M + i with M = 2^l and i, j, k = 0 .. M-1:
// the nodes of index 0 are the lower boundary (their rows, right-hand sides
// and solutions are zero), those of index M do not exist.  The neighbour of
// flat node n in direction (dx, dy, dz) is n + (dz M + dy) M + dx for every
// interior n: beyond the upper boundary this is a node of index 0, which
// holds zero.
#pragma once
#include <hip/hip_runtime.h>

namespace msfec_detail {

struct Q1tRows {
  const double* verts;  // n_cells x 8 x 3
  const double* a;      // n_cells x M^3 x 8 x 6: the symmetric tensor at the Gauss points
  double* st;           // n_cells x 27 x M^3: rows, entry-major ((dz+1) 9 + (dy+1) 3 + dx+1)
  double* rhs;          // n_cells x 12 x M^3: -(a N_n, grad phi) of the 12 coarse Nedelec functions
  int* bad;             // n_cells: set to 1 where a tensor is not positive definite
  int n_cells;
};

struct Q1tCg {
  const double* st;   // as Q1tRows::st
  const double* rhs;  // n_cells x nr x M^3
  double* x;          // n_cells x nr x M^3
  const int* skip;    // n_cells, or null: cells left alone
  int* iters;         // n_cells x nr x 2: iterations, state (0 ok, 1 limit, 2 breakdown, 3 not finite)
  int n_cells, nr, max_iter;
  double tol;         // |r| <= tol |b|
};

hipError_t q1t_rows(int l, const Q1tRows& g, hipStream_t s);
// conjugate gradients (l = 3, 4) or elimination (l = 1, 2)
hipError_t q1t_solve(int l, const Q1tCg& g, hipStream_t s);

}  // namespace msfec_detail
