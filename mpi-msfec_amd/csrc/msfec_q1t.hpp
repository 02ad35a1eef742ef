// Q1 problems with a tensor coefficient on the 2^l-refined box of one coarse
// cell (3-D): the assembled rows of the interior nodes (27 points, symmetric, the
// lower half of them kept), and conjugate gradients on them.  Host entry points of msfec_q1t.hip.
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
  const double* verts;   // n_cells x 8 x 3
  const double* a;       // n_cells x M^3 x 8 x 6: the symmetric tensor at the Gauss points,
                         // or with `scalar` one value per fine cell
  const double* reac;    // one value per fine cell, or null: reac0 everywhere
  double* st;            // n_cells x 15 x M^3, entry-major: the entries to the lower neighbours and
                         // the diagonal ((dz+1) 9 + (dy+1) 3 + dx+1 = 0 .. 13), zero to boundary
                         // nodes, and the inverse diagonal
  double* rhs;           // n_cells x nr x M^3
  int* bad;              // (edge) n_cells: set to 1 where a tensor is not positive definite
  int n_cells, nr;       // nr = 12 (edge) or at most 8 (nodal) right-hand sides
  bool scalar, edge;     // edge: -(a N_n, grad phi) of the 12 coarse Nedelec functions;
                         // otherwise -K g_n of the coarse Q1 functions on the boundary
  double reac0;
};

struct Q1tCg {
  const double* st;   // as Q1tRows::st
  const double* rhs;  // n_cells x nr x M^3
  double* x;          // n_cells x nr x M^3
  const int* skip;    // n_cells, or null: cells left alone
  int* iters;         // n_cells x nr x 2: iterations, state (0 ok, 1 limit, 2 breakdown, 3 not finite)
  int n_cells, nr, max_iter;
  bool direct;        // l <= 2: elimination
  double tol;         // |r| <= tol |b|
};

// Psi, element matrix and load of the Q1 bases from their interior values
struct Q1tBasis {
  const double* verts;
  const double* a;
  const double* reac;
  const double* f;     // load, or null: f0
  const double* x;     // n_cells x nr x M^3; nr = 7: the last basis is one minus the others
  const int* iters;    // n_cells x nr x 2
  double* part;        // n_cells x slabs x 48 (q1t_slabs)
  double* Psi;         // n_cells x 8 x (M + 1)^3
  double* Mat;         // n_cells x 64
  double* b;           // n_cells x 8
  int* cgit;           // n_cells x 8 x 2
  int* status;
  int n_cells, nr;
  int per_point;       // load values per fine cell: 1 or 8
  bool scalar;
  double reac0, f0;
};

int q1t_slabs(int l);
hipError_t q1t_basis(int l, const Q1tBasis& g, hipStream_t s);
hipError_t q1t_rows(int l, const Q1tRows& g, hipStream_t s);
// conjugate gradients, or elimination with `direct` (l <= 2 only)
hipError_t q1t_solve(int l, const Q1tCg& g, hipStream_t s);

}  // namespace msfec_detail
