// The Ned_RT bases without a reaction term, by the discrete exact sequence
// (msfec_nrt_seq.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace msfec_detail {

struct NrtSeq {
  const double* verts;  // n_cells x 8 x 3
  const double* ainv;   // n_cells x M^3 x 8 x 6
  const double* bq;     // n_cells x M^3 x 8
  const double* fq;     // n_cells x M^3 x 8 x 3, or null
  double* W;            // n_cells x (M^3 + 1): 1 / (integral of B / |c|^2) per fine cell, and their sum
  double* st;           // n_cells x 15 x M^3
  double* rhs;          // n_cells x 12 x M^3
  double* phi;          // n_cells x 12 x M^3
  int* iters;           // n_cells x 12 x 2
  int* general;         // n_cells: 1 where the cell is left to the general solver
  double* X;            // n_cells x 18 x N
  double* Mat;          // n_cells x 18 x 18
  double* b;            // n_cells x 18
  int* status;          // n_cells
  int* its;             // n_cells x 18, or null
  int n_cells, max_iter;
  double rtol;
};

// cells not flagged in g.general hold their results afterwards, the flagged
// ones are untouched; `mid` (or null) is recorded before and after the solve
hipError_t nrt_seq(int l, const NrtSeq& g, hipStream_t s, hipEvent_t* mid);

}  // namespace msfec_detail
