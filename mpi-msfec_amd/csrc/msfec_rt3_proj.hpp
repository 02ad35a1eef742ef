// The 3-D RT_DQ bases by projected conjugate gradients (msfec_rt3_proj.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace msfec_detail {

struct Rt3Proj {
  const double* verts;  // n_cells x 8 x 3
  const double* ainv;   // n_cells x M^3 x 8 x 6
  const double* fq;     // n_cells x M^3 x 8, or null
  double* MF;           // n_cells x 11 x M^3 x 2: the 21 entries of every fine cell's face mass
  double* bound;        // n_cells x rt3_proj_blocks x 2: extreme eigenvalue bounds of A^-1
  double* part;         // n_cells x rt3_proj_blocks x 32: partial sums of the element matrix
  int* general;         // n_cells: 1 where the cell is left to the general solver
  double* S;            // n_cells x 6 x nf
  double* Mat;          // n_cells x 49
  double* b;            // n_cells x 7
  int* its;             // n_cells x 6
  int* flg;             // n_cells x 6
  int* status;          // n_cells
  int n_cells, max_iter;
  double rtol;
};

int rt3_proj_blocks(int l);
// face masses, then the fluxes of the cells that the method suits (the others
// are flagged in `general`)
hipError_t rt3_proj_masses(int l, const Rt3Proj& g, hipStream_t s);
hipError_t rt3_proj_solve(int l, const Rt3Proj& g, hipStream_t s);
// element matrices and loads of the cells that are not flagged, and the status of all
hipError_t rt3_proj_element(int l, const Rt3Proj& g, hipStream_t s);

}  // namespace msfec_detail
