// Constants of the reference cell in 3-D.
#pragma once

namespace msfec_cell {

// QGauss(2) on [0, 1]
constexpr double kGp[2] = {0.21132486540518711775, 0.78867513459481288225};
// deal.II's line order on the unit cube: axis, and the fixed values of the
// two other coordinates (lower axis first)
constexpr int kLnAx[12] = {1, 1, 0, 0, 1, 1, 0, 0, 2, 2, 2, 2};
constexpr int kLnF1[12] = {0, 1, 0, 1, 0, 1, 0, 1, 0, 1, 0, 1};
constexpr int kLnF2[12] = {0, 0, 0, 0, 1, 1, 1, 1, 0, 0, 1, 1};

}  // namespace msfec_cell
