// 9-point systems of a refined box in 2-D by block cyclic reduction over the
// lines of nodes.
//
// The band factorisation of such a system is a chain of n / 4 steps that one
// wave takes one after the other, 2 us each with the way back.
// Here the lines 1, 3, 5, ... are eliminated at once, each by a wave of its
// own, then 2, 6, 10, ..., and so on: l levels of which each costs about one
// factorisation of a line block.  A line J with neighbours A and B (s = 1, 2,
// 4, ... lines away): D_J = L L^T, W = L^-1 [K_JA K_JB F_J], then
// K_AA -= W_A^T W_A, K_BB -= W_B^T W_B, K_AB -= W_A^T W_B, and the same for
// the right-hand sides; back, x_J = L^-T (W_F - W_A x_A - W_B x_B).
//
// All blocks are 16 x 16 tiles in the accumulator layout of
// v_mfma_f64_16x16x4f64: entry (i, j) in register i / 4 of lane j + 16 (i % 4).
// Register c is then also both the operand X^T[:, 4c .. 4c+3] and the operand
// X[4c .. 4c+3, :], so that X^T Y of two tiles takes four instructions and no
// exchange; with the inverse U = L^-T of a factor as a tile, every product
// above has that form.  A tile in memory is row-major, a register a coalesced
// load.
//
// Bound by the chain of a level (two passes of 16 dependent pivots at 31 nodes a
// line) and by the matrix instructions, 64 clocks each: 1024 systems of 15^2
// nodes take 71 us, 111 by the band factorisation with one wave per cell; 121
// of 31^2 145 us and 463.  Products with explicit inverses in place of
// substitutions leave 3 to 10 % more rounding in the fluxes (l = 4 8.0e-16 and
// 7.8e-16 in the mean, l = 5 with tensors 2.0e-15 and 1.8e-15; multipliers with
// 1 / pivot instead of two factors with its root changed nothing and took 2 %).
#include "msfec_lines.hpp"

#include "msfec.h"
#include "msfec_wave.hpp"

namespace {

typedef double v4 __attribute__((ext_vector_type(4)));

constexpr int kLen = 24, kRhs = 16;  // a row of the table, its right-hand sides

template <int TT>
struct Lines {
  static constexpr int M = 16 * TT, MI = M - 1, TB = TT * TT;
  static constexpr int NW = TT == 1 ? 4 : 8;
  // of the diagonal blocks the upper tiles (0,0), (0,1), (1,1)
  static constexpr int ND = TT == 1 ? 1 : 3;
  // per line: L^-1 of the diagonal tiles and what links them; W of both
  // neighbours (before: the blocks themselves); W_F
  static constexpr int WL = ND * 256, WR = WL + TB * 256, WF = WR + TB * 256, LINE = WF + TT * 128;
};

// lane K of each row of 16 lanes, in all of them
template <int K>
__device__ __forceinline__ double row_lane(double v) {
  return __hiloint2double(
      __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x150 + K, 0xf, 0xf, false),
      __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x150 + K, 0xf, 0xf, false));
}

// c + X^T Y, c - X^T Y
__device__ __forceinline__ v4 mul(const v4& x, const v4& y, v4 c) {
#pragma unroll
  for (int k = 0; k < 4; ++k) c = __builtin_amdgcn_mfma_f64_16x16x4f64(x[k], y[k], c, 0, 0, 0);
  return c;
}
__device__ __forceinline__ v4 mul_neg(const v4& x, const v4& y, v4 c) {
#pragma unroll
  for (int k = 0; k < 4; ++k) c = __builtin_amdgcn_mfma_f64_16x16x4f64(x[k], y[k], c, 0, 0, 1);
  return c;
}

// z := L^-1 for z = L L^T, in place: after step K the columns up to K hold
// L^-1 and the others the Schur complement.  false if a pivot is not positive
// and finite.
template <int K>
__device__ __forceinline__ void chol_step(v4& z, int lane, bool& ok) {
  constexpr int R = K / 4, H = K % 4;
  const int lh = lane >> 4, ll = lane & 15;
  const double piv = msfec_wave::lane_value(z[R], 16 * H + K);
  ok = ok && piv > 0.0 && piv < INFINITY;
  const double rs = msfec_wave::inv_sqrt(piv);
  const int from = (16 * H + ll) * 4;
  double row = __hiloint2double(__builtin_amdgcn_ds_bpermute(from, __double2hiint(z[R])),
                                __builtin_amdgcn_ds_bpermute(from, __double2loint(z[R])));
  row = ll == K ? rs : row * rs;
#pragma unroll
  for (int r = R; r < 4; ++r) {
    const double m = row_lane<K>(z[r]) * rs;
    const double v = fma(-m, row, ll == K ? 0.0 : z[r]);
    if (r > R) z[r] = v;
    else z[r] = lh > H ? v : lh == H ? row : z[r];
  }
  if constexpr (K < 15) chol_step<K + 1>(z, lane, ok);
}
__device__ __forceinline__ bool inverse_factor(v4& z, int lane) {
  bool ok = true;
  chol_step<0>(z, lane, ok);
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if ((lane & 15) > 4 * r + (lane >> 4)) z[r] = 0.0;
  return ok;
}
// the transpose: the product of x^T with the unit tile, exact
__device__ __forceinline__ v4 transpose(const v4& x, int lane) {
  v4 e, c = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int r = 0; r < 4; ++r) e[r] = (lane & 15) == 4 * r + (lane >> 4) ? 1.0 : 0.0;
  return mul(x, e, c);
}

__device__ __forceinline__ v4 load_tile(const double* p, int lane) {
  v4 t;
#pragma unroll
  for (int r = 0; r < 4; ++r) t[r] = p[64 * r + lane];
  return t;
}
__device__ __forceinline__ void store_tile(double* p, const v4& t, int lane) {
#pragma unroll
  for (int r = 0; r < 4; ++r) p[64 * r + lane] = t[r];
}
// tiles of 8 columns: right-hand sides and solutions
__device__ __forceinline__ v4 load_half(const double* p, int lane) {
  v4 t;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const double v = p[8 * (4 * r + (lane >> 4)) + (lane & 7)];
    t[r] = (lane & 8) ? 0.0 : v;
  }
  return t;
}
__device__ __forceinline__ void store_half(double* p, const v4& t, int lane) {
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (!(lane & 8)) p[8 * (4 * r + (lane >> 4)) + (lane & 7)] = t[r];
}
// the operand of the transposed tile: x with x^T in the accumulator layout
__device__ __forceinline__ v4 load_transposed(const double* p, int lane) {
  v4 t;
#pragma unroll
  for (int c = 0; c < 4; ++c) t[c] = p[16 * (lane & 15) + 4 * c + (lane >> 4)];
  return t;
}

template <int TT>
__global__ __launch_bounds__(64 * Lines<TT>::NW, TT == 1 ? 4 : 2) void lines_kernel(const double* __restrict__ rows,
                                                                   double* __restrict__ work,
                                                                   double* __restrict__ X,
                                                                   int* __restrict__ status) {
  typedef Lines<TT> C;
  constexpr int M = C::M, MI = C::MI, NW = C::NW, ND = C::ND;
  // blocks and right-hand sides of the lines that are left (even ones); on the
  // way back the solution of all lines
  constexpr int LEFT = M / 2 - 1, DF = ND * 256 + TT * 128;
  constexpr int SIZE = LEFT * DF > MI * TT * 128 ? LEFT * DF : MI * TT * 128;
  __shared__ double S[SIZE];
  __shared__ int bad[NW];
  const int cell = blockIdx.x, lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lh = lane >> 4, ll = lane & 15;
  const double* rc = rows + (size_t)cell * MI * MI * kLen;
  double* wc = work + (size_t)cell * MI * C::LINE;
  double* xc = X + (size_t)cell * MI * MI * 8;
  // row of node i (from 0) of line J, its lower entries
  auto row_of = [&](int J, int i) { return rc + (size_t)((J - 1) * MI + i) * kLen; };
  auto left = [&](int J, int i) { return row_of(J, i)[1]; };                       // i > 0
  auto below_right = [&](int J, int i) { return row_of(J, i)[1 + (i > 0)]; };      // J > 1, i < MI - 1
  auto below = [&](int J, int i) { return row_of(J, i)[1 + (i > 0) + (i < MI - 1)]; };
  auto below_left = [&](int J, int i) { return row_of(J, i)[3 + (i < MI - 1)]; };  // i > 0
  // entries of the blocks of line J; the last node of the M is a unit row
  auto diag = [&](int J, int i, int j) {
    double v = 0.0;
    if (i == j) v = i < MI ? row_of(J, i)[0] : 1.0;
    else if (i - j == 1 && i < MI) v = left(J, i);
    else if (j - i == 1 && j < MI) v = left(J, j);
    return v;
  };
  auto lower = [&](int J, int i, int j) {  // to line J - 1
    double v = 0.0;
    if (i < MI && j < MI) {
      if (i == j) v = below(J, i);
      else if (j - i == 1) v = below_right(J, i);
      else if (i - j == 1) v = below_left(J, i);
    }
    return v;
  };
  auto rhs = [&](int J, int t) {
    v4 f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * t + 4 * r + lh;
      f[r] = i < MI && ll < 8 ? row_of(J, i)[kRhs + ll] : 0.0;
    }
    return f;
  };
  // upper tile d of a diagonal block: its row and column of tiles
  auto tr = [](int d) { return d >> 1; };
  auto tc = [](int d) { return (d + 1) >> 1; };
  auto diag_tile = [&](int J, int d) {
    v4 t;
#pragma unroll
    for (int r = 0; r < 4; ++r) t[r] = diag(J, 16 * tr(d) + 4 * r + lh, 16 * tc(d) + ll);
    return t;
  };
  double* const Sd = S;                   // [line / 2 - 1][ND][256]
  double* const Sf = S + LEFT * ND * 256;  // [line / 2 - 1][TT][128]
  for (int q = wave; q < LEFT; q += NW) {
#pragma unroll
    for (int d = 0; d < ND; ++d) store_tile(Sd + (q * ND + d) * 256, diag_tile(2 * q + 2, d), lane);
#pragma unroll
    for (int t = 0; t < TT; ++t) store_half(Sf + (q * TT + t) * 128, rhs(2 * q + 2, t), lane);
  }
  bool ok = true;
#pragma unroll 1
  for (int s = 1; s < M; s *= 2) {
    const int count = M / (2 * s);
#pragma unroll 1
    for (int q0 = 0; q0 < count; q0 += NW) {
      const bool on = q0 + wave < count;
      const int J = s * (2 * (q0 + wave) + 1);
      const bool has_a = on && J - s > 0, has_b = on && J + s < M;
      double* const line = wc + (size_t)(J - 1) * C::LINE;
      v4 A[TT][TT], B[TT][TT], F[TT];
      if (s > 1) __syncthreads();  // the level before is done with the diagonal blocks
      if (on) {
        v4 D[ND];
        if (s == 1) {
#pragma unroll
          for (int d = 0; d < ND; ++d) D[d] = diag_tile(J, d);
#pragma unroll
          for (int t = 0; t < TT; ++t) {
            F[t] = rhs(J, t);
#pragma unroll
            for (int u = 0; u < TT; ++u)
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const int i = 16 * t + 4 * r + lh, j = 16 * u + ll;
                A[t][u][r] = has_a ? lower(J, i, j) : 0.0;
                B[t][u][r] = has_b ? lower(J + 1, j, i) : 0.0;
              }
          }
        } else {
          const int e = J / 2 - 1;
#pragma unroll
          for (int d = 0; d < ND; ++d) D[d] = load_tile(Sd + (e * ND + d) * 256, lane);
#pragma unroll
          for (int t = 0; t < TT; ++t) {
            F[t] = load_half(Sf + (e * TT + t) * 128, lane);
#pragma unroll
            for (int u = 0; u < TT; ++u) {
              const v4 zero = {0.0, 0.0, 0.0, 0.0};
              A[t][u] = has_a ? load_tile(line + C::WL + (t * TT + u) * 256, lane) : zero;
              B[t][u] = has_b ? load_tile(line + C::WR + (t * TT + u) * 256, lane) : zero;
            }
          }
        }
        const v4 zero = {0.0, 0.0, 0.0, 0.0};
        ok = inverse_factor(D[0], lane) && ok;
        const v4 U0 = transpose(D[0], lane);
#pragma unroll
        for (int u = 0; u < TT; ++u) {
          A[0][u] = mul(U0, A[0][u], zero);
          B[0][u] = mul(U0, B[0][u], zero);
        }
        F[0] = mul(U0, F[0], zero);
        store_tile(line, D[0], lane);
        if constexpr (TT == 2) {
          const v4 link = mul(U0, D[1], zero);
          v4 last = mul_neg(link, link, D[ND - 1]);
          ok = inverse_factor(last, lane) && ok;
          const v4 U1 = transpose(last, lane);
#pragma unroll
          for (int u = 0; u < TT; ++u) {
            A[TT - 1][u] = mul(U1, mul_neg(link, A[0][u], A[TT - 1][u]), zero);
            B[TT - 1][u] = mul(U1, mul_neg(link, B[0][u], B[TT - 1][u]), zero);
          }
          F[TT - 1] = mul(U1, mul_neg(link, F[0], F[TT - 1]), zero);
          store_tile(line + 256, link, lane);
          store_tile(line + 512, last, lane);
        }
#pragma unroll
        for (int t = 0; t < TT; ++t) {
          store_half(line + C::WF + t * 128, F[t], lane);
#pragma unroll
          for (int u = 0; u < TT; ++u) {
            if (has_a) store_tile(line + C::WL + (t * TT + u) * 256, A[t][u], lane);
            if (has_b) store_tile(line + C::WR + (t * TT + u) * 256, B[t][u], lane);
          }
        }
      }
      __syncthreads();  // the blocks of the lines that are left are filled and free
      auto update = [&](const v4(&W)[TT][TT], int to) {
        const int e = to / 2 - 1;
#pragma unroll
        for (int d = 0; d < ND; ++d) {
          double* p = Sd + (e * ND + d) * 256;
          v4 c = load_tile(p, lane);
#pragma unroll
          for (int t = 0; t < TT; ++t) c = mul_neg(W[t][tr(d)], W[t][tc(d)], c);
          store_tile(p, c, lane);
        }
#pragma unroll
        for (int u = 0; u < TT; ++u) {
          double* p = Sf + (e * TT + u) * 128;
          v4 c = load_half(p, lane);
#pragma unroll
          for (int t = 0; t < TT; ++t) c = mul_neg(W[t][u], F[t], c);
          store_half(p, c, lane);
        }
      };
      if (has_a) update(A, J - s);
      if (has_a && has_b) {
        // the new coupling, as the block of the one that goes next
        const bool first = ((J - s) / (2 * s)) & 1;
        double* p = first ? wc + (size_t)(J - s - 1) * C::LINE + C::WR
                          : wc + (size_t)(J + s - 1) * C::LINE + C::WL;
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
          for (int u = 0; u < TT; ++u) {
            v4 c = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int k = 0; k < TT; ++k)
              c = first ? mul_neg(A[k][t], B[k][u], c) : mul_neg(B[k][t], A[k][u], c);
            store_tile(p + (t * TT + u) * 256, c, lane);
          }
      }
      __syncthreads();
      if (has_b) update(B, J + s);
    }
  }
  if (lane == 0) bad[wave] = !ok;
  // back: Sx [line - 1][TT][16][8]
  double* const Sx = S;
#pragma unroll 1
  for (int s = M / 2; s > 0; s /= 2) {
    const int count = M / (2 * s);
#pragma unroll 1
    for (int q = wave; q < (count + NW - 1) / NW * NW; q += NW) {
      const bool on = q < count;
      const int J = s * (2 * q + 1);
      const bool has_a = on && J - s > 0, has_b = on && J + s < M;
      const double* line = wc + (size_t)(J - 1) * C::LINE;
      v4 Z[TT], A[TT][TT], B[TT][TT], I[ND];
      if (on) {
#pragma unroll
        for (int d = 0; d < ND; ++d)
          I[d] = d == 1 ? load_transposed(line + 256, lane) : load_tile(line + d * 256, lane);
#pragma unroll
        for (int t = 0; t < TT; ++t) {
          Z[t] = load_half(line + C::WF + t * 128, lane);
#pragma unroll
          for (int u = 0; u < TT; ++u) {
            if (has_a) A[t][u] = load_transposed(line + C::WL + (t * TT + u) * 256, lane);
            if (has_b) B[t][u] = load_transposed(line + C::WR + (t * TT + u) * 256, lane);
          }
        }
      }
      __syncthreads();  // the level before is done (first: with the blocks)
      if (on) {
        const v4 zero = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int u = 0; u < TT; ++u) {
          if (has_a) {
            const v4 x = load_half(Sx + ((J - s - 1) * TT + u) * 128, lane);
#pragma unroll
            for (int t = 0; t < TT; ++t) Z[t] = mul_neg(A[t][u], x, Z[t]);
          }
          if (has_b) {
            const v4 x = load_half(Sx + ((J + s - 1) * TT + u) * 128, lane);
#pragma unroll
            for (int t = 0; t < TT; ++t) Z[t] = mul_neg(B[t][u], x, Z[t]);
          }
        }
        if constexpr (TT == 2) {
          Z[TT - 1] = mul(I[ND - 1], Z[TT - 1], zero);
          Z[0] = mul_neg(I[ND / 2], Z[TT - 1], Z[0]);
        }
        Z[0] = mul(I[0], Z[0], zero);
#pragma unroll
        for (int t = 0; t < TT; ++t) {
          store_half(Sx + ((J - 1) * TT + t) * 128, Z[t], lane);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int i = 16 * t + 4 * r + lh;
            if (i < MI && ll < 8) xc[(size_t)((J - 1) * MI + i) * 8 + ll] = Z[t][r];
          }
        }
      }
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int any = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) any |= bad[w];
    status[cell] = any ? MSFEC_CELL_NOT_SPD : MSFEC_CELL_OK;
  }
}

template <int TT>
hipError_t launch(int n_cells, const double* rows, double* work, double* X, int* status, hipStream_t s) {
  hipLaunchKernelGGL((lines_kernel<TT>), dim3(n_cells), dim3(64 * Lines<TT>::NW), 0, s, rows, work, X,
                     status);
  return hipGetLastError();
}

}  // namespace

namespace msfec_detail {

size_t lines_doubles(int l) {
  return l == 4 ? (size_t)Lines<1>::MI * Lines<1>::LINE : (size_t)Lines<2>::MI * Lines<2>::LINE;
}

hipError_t lines_solve(int l, int n_cells, const double* rows, double* work, double* X,
                       int* status, hipStream_t s) {
  return l == 4 ? launch<1>(n_cells, rows, work, X, status, s)
                : launch<2>(n_cells, rows, work, X, status, s);
}

}  // namespace msfec_detail
