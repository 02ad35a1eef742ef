// Ned_RT without a reaction term: the 18 bases of a box by the discrete exact
// sequence instead of one indefinite system per basis.
//
// With d0, d1, d2 the gradient, curl and divergence of the fine complex
// Q1 -> Nedelec -> Raviart-Thomas -> DQ0 (entries +-1 on line integrals,
// fluxes and outflows), Me the edge mass with A^-1, Mf the plain face mass
// and D the diagonal of (B, 1)_c / |c|^2, the system of ned_rt_basis.cc:488-511
// with R = 0 reads on the interior edges and faces
//   Me sigma - d1^T Mf u = 0,   Mf d1 sigma + d2^T D d2 u = Mf d1 N_n  (0 for a face basis).
// Testing the second equation with curls shows d1 sigma = d1 N_n, so
//   edge basis:  sigma = N_n + d0 phi,  d0^T Me (N_n + d0 phi) = 0
// (phi vanishing on the boundary: a Q1 problem with the tensor A^-1), and
//   face basis:  sigma = 0.
// What is left of it is d2^T D d2 u = 0: D d2 u is one constant per cell, so
// the divergence of u is known (zero for an edge basis; for a face basis the
// outflow +-1 shared out in proportion to 1/D).  The first equation then
// gives d1^T Mf u = Me sigma on the interior edges.  u from its divergence
// and this weak curl is a problem with constant coefficients on a tensor
// grid: sines and cosines diagonalise it, mode by mode with
// kappa = 2 sin(k pi / 2M) per direction,
//   edge basis:  y x kappa = g^,  kappa . Mf^-1 y = 0,  u^ = Mf^-1 y,
//   face basis:  u^ = Mf^-1 kappa p^,  kappa . Mf^-1 kappa p^ = d^.
// So 12 scalar problems of (M - 1)^3 unknowns and 13 sets of trigonometric
// transforms per coarse cell replace 18 indefinite solves of all interior
// edges and faces.  Measured, a whole pass with its copies: 4096 cells at l = 2
// 6.81 ms by the dense factorisation, 0.73 ms here; 8 cells at l = 4 with the
// contrast 0.9 of the reference example 345 ms by MINRES (773 iterations),
// 0.95 ms here (50 iterations of CG).
//
// That needs A^-1 positive definite at every Gauss point and B > 0 (and
// finite data): a cell that is not so is flagged and left to the general
// solvers of msfec_nrt.hip, which find out what can be said of it.
#include "msfec_nrt_seq.hpp"

#include "msfec.h"
#include "msfec_cell.hpp"
#include "msfec_q1t.hpp"
#include "msfec_trig.hpp"
#include "msfec_wave.hpp"

namespace {

using msfec_detail::NrtSeq;
using namespace msfec_trig;
using namespace msfec_cell;
using msfec_wave::block_sums;
using msfec_wave::wave_sum;

template <int M>
struct Seq {
  static constexpr int S = M + 1, S3 = S * S * S, M3 = M * M * M;
  static constexpr int NX = M * S * S, NE = 3 * NX, NF1 = M * M * S, N = NE + 3 * NF1;
  static constexpr int NT = M >= 16 ? 512 : (M >= 8 ? 256 : 64);
  static constexpr int NW = NT / 64;
};

// 1 / D per fine cell and their sum; starts the flag of the cell.
template <int M>
__global__ __launch_bounds__(1024) void nrt_seq_weights_kernel(NrtSeq g) {
  constexpr int M3 = M * M * M;
  __shared__ double red[16];
  __shared__ int rbad[16];
  const int cell = blockIdx.x, tid = threadIdx.x, nt = blockDim.x, nw = nt >> 6;
  const double* v = g.verts + (size_t)cell * 24;
  const double vol = (v[3] - v[0]) * (v[7] - v[1]) * (v[14] - v[2]) / M3;
  double* W = g.W + (size_t)cell * (M3 + 1);
  const double2* b2 = reinterpret_cast<const double2*>(g.bq + (size_t)cell * M3 * 8);
  double sum = 0.0;
  int bad = 0;
  for (int c = tid; c < M3; c += nt) {
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const double2 t = b2[c * 4 + q];
      bad |= !(t.x > 0.0) || !(t.y > 0.0);
      s += t.x;
      s += t.y;
    }
    bad |= !isfinite(s);  // an infinite B would only lower the weight to 0
    const double w = vol / (s * 0.125);
    W[c] = w;
    sum += w;
  }
  sum = wave_sum(sum);
  bad = __any(bad);
  if ((tid & 63) == 0) {
    red[tid >> 6] = sum;
    rbad[tid >> 6] = bad;
  }
  __syncthreads();
  if (tid == 0) {
    for (int i = 1; i < nw; ++i) {
      sum += red[i];
      bad |= rbad[i];
    }
    W[M3] = sum;
    g.general[cell] = bad || !(sum > 0.0) || !isfinite(sum);
  }
}

// Coefficient of face F in the curl of the Nedelec function of line L: the
// sense of the line in the circulation around the face, 0 when it is not on
// it.
constexpr int seq_inc(int F, int L) {
  const int ax = kLnAx[L], o1 = ax == 0 ? 1 : 0;
  const int f1 = kLnF1[L], f2 = kLnF2[L], d = F / 2, s = F % 2;
  if (d == ax) return 0;
  if ((d == o1 ? f1 : f2) != s) return 0;
  const int a = (d + 1) % 3, bb = (d + 2) % 3;
  if (ax == a) return (bb == o1 ? f1 : f2) == 0 ? 1 : -1;
  return (a == o1 ? f1 : f2) == 1 ? 1 : -1;
}

// index of edge (axis a) and face (axis a) at (i, j, k)
template <int M>
__device__ __forceinline__ int edge_at(int a, int i, int j, int k) {
  constexpr int S = M + 1, NX = M * S * S;
  if (a == 0) return (k * S + j) * M + i;
  if (a == 1) return NX + (k * M + j) * S + i;
  return 2 * NX + (k * S + j) * S + i;
}

// Workgroup n of a coarse cell: n < 12 the edge basis n, with its column of
// the edge block of the element matrix; n = 12 the 6 face bases and the rest
// of the element matrix and load.
//
// LDS holds the three components on the (M + 1)^3 lattice (118 KB for
// M = 16): Me sigma on the edges, then its transform, then u on the faces.
// 311 us for 4096 cells at M = 4, bound by instruction issue (a wave per
// basis, 4 k instructions); 104 us for 8 cells at M = 16, one round of
// workgroups, bound by the chain of LDS passes and the reads of A^-1.
template <int M>
__global__ __launch_bounds__(Seq<M>::NT) void nrt_seq_basis_kernel(NrtSeq g) {
  typedef Seq<M> Q;
  constexpr int S = Q::S, S3 = Q::S3, M3 = Q::M3, NT = Q::NT, NE = Q::NE, NF1 = Q::NF1;
  extern __shared__ double E[];  // 3 x S^3
  __shared__ double red[Q::NW][16], tot[16], kap[M], tim[3][M];
  const int slot = blockIdx.x >> 3, cell = (slot / 13) * 8 + (blockIdx.x & 7), n = slot % 13;
  if (cell >= g.n_cells || g.general[cell]) return;
  const int tid = threadIdx.x;
  const double* v = g.verts + (size_t)cell * 24;
  const double H[3] = {v[3] - v[0], v[7] - v[1], v[14] - v[2]};
  const double h[3] = {H[0] / M, H[1] / M, H[2] / M};
  const double ih[3] = {M / H[0], M / H[1], M / H[2]};
  const double w8 = h[0] * h[1] * h[2] * 0.125;
  const double mf[3] = {h[0] * ih[1] * ih[2], h[1] * ih[0] * ih[2], h[2] * ih[0] * ih[1]};
  double* X = g.X + (size_t)cell * 18 * Q::N;
  double* Mc = g.Mat + (size_t)cell * 324;
  for (int i = tid; i < 3 * S3; i += NT) E[i] = 0.0;
  if (tid < M) {
    // kappa and the inverse face mass of mode k in each direction
    kap[tid] = 2.0 * sinpi(tid * (0.5 / M));
    const double t = fma(cospi(tid * (1.0 / M)), 1.0 / 3.0, 2.0 / 3.0);
#pragma unroll
    for (int d = 0; d < 3; ++d) tim[d][tid] = 1.0 / (mf[d] * t);
  }
  __syncthreads();
  if (n < 12) {
    const int ax = kLnAx[n], f1 = kLnF1[n], f2 = kLnF2[n];
    const int o1 = ax == 0 ? 1 : 0, o2 = ax == 2 ? 1 : 2;
    const double* phi = g.phi + ((size_t)cell * 12 + n) * M3;
    auto node = [&](int i, int j, int k) {
      return (i < M && j < M && k < M) ? phi[(k * M + j) * M + i] : 0.0;
    };
    // sigma on the edge of axis a starting at (i, j, k)
    auto coarse = [&](int a, int i, int j, int k) {
      if (a != ax) return 0.0;
      const double t1 = (o1 == 0 ? i : j) * (1.0 / M), t2 = (o2 == 2 ? k : j) * (1.0 / M);
      return (f1 ? t1 : 1.0 - t1) * (f2 ? t2 : 1.0 - t2) * (1.0 / M);
    };
    double* x = X + (size_t)n * Q::N;
    for (int e = tid; e < NE; e += NT) {
      const int a = e / Q::NX;
      int r = e - a * Q::NX;
      const int nx = a == 0 ? M : S, ny = a == 1 ? M : S;
      const int i = r % nx;
      r /= nx;
      const int j = r % ny, k = r / ny;
      x[e] = coarse(a, i, j, k) + (node(i + (a == 0), j + (a == 1), k + (a == 2)) - node(i, j, k));
    }
    // Me sigma: one fine cell per thread, its 12 products added in 4 steps
    // that never meet on an edge (every sum has its order)
#pragma unroll 1
    for (int c = tid; c < (M3 + NT - 1) / NT * NT; c += NT) {
      const int i = c % M, j = (c / M) % M, k = c / (M * M);
      double y[12];
      if (c < M3) {
        double nd[8], sg[12];
#pragma unroll
        for (int t = 0; t < 8; ++t) nd[t] = node(i + (t & 1), j + ((t >> 1) & 1), k + (t >> 2));
#pragma unroll
        for (int Ln = 0; Ln < 12; ++Ln) {
          const int a = kLnAx[Ln], p = a == 0 ? 1 : 0, q = a == 2 ? 1 : 2;
          const int lo = (kLnF1[Ln] << p) | (kLnF2[Ln] << q);
          const int di = (lo & 1), dj = (lo >> 1) & 1, dk = lo >> 2;
          sg[Ln] = (coarse(a, i + di, j + dj, k + dk) + (nd[lo | (1 << a)] - nd[lo])) * ih[a];
          y[Ln] = 0.0;
        }
        const double2* A = reinterpret_cast<const double2*>(g.ainv + ((size_t)cell * M3 + c) * 48);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const double qx = kGp[q & 1], qy = kGp[(q >> 1) & 1], qz = kGp[q >> 2];
          const double2 a01 = A[q * 3], a23 = A[q * 3 + 1], a45 = A[q * 3 + 2];
          double ev[3] = {0.0, 0.0, 0.0};
          double lw[12];
#pragma unroll
          for (int Ln = 0; Ln < 12; ++Ln) {
            const int a = kLnAx[Ln];
            const double u = a == 0 ? qy : qx, t = a == 2 ? qy : qz;
            lw[Ln] = (kLnF1[Ln] ? u : 1.0 - u) * (kLnF2[Ln] ? t : 1.0 - t);
            ev[a] = fma(lw[Ln], sg[Ln], ev[a]);
          }
          const double J[3] = {a01.x * ev[0] + a01.y * ev[1] + a23.x * ev[2],
                               a01.y * ev[0] + a23.y * ev[1] + a45.x * ev[2],
                               a23.x * ev[0] + a45.x * ev[1] + a45.y * ev[2]};
#pragma unroll
          for (int Ln = 0; Ln < 12; ++Ln) y[Ln] = fma(lw[Ln], J[kLnAx[Ln]], y[Ln]);
        }
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (c < M3) {
#pragma unroll
          for (int Ln = 0; Ln < 12; ++Ln) {
            if ((kLnF1[Ln] | (kLnF2[Ln] << 1)) != t) continue;
            const int a = kLnAx[Ln], p = a == 0 ? 1 : 0, q = a == 2 ? 1 : 2;
            const int lo = (kLnF1[Ln] << p) | (kLnF2[Ln] << q);
            E[a * S3 + ((k + (lo >> 2)) * S + j + ((lo >> 1) & 1)) * S + i + (lo & 1)] +=
                y[Ln] * (w8 * ih[a]);
          }
        }
        __syncthreads();
      }
    }
    // column n of the edge block in its energy form sigma_i . Me sigma_n =
    // N_i . Me sigma_n + phi_i . d0^T Me sigma_n: second order in the error of phi
    double acc[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) acc[t] = 0.0;
    for (int e = tid; e < NE; e += NT) {
      const int a = e / Q::NX;
      int r = e - a * Q::NX;
      const int nx = a == 0 ? M : S, ny = a == 1 ? M : S;
      const int i = r % nx;
      r /= nx;
      const int j = r % ny, k = r / ny;
      const double y = E[a * S3 + (k * S + j) * S + i] * (1.0 / M);
      const double t1 = (a == 0 ? j : i) * (1.0 / M), t2 = (a == 2 ? j : k) * (1.0 / M);
#pragma unroll
      for (int t = 0; t < 12; ++t)
        if (kLnAx[t] == a)
          acc[t] = fma(y, (kLnF1[t] ? t1 : 1.0 - t1) * (kLnF2[t] ? t2 : 1.0 - t2), acc[t]);
    }
    const double* ph = g.phi + (size_t)cell * 12 * M3;
    for (int c = tid; c < M3; c += NT) {
      const int i = c % M, j = (c / M) % M, k = c / (M * M);
      if (i == 0 || j == 0 || k == 0) continue;
      const double* p = E + (k * S + j) * S + i;
      const double y = (p[-1] - p[0]) + (p[S3 - S] - p[S3]) + (p[2 * S3 - S * S] - p[2 * S3]);
#pragma unroll
      for (int t = 0; t < 12; ++t) acc[t] = fma(ph[(size_t)t * M3 + c], y, acc[t]);
    }
    const double col = block_sums<Q::NW>(acc, red);
    if (tid < 12) Mc[tid * 18 + n] = col;
    transform<M, NT, EdgeToModes>(E, 3);
  } else {
    // d' = 1/D over its sum - 1/M^3: the divergence of the +1 faces less
    // that of the coarse function
    const double* W = g.W + (size_t)cell * (M3 + 1);
    const double sc = 1.0 / W[M3];
    for (int c = tid; c < M3; c += NT)
      E[((c / (M * M)) * S + (c / M) % M) * S + c % M] = fma(W[c], sc, -1.0 / M3);
    __syncthreads();
    transform<M, NT, CellToModes>(E, 1);
  }
  for (int c = tid; c < M3; c += NT) {
    const int kx = c % M, ky = (c / M) % M, kz = c / (M * M);
    const double kp[3] = {kap[kx], kap[ky], kap[kz]}, im[3] = {tim[0][kx], tim[1][ky], tim[2][kz]};
    // the transforms are not normalised: (2/M)^3 for both ways, half of it
    // for each constant mode
    const double scale = (kx ? 2.0 : 1.0) * (ky ? 2.0 : 1.0) * (kz ? 2.0 : 1.0) * (1.0 / M3);
    const double den =
        fma(kp[0] * kp[0], im[0], fma(kp[1] * kp[1], im[1], kp[2] * kp[2] * im[2]));
    double* p = E + (kz * S + ky) * S + kx;
    double u[3] = {0.0, 0.0, 0.0};
    if (c > 0) {
      if (n < 12) {
        const double gx = (ky && kz) ? p[0] : 0.0, gy = (kx && kz) ? p[S3] : 0.0,
                     gz = (kx && ky) ? p[2 * S3] : 0.0;
        const double ik = scale / (kp[0] * kp[0] + kp[1] * kp[1] + kp[2] * kp[2]);
        const double y[3] = {(kp[1] * gz - kp[2] * gy) * ik, (kp[2] * gx - kp[0] * gz) * ik,
                             (kp[0] * gy - kp[1] * gx) * ik};
        const double s = -(kp[0] * y[0] * im[0] + kp[1] * y[1] * im[1] + kp[2] * y[2] * im[2]) / den;
#pragma unroll
        for (int d = 0; d < 3; ++d) u[d] = fma(s, kp[d], y[d]) * im[d];
      } else {
        const double ph = p[0] * scale / den;
#pragma unroll
        for (int d = 0; d < 3; ++d) u[d] = kp[d] * ph * im[d];
      }
    }
    p[0] = u[0];
    p[S3] = u[1];
    p[2 * S3] = u[2];
  }
  __syncthreads();
  transform<M, NT, ModesToFace>(E, 3);
  // the faces of the basis (or of the 6 face bases, c_n +- u*)
  double acc[16];
#pragma unroll
  for (int t = 0; t < 16; ++t) acc[t] = 0.0;
  for (int f = tid; f < 3 * NF1; f += NT) {
    const int a = f / NF1;
    int r = f - a * NF1;
    const int nx = a == 0 ? S : M, ny = a == 1 ? S : M;
    const int i = r % nx;
    r /= nx;
    const int j = r % ny, k = r / ny;
    const int lev = a == 0 ? i : (a == 1 ? j : k);
    const double u = (lev > 0 && lev < M) ? E[a * S3 + (k * S + j) * S + i] : 0.0;
    if (n < 12) {
      X[(size_t)n * Q::N + NE + f] = u;
    } else {
      const double hi = lev * (1.0 / M), lo = 1.0 - hi;
#pragma unroll
      for (int b = 0; b < 6; ++b) {
        const double c = (b >> 1) == a ? ((b & 1) ? hi : lo) * (1.0 / (M * M)) : 0.0;
        X[(size_t)(12 + b) * Q::N + NE + f] = (b & 1) ? c + u : c - u;
        if ((b >> 1) == a) acc[b] = fma(u, c, acc[b]);  // (c_b, u*) over the face mass
      }
    }
  }
  if (n < 12) return;
  for (int e = tid; e < 6 * NE; e += NT) {
    const int b = e / NE;
    X[(size_t)(12 + b) * Q::N + e - b * NE] = 0.0;
  }
  // (c_b, f) and (u*, f)
  if (g.fq)
    for (int c = tid; c < M3; c += NT) {
      const int i = c % M, j = (c / M) % M, k = c / (M * M);
      const double* f = g.fq + ((size_t)cell * M3 + c) * 24;
      double m0[3] = {0.0, 0.0, 0.0}, m1[3] = {0.0, 0.0, 0.0};
#pragma unroll
      for (int q = 0; q < 8; ++q)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const double t = kGp[(q >> d) & 1], y = f[q * 3 + d];
          m0[d] = fma(1.0 - t, y, m0[d]);
          m1[d] = fma(t, y, m1[d]);
        }
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const int lev = d == 0 ? i : (d == 1 ? j : k);
        const double wd = w8 * ih[d == 0 ? 1 : 0] * ih[d == 2 ? 1 : 2];
        const double* p = E + d * S3 + (k * S + j) * S + i;
        const int up = d == 0 ? 1 : (d == 1 ? S : S * S);
        const double a = m0[d] * wd, b = m1[d] * wd;
        const double c0 = lev * (1.0 / M), c1 = (lev + 1) * (1.0 / M);
        acc[6 + 2 * d] += ((1.0 - c0) * a + (1.0 - c1) * b) * (1.0 / (M * M));
        acc[7 + 2 * d] += (c0 * a + c1 * b) * (1.0 / (M * M));
        acc[12] += (lev > 0 ? p[0] : 0.0) * a + (lev < M - 1 ? p[up] : 0.0) * b;
      }
    }
  const double sum = block_sums<Q::NW>(acc, red);
  if (tid < 16) tot[tid] = sum;
  __syncthreads();
  {
    for (int e = tid; e < 18 * 18; e += NT) {
      const int i = e / 18, j = e % 18;
      if (i < 12 && j < 12) continue;
      double val;
      if (i >= 12 && j >= 12) {
        // u_i d2^T D d2 u_j: both divergences are +-1 shared out by 1/D
        val = (((i ^ j) & 1) ? -1.0 : 1.0) / g.W[(size_t)cell * (M3 + 1) + M3];
      } else {
        // -(curl sigma_e, u_f) = -(curl N_e, c_f +- u*), curl N_e = sum of inc c_F
        const int ed = i < 12 ? i : j, fc = (i < 12 ? j : i) - 12;
        double s = 0.0;
#pragma unroll
        for (int F = 0; F < 6; ++F) {
          int inc = 0;
#pragma unroll
          for (int t = 0; t < 12; ++t) inc = t == ed ? seq_inc(F, t) : inc;
          const double big = H[F >> 1] / (H[(F >> 1) == 0 ? 1 : 0] * H[(F >> 1) == 2 ? 1 : 2]);
          double y = (F >> 1) == (fc >> 1) ? big * (F == fc ? 1.0 / 3.0 : 1.0 / 6.0) : 0.0;
          y += ((fc & 1) ? 1.0 : -1.0) * mf[F >> 1] * tot[F];
          s += inc * y;
        }
        val = i < 12 ? -s : s;
      }
      Mc[e] = val;
    }
  }
  if (tid < 18) {
    double s = 0.0;
#pragma unroll
    for (int b = 0; b < 6; ++b)
      if (tid == 12 + b) s = tot[6 + b] + ((b & 1) ? tot[12] : -tot[12]);
    g.b[(size_t)cell * 18 + tid] = s;
  }
}

// One wave per cell.
__global__ __launch_bounds__(256) void nrt_seq_status_kernel(NrtSeq g) {
  const int cell = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (cell >= g.n_cells || g.general[cell]) return;
  bool bad = false;
  for (int k = lane; k < 324; k += 64) bad |= !isfinite(g.Mat[(size_t)cell * 324 + k]);
  int state = 0;
  if (lane < 12) {
    const int* it = g.iters + ((size_t)cell * 12 + lane) * 2;
    state = it[1];
    if (g.its) g.its[(size_t)cell * 18 + lane] = it[0];
  } else if (lane < 18 && g.its) {
    g.its[(size_t)cell * 18 + lane] = 0;
  }
  const int st = (__any(bad) || __any(state == 3)) ? MSFEC_CELL_NONFINITE
                 : __any(state == 2)               ? MSFEC_CELL_NOT_SPD
                 : __any(state == 1)               ? MSFEC_CELL_NOT_CONVERGED
                                                   : MSFEC_CELL_OK;
  if (lane == 0) g.status[cell] = st;
}

#define SEQ_HIP(call)                  \
  do {                                 \
    const hipError_t e_ = (call);      \
    if (e_ != hipSuccess) return e_;   \
  } while (0)

template <int M>
hipError_t launch(int l, const NrtSeq& g, hipStream_t s, hipEvent_t* mid) {
  constexpr int M3 = M * M * M;
  hipLaunchKernelGGL(nrt_seq_weights_kernel<M>, dim3(g.n_cells),
                     dim3(M3 < 64 ? 64 : (M3 > 1024 ? 1024 : M3)), 0, s, g);
  SEQ_HIP(hipGetLastError());
  msfec_detail::Q1tRows rw{};
  rw.verts = g.verts;
  rw.a = g.ainv;
  rw.st = g.st;
  rw.rhs = g.rhs;
  rw.bad = g.general;
  rw.n_cells = g.n_cells;
  rw.nr = 12;
  rw.edge = true;
  SEQ_HIP(msfec_detail::q1t_rows(l, rw, s));
  if (mid) SEQ_HIP(hipEventRecord(mid[0], s));
  msfec_detail::Q1tCg cg{};
  cg.st = g.st;
  cg.rhs = g.rhs;
  cg.x = g.phi;
  cg.skip = g.general;
  cg.iters = g.iters;
  cg.n_cells = g.n_cells;
  cg.nr = 12;
  cg.direct = true;
  cg.max_iter = g.max_iter;
  cg.tol = g.rtol;
  SEQ_HIP(msfec_detail::q1t_solve(l, cg, s));
  if (mid) SEQ_HIP(hipEventRecord(mid[1], s));
  const size_t lds = (size_t)3 * Seq<M>::S3 * sizeof(double);
  if (lds > 48 * 1024)
    SEQ_HIP(hipFuncSetAttribute((const void*)nrt_seq_basis_kernel<M>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(nrt_seq_basis_kernel<M>, dim3((g.n_cells + 7) / 8 * 8 * 13), dim3(Seq<M>::NT), lds,
                     s, g);
  SEQ_HIP(hipGetLastError());
  hipLaunchKernelGGL(nrt_seq_status_kernel, dim3((g.n_cells + 3) / 4), dim3(256), 0, s, g);
  return hipGetLastError();
}

}  // namespace

namespace msfec_detail {

hipError_t nrt_seq(int l, const NrtSeq& g, hipStream_t s, hipEvent_t* mid) {
  switch (l) {
    case 1: return launch<2>(l, g, s, mid);
    case 2: return launch<4>(l, g, s, mid);
    case 3: return launch<8>(l, g, s, mid);
    default: return launch<16>(l, g, s, mid);
  }
}

}  // namespace msfec_detail
