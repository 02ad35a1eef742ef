// RT_DQ in three dimensions by projected conjugate gradients.
//
// The flux of basis n is the coarse Raviart-Thomas function c_n plus a
// divergence-free flux without normal trace, the one that minimises
// (sigma, A^-1 sigma).  Jacobi-PCG on a potential of that flux (the curl-curl
// system, msfec_nrt.hip) needs iterations in proportion to M.  On the fluxes
// themselves, with the orthogonal projection onto the divergence-free ones in
// the plain face mass Mf as the preconditioner, the iterations depend on the
// contrast of A^-1 alone:
//   z = projection of Mf^-1 r,  p = z + beta p,  q = M_A p,  r -= alpha q.
// On a box the projection is a scaling of the modes of sines and cosines
// (msfec_trig.hpp): z^ = Mf^-1 (r^ - kappa s), kappa . z^ = 0, at
// the cost of 36 LDS passes over a component.
// 64 cells of 16^3 with the coefficients of the reference example: 49
// iterations and 3.3 ms, against 180 and 30.4 ms on the curl-curl system with
// its vectors in memory.
//
// Cells whose A^-1 is not positive definite or not finite, or varies by more than
// kMaxContrast, are flagged and left to the curl-curl solver.
#include "msfec_rt3_proj.hpp"

#include "msfec.h"
#include "msfec_cell.hpp"
#include "msfec_trig.hpp"
#include "msfec_wave.hpp"

namespace {

using msfec_detail::Rt3Proj;
using namespace msfec_cell;
using msfec_wave::block_sums;
using msfec_wave::buffer_f64;
using msfec_wave::from_left;
using msfec_wave::from_right;
using msfec_wave::wave_sum;
using msfec_wave::waves_sum;
using namespace msfec_trig;

// Largest ratio that is solved here of the bounds of the eigenvalues of A^-1 in a
// cell: the largest trace over the smallest 4 det / trace^2, for isotropic
// tensors 6.75 times their contrast.  Iterations grow with its square root, those
// of the curl-curl solver hardly.  Batches on one side alone, 8 cells with
// lognormal A^-1, here and there: 16^3 at a ratio of 1e4 4.2 and 12 ms, 3e5 12
// and 17, 1e7 40 and 22; 8^3 at 1e5 1.0 and 4.8 ms, 1e6 2.5 and 6.8, 2e7 6.1 and
// 7.2; 4^3 at 1e7 0.6 and 1.7 ms.  They cross at about 2e6 (16^3) and 5e7 (8^3).
// The line is lower because a batch with cells on both sides of it runs both
// solvers, one after the other: 8 cells of 16^3 with ratios of 6e4 to 2e5 take
// 16.7 ms, 13.3 with the curl-curl solver alone; at 1e6 the first half of such a
// batch would add 13 ms to the second.
constexpr double kMaxContrast = 1e5;

template <int M>
struct Cfg {
  static constexpr int M2 = M * M, M3 = M2 * M, S = M + 1, S3 = S * S * S, NF1 = M2 * S;
  // solver: NS segments of LZ cells per column in z
  static constexpr int LZ = M >= 16 ? 8 : (M >= 8 ? 2 : 1), NS = M / LZ;
  static constexpr int USE = M2 * NS, NT = USE < 64 ? 64 : USE, NW = NT / 64;
  // masses and element matrices: one fine cell per thread
  static constexpr int CT = M3 < 64 ? 64 : (M3 > 256 ? 256 : M3), BLOCKS = M3 > 256 ? M3 / 256 : 1;
};

constexpr int pair_of(int F, int G) {
  const int hi = F > G ? F : G, lo = F > G ? G : F;
  return hi * (hi + 1) / 2 + lo;
}

__device__ __forceinline__ void sizes(const double* v, int m, double* H, double* h) {
  H[0] = v[3] - v[0];
  H[1] = v[7] - v[1];
  H[2] = v[14] - v[2];
  for (int d = 0; d < 3; ++d) h[d] = H[d] / m;
}

// (psi_F, A^-1 psi_G) of every fine cell by its 8 Gauss points, two entries
// side by side (16-byte loads in the solver), and bounds of the eigenvalues of
// A^-1: the trace from above, 4 det / trace^2 from below.
template <int M>
__global__ __launch_bounds__(Cfg<M>::CT) void rt3_proj_mass_kernel(Rt3Proj g) {
  typedef Cfg<M> C;
  __shared__ double red[C::CT / 64][2];
  const int cell = blockIdx.x / C::BLOCKS, blk = blockIdx.x % C::BLOCKS, tid = threadIdx.x;
  const int c = blk * C::CT + tid;
  double H[3], h[3];
  sizes(g.verts + (size_t)cell * 24, M, H, h);
  const double ih[3] = {1.0 / (h[1] * h[2]), 1.0 / (h[0] * h[2]), 1.0 / (h[0] * h[1])};
  const double w = h[0] * h[1] * h[2] * 0.125;
  double top = 0.0, low = 1e300;
  if (c < C::M3) {
    const double2* A = reinterpret_cast<const double2*>(g.ainv + ((size_t)cell * C::M3 + c) * 48);
    double m[22];
#pragma unroll
    for (int e = 0; e < 22; ++e) m[e] = 0.0;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const double2 a01 = A[q * 3], a23 = A[q * 3 + 1], a45 = A[q * 3 + 2];
      const double t[6] = {a01.x, a01.y, a23.x, a23.y, a45.x, a45.y};
      const double m2 = t[0] * t[3] - t[1] * t[1];
      const double det = t[0] * (t[3] * t[5] - t[4] * t[4]) - t[1] * (t[1] * t[5] - t[4] * t[2]) +
                         t[2] * (t[1] * t[4] - t[3] * t[2]);
      const double tr = t[0] + t[3] + t[5];
      if (t[0] > 0.0 && m2 > 0.0 && det > 0.0 && isfinite(det) && isfinite(tr)) {
        top = fmax(top, tr);
        low = fmin(low, 4.0 * det / (tr * tr));
      } else {
        low = -1.0;
      }
      double v[6];
#pragma unroll
      for (int F = 0; F < 6; ++F) {
        const double X = kGp[(q >> (F >> 1)) & 1];
        v[F] = ((F & 1) ? X : 1.0 - X) * ih[F >> 1];
      }
#pragma unroll
      for (int F = 0; F < 6; ++F)
#pragma unroll
        for (int G = 0; G <= F; ++G) {
          const int lo = G >> 1, hi = F >> 1;
          const int comp = lo == 0 ? hi : (lo == 1 ? 2 + hi : 5);
          m[pair_of(F, G)] = fma(v[F] * v[G], t[comp], m[pair_of(F, G)]);
        }
    }
    double2* out = reinterpret_cast<double2*>(g.MF) + (size_t)cell * 11 * C::M3;
#pragma unroll
    for (int e = 0; e < 11; ++e) out[e * C::M3 + c] = make_double2(m[2 * e] * w, m[2 * e + 1] * w);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    top = fmax(top, __shfl_xor(top, off));
    low = fmin(low, __shfl_xor(low, off));
  }
  if ((tid & 63) == 0) {
    red[tid >> 6][0] = top;
    red[tid >> 6][1] = low;
  }
  __syncthreads();
  if (tid == 0) {
#pragma unroll
    for (int i = 1; i < C::CT / 64; ++i) {
      top = fmax(top, red[i][0]);
      low = fmin(low, red[i][1]);
    }
    g.bound[((size_t)cell * C::BLOCKS + blk) * 2] = top;
    g.bound[((size_t)cell * C::BLOCKS + blk) * 2 + 1] = low;
  }
}

typedef unsigned mass_v4 __attribute__((ext_vector_type(4)));

// One face basis of one coarse cell per workgroup; a thread owns LZ fine cells
// of a column in z and the lower face of each of them in every direction (r and p
// of these in registers, as far as they go: 336 bytes a lane of the kernel for
// M = 16 are in scratch; x in the output buffer).  M_A p cell by cell: the upper faces of a cell
// belong to its neighbours, whose p come, and to whom the products go, by lane
// shifts along x, through LDS along y and in the column along z.  Then r goes
// to the lattice E in LDS, which the transforms turn into z.
template <int M>
__global__ __launch_bounds__(Cfg<M>::NT) void rt3_proj_cg_kernel(Rt3Proj g) {
  typedef Cfg<M> C;
  constexpr int S = C::S, S3 = C::S3, M2 = C::M2, M3 = C::M3, LZ = C::LZ, NT = C::NT;
  extern __shared__ double lds[];
  double* E = lds;                 // 3 x S^3
  double* U = E + 3 * S3;          // M^3: products for the faces above in y
  double* V = U + M3;              // NS x M^2: for the face above a segment
  double* red = V + C::NS * M2;    // 2 x NW
  double* kap = red + 2 * C::NW;   // M
  double* tim = kap + M;           // 3 x M
  const int slot = blockIdx.x >> 3, cell = (slot / 6) * 8 + (blockIdx.x & 7), nb = slot % 6;
  if (cell >= g.n_cells) return;
  double top = 0.0, low = 1e300;
  for (int i = 0; i < C::BLOCKS; ++i) {
    top = fmax(top, g.bound[((size_t)cell * C::BLOCKS + i) * 2]);
    low = fmin(low, g.bound[((size_t)cell * C::BLOCKS + i) * 2 + 1]);
  }
  const bool general = !(low > 0.0) || !(top <= kMaxContrast * low);
  const int tid = threadIdx.x;
  if (nb == 0 && tid == 0) g.general[cell] = general;
  if (general) return;
  // (M = 2: the threads beyond the columns follow the first and write nothing)
  const bool on = C::USE >= 64 || tid < C::USE;
  const int own = on ? tid : 0;
  const int col = own % M2, seg = own / M2, i = col % M, j = col / M, k0 = seg * LZ;
  double H[3], h[3];
  sizes(g.verts + (size_t)cell * 24, M, H, h);
  // the mass of the projection in units of A^-1 (a power of two: no rounding), so that
  // p is of the size of the flux and p . M_A p linear in A^-1; with the plain mass it is
  // cubic and falls below the range of a double for A^-1 = 1e-100
  const double unit = ldexp(1.0, ilogb(top));
  const double mf[3] = {unit * (h[0] / (h[1] * h[2])), unit * (h[1] / (h[0] * h[2])),
                        unit * (h[2] / (h[0] * h[1]))};
  for (int e = tid; e < 3 * S3; e += NT) E[e] = 0.0;
  if (tid < M) {
    kap[tid] = 2.0 * sinpi(tid * (0.5 / M));
    const double t = fma(cospi(tid * (1.0 / M)), 1.0 / 3.0, 2.0 / 3.0);
#pragma unroll
    for (int d = 0; d < 3; ++d) tim[d * M + tid] = 1.0 / (mf[d] * t);
  }
  const int at0 = (k0 * S + j) * S + i;  // lattice point of the first cell
  const __amdgpu_buffer_rsrc_t rsrc = msfec_wave::buffer_of(g.MF + (size_t)cell * 22 * M3, 22 * M3 * 8);
  const int lane0 = (k0 * M2 + col) * 16;
  auto pair = [&](int e, int t) {
    const mass_v4 m = __builtin_amdgcn_raw_buffer_load_b128(rsrc, lane0, (e * M3 + t * M2) * 16, 0);
    return make_double2(__hiloint2double((int)m.y, (int)m.x), __hiloint2double((int)m.w, (int)m.z));
  };
  // coarse flux through the face of axis d at level lev
  auto coarse = [&](int d, int lev) {
    const double t = lev * (1.0 / M);
    return d == (nb >> 1) ? ((nb & 1) ? t : 1.0 - t) * (1.0 / M2) : 0.0;
  };
  double r[3][LZ], p[3][LZ];
  // x waits at the place of its faces in g.S: it is touched once an iteration,
  // and its 3 LZ values would not fit the registers (240 of them in scratch at
  // M = 16; a pass of 64 cells took 3.53 ms with it there and 3.20 ms so)
  double* out = g.S + ((size_t)cell * 6 + nb) * 3 * C::NF1;
  const __amdgpu_buffer_rsrc_t xb = msfec_wave::buffer_of(out, 3 * C::NF1 * 8);
  const int face[3] = {((k0 * M + j) * S + i) * 8, (C::NF1 + (k0 * S + j) * M + i) * 8,
                       (2 * C::NF1 + (k0 * M + j) * M + i) * 8};
  auto step = [](int d) { return (d == 2 ? M2 : M * S) * 8; };  // to the next cell of the column
  // q = M_A p on the lower faces: x and z parts in the lattice (z of the first
  // cell, whose place the segment below reads, in qz), y part in qy without
  // what U brings, z of the first cell without what V brings; returns
  // p . M_A p.  With `first`, of the coarse function instead of p.
  double qy[LZ], qz = 0.0;
  auto apply = [&](bool first) __attribute__((always_inline)) {
    double quad = 0.0, carry = 0.0;
    double2 m[11];
#pragma unroll
    for (int e = 0; e < 11; ++e) m[e] = pair(e, 0);
#pragma unroll
    for (int t = 0; t < LZ; ++t) {
      double c[6], z[6];
      const int at = at0 + t * S * S;
      if (first) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          c[s] = coarse(0, i + s);
          c[2 + s] = coarse(1, j + s);
          c[4 + s] = coarse(2, k0 + t + s);
        }
      } else {
        c[0] = p[0][t];
        c[1] = from_right(p[0][t]);
        c[2] = p[1][t];
        c[3] = E[S3 + at + S];
        c[4] = p[2][t];
        if (t + 1 < LZ) c[5] = p[2][t + 1 < LZ ? t + 1 : t];
        else c[5] = E[2 * S3 + at + S * S];
      }
#pragma unroll
      for (int F = 0; F < 6; ++F) z[F] = 0.0;
      // every pair of entries is read for the next cell as soon as it is used
#pragma unroll
      for (int e = 0; e < 11; ++e) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int en = 2 * e + u;
          const int F = en < 1 ? 0 : en < 3 ? 1 : en < 6 ? 2 : en < 10 ? 3 : en < 15 ? 4 : 5;
          const int G = en - F * (F + 1) / 2;
          if (en > 20) continue;
          const double a = u ? m[e].y : m[e].x;
          z[F] = fma(a, c[G], z[F]);
          if (F != G) z[G] = fma(a, c[F], z[G]);
        }
        if (t + 1 < LZ) m[e] = pair(e, t + 1);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int F = 0; F < 6; ++F) quad = fma(c[F], z[F], quad);
      const double qx = z[0] + from_left(z[1]);
      if (on) {
        E[at] = qx;
        U[(k0 + t) * M2 + col] = z[3];
        if (t > 0) E[2 * S3 + at] = z[4] + carry;
      }
      qy[t] = z[2];
      if (t == 0) qz = z[4];
      carry = z[5];
    }
    if (on) V[seg * M2 + col] = carry;
    return on ? quad : 0.0;
  };
  // q of the faces of cell t, after a barrier
  auto product = [&](int t, double* q) __attribute__((always_inline)) {
    const int at = at0 + t * S * S;
    q[0] = E[at];
    q[1] = qy[t] + (j > 0 ? U[(k0 + t) * M2 + col - M] : 0.0);
    q[2] = t > 0 ? E[2 * S3 + at] : qz + (seg > 0 ? V[(seg - 1) * M2 + col] : 0.0);
  };
  // r in the lattice -> z in the lattice; returns r . z from the modes (a sum
  // of squares, where the plain product would cancel)
  auto project = [&]() __attribute__((always_inline)) {
    transform<M, NT, FaceToModes>(E, 3);
    double rz = 0.0;
    for (int c = tid; c < M3; c += NT) {
      const int kx = c % M, ky = (c / M) % M, kz = c / M2;
      const double kp[3] = {kap[kx], kap[ky], kap[kz]};
      const double im[3] = {tim[kx], tim[M + ky], tim[2 * M + kz]};
      const double scale = (kx ? 2.0 : 1.0) * (ky ? 2.0 : 1.0) * (kz ? 2.0 : 1.0) * (1.0 / M3);
      double* e = E + (kz * S + ky) * S + kx;
      double w[3] = {kx ? e[0] : 0.0, ky ? e[S3] : 0.0, kz ? e[2 * S3] : 0.0};
      double num = 0.0, den = 0.0;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        num = fma(kp[d] * im[d], w[d], num);
        den = fma(kp[d] * im[d], kp[d], den);
      }
      const double s = c > 0 ? num / den : 0.0;
      double sq = 0.0;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        w[d] = fma(-s, kp[d], w[d]);
        const double z = w[d] * im[d];
        sq = fma(w[d], z, sq);
        e[d * S3] = c > 0 ? z * scale : 0.0;
      }
      rz = fma(sq, c > 0 ? scale : 0.0, rz);
    }
    rz = wave_sum(rz);
    if ((tid & 63) == 0) red[C::NW + (tid >> 6)] = rz;
    __syncthreads();
    transform<M, NT, ModesToFace>(E, 3);
    return waves_sum<C::NW>(red + C::NW);
  };
  __syncthreads();  // the lattice is zeroed: its points belong to other threads below
  apply(true);
  __syncthreads();
#pragma unroll
  for (int t = 0; t < LZ; ++t) {
    double q[3];
    product(t, q);
#pragma unroll
    for (int d = 0; d < 3; ++d) r[d][t] = -q[d];
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < LZ; ++t)
#pragma unroll
    for (int d = 0; d < 3; ++d)
      if (on) E[d * S3 + at0 + t * S * S] = r[d][t];
  __syncthreads();
  double rz = project();
  // the first r is Mf z: what the projection dropped of it (most of M_A c_n
  // where A^-1 is nearly constant) would only carry rounding along
#pragma unroll
  for (int t = 0; t < LZ; ++t) {
    const int lev[3] = {i, j, k0 + t};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const int next = d == 0 ? 1 : (d == 1 ? S : S * S);
      const double* e = E + d * S3 + at0 + t * S * S;
      if (on) buffer_f64(xb, face[d], t * step(d), 0.0);
      p[d][t] = e[0];
      r[d][t] = lev[d] > 0 ? mf[d] * fma(2.0 / 3.0, e[0], (e[-next] + e[next]) * (1.0 / 6.0)) : 0.0;
    }
  }
  // half of rtol: with rtol itself the fluxes were off by up to 1.7 times what
  // |r| <= rtol |b| leaves on the curl-curl system (8^3 cells of the reference
  // example's tensor 2.8e-14 and 1.7e-14; 1.4e-14 so), for one iteration in 40.
  // Not below 1e-15 unless rtol is: rounding need not let it go on.
  const double tol = fmax(0.5 * g.rtol, fmin(g.rtol, 1e-15));
  const double stop = tol * tol * rz;
  int it = 0, flag = MSFEC_CELL_OK;
  __syncthreads();
  while (rz > stop) {
    if (it >= g.max_iter) {
      flag = MSFEC_CELL_NOT_CONVERGED;
      break;
    }
#pragma unroll
    for (int t = 0; t < LZ; ++t)
      if (on) E[S3 + at0 + t * S * S] = p[1][t];
    if (on) E[2 * S3 + at0] = p[2][0];
    __syncthreads();
    double pq = wave_sum(apply(false));
    if ((tid & 63) == 0) red[tid >> 6] = pq;
    __syncthreads();
    pq = waves_sum<C::NW>(red);
    if (!(pq > 0.0)) {
      flag = isfinite(pq) ? MSFEC_CELL_NOT_SPD : MSFEC_CELL_NONFINITE;
      break;
    }
    const double alpha = rz / pq;
    double x[2][3];
#pragma unroll
    for (int d = 0; d < 3; ++d) x[0][d] = buffer_f64(xb, face[d], 0);
#pragma unroll
    for (int t = 0; t < LZ; ++t) {
      if (t + 1 < LZ)
#pragma unroll
        for (int d = 0; d < 3; ++d) x[(t + 1) & 1][d] = buffer_f64(xb, face[d], (t + 1) * step(d));
      __builtin_amdgcn_sched_barrier(0);
      double q[3];
      product(t, q);
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        if (on) buffer_f64(xb, face[d], t * step(d), fma(alpha, p[d][t], x[t & 1][d]));
        r[d][t] = fma(-alpha, q[d], r[d][t]);
        if (on) E[d * S3 + at0 + t * S * S] = r[d][t];
      }
    }
    __syncthreads();
    const double rz1 = project();
    const double beta = rz1 / rz;
    rz = rz1;
#pragma unroll
    for (int t = 0; t < LZ; ++t)
#pragma unroll
      for (int d = 0; d < 3; ++d) p[d][t] = fma(beta, p[d][t], E[d * S3 + at0 + t * S * S]);
    ++it;
  }
  if (!isfinite(rz)) flag = MSFEC_CELL_NONFINITE;
  // The transforms leave rounding of the size of the largest flux in every p, and
  // x gathers its divergence, which the energy in M notices to first order: the
  // flux of that divergence is taken out again.  The balance of a fine cell is
  // then off by 1.6 eps of the largest flux at most (without, 50 at a contrast
  // of 1e3, 500 at 1e5) and M by 1e-15 (without, 4e-15 and 2e-14), for 80 us of
  // 3.2 ms (64 cells of 16^3).
  __syncthreads();
#pragma unroll
  for (int t = 0; t < LZ; ++t) {
    const int lev[3] = {i, j, k0 + t};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double x = buffer_f64(xb, face[d], t * step(d));
      if (on) E[d * S3 + at0 + t * S * S] = lev[d] > 0 ? x : 0.0;
    }
  }
  __syncthreads();
  double div[LZ];
#pragma unroll
  for (int t = 0; t < LZ; ++t) {
    const double* e = E + at0 + t * S * S;
    div[t] = (e[1] - e[0]) + (e[S3 + S] - e[S3]) + (e[2 * S3 + S * S] - e[2 * S3]);
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < LZ; ++t)
    if (on) E[at0 + t * S * S] = div[t];
  __syncthreads();
  transform<M, NT, CellToModes>(E, 1);
  for (int c = tid; c < M3; c += NT) {
    const int kx = c % M, ky = (c / M) % M, kz = c / M2;
    const double kp[3] = {kap[kx], kap[ky], kap[kz]};
    const double im[3] = {tim[kx], tim[M + ky], tim[2 * M + kz]};
    const double scale = (kx ? 2.0 : 1.0) * (ky ? 2.0 : 1.0) * (kz ? 2.0 : 1.0) * (1.0 / M3);
    double* e = E + (kz * S + ky) * S + kx;
    const double den = fma(kp[0] * kp[0], im[0], fma(kp[1] * kp[1], im[1], kp[2] * kp[2] * im[2]));
    const double s = c > 0 ? e[0] * scale / den : 0.0;
#pragma unroll
    for (int d = 0; d < 3; ++d) e[d * S3] = kp[d] * s * im[d];
  }
  __syncthreads();
  transform<M, NT, ModesToFace>(E, 3);
#pragma unroll
  for (int t = 0; t < LZ; ++t) {
    if (!on) break;
    const int k = k0 + t, lev[3] = {i, j, k};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double x = buffer_f64(xb, face[d], t * step(d)) - E[d * S3 + at0 + t * S * S];
      buffer_f64(xb, face[d], t * step(d), coarse(d, lev[d]) + (lev[d] > 0 ? x : 0.0));
    }
    if (i == M - 1) out[(k * M + j) * S + M] = coarse(0, M);
    if (j == M - 1) out[C::NF1 + (k * S + M) * M + i] = coarse(1, M);
    if (k == M - 1) out[2 * C::NF1 + (M * M + j) * M + i] = coarse(2, M);
  }
  if (tid == 0) {
    g.its[(size_t)cell * 6 + nb] = it;
    g.flg[(size_t)cell * 6 + nb] = flag;
  }
}

// Partial sums of the element matrix (rt_dq_basis.cc:822-914, with u = 1), one
// fine cell per thread: sigma_i^T M_A sigma_j, the net outflows and the load.
template <int M>
__global__ __launch_bounds__(Cfg<M>::CT) void rt3_proj_element_kernel(Rt3Proj g) {
  typedef Cfg<M> C;
  constexpr int S = C::S;
  __shared__ double red[C::CT / 64][16];
  const int cell = blockIdx.x / C::BLOCKS, blk = blockIdx.x % C::BLOCKS, tid = threadIdx.x;
  if (g.general[cell]) return;
  const int c = blk * C::CT + tid, i = c % M, j = (c / M) % M, k = c / C::M2;
  double acc[32];
#pragma unroll
  for (int t = 0; t < 32; ++t) acc[t] = 0.0;
  if (c < C::M3) {
    const double2* mp = reinterpret_cast<const double2*>(g.MF) + (size_t)cell * 11 * C::M3 + c;
    double m[22], s[6][6];
#pragma unroll
    for (int e = 0; e < 11; ++e) {
      const double2 t = mp[e * C::M3];
      m[2 * e] = t.x;
      m[2 * e + 1] = t.y;
    }
    const int face[6] = {(k * M + j) * S + i,
                         (k * M + j) * S + i + 1,
                         C::NF1 + (k * S + j) * M + i,
                         C::NF1 + (k * S + j + 1) * M + i,
                         2 * C::NF1 + (k * M + j) * M + i,
                         2 * C::NF1 + ((k + 1) * M + j) * M + i};
#pragma unroll
    for (int n = 0; n < 6; ++n)
#pragma unroll
      for (int F = 0; F < 6; ++F) s[n][F] = g.S[((size_t)cell * 6 + n) * 3 * C::NF1 + face[F]];
    int e = 0;
#pragma unroll
    for (int n = 0; n < 6; ++n) {
      double ms[6];
#pragma unroll
      for (int F = 0; F < 6; ++F) {
        ms[F] = 0.0;
#pragma unroll
        for (int G = 0; G < 6; ++G) ms[F] = fma(m[pair_of(F, G)], s[n][G], ms[F]);
      }
#pragma unroll
      for (int y = 0; y <= n; ++y, ++e)
#pragma unroll
        for (int F = 0; F < 6; ++F) acc[e] = fma(ms[F], s[y][F], acc[e]);
      acc[21 + n] = (s[n][1] - s[n][0]) + (s[n][3] - s[n][2]) + (s[n][5] - s[n][4]);
    }
    if (g.fq) {
      double H[3], h[3];
      sizes(g.verts + (size_t)cell * 24, M, H, h);
      const double2* f = reinterpret_cast<const double2*>(g.fq + ((size_t)cell * C::M3 + c) * 8);
      double t = 0.0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const double2 y = f[q];
        t += y.x;
        t += y.y;
      }
      acc[27] = t * h[0] * h[1] * h[2] * 0.125;
    }
  }
#pragma unroll
  for (int t = 0; t < 32; t += 16) {
    const double y = block_sums<C::CT / 64>(acc + t, red);
    if (tid < 16) g.part[((size_t)cell * C::BLOCKS + blk) * 32 + t + tid] = y;
  }
}

// One wave per cell: the sums, and the status of every cell (the flagged ones
// from the general solver's element matrix).
__global__ __launch_bounds__(256) void rt3_proj_finish_kernel(Rt3Proj g, int blocks) {
  const int cell = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (cell >= g.n_cells) return;
  double* Mc = g.Mat + (size_t)cell * 49;
  double* bc = g.b + (size_t)cell * 7;
  bool bad = false;
  if (g.general[cell]) {
    if (lane < 49) bad = !isfinite(Mc[lane]);
  } else if (lane < 28) {
    double s = 0.0;
    for (int t = 0; t < blocks; ++t) s += g.part[((size_t)cell * blocks + t) * 32 + lane];
    if (lane < 21) {
      const int n = lane < 1 ? 0 : lane < 3 ? 1 : lane < 6 ? 2 : lane < 10 ? 3 : lane < 15 ? 4 : 5;
      const int y = lane - n * (n + 1) / 2;
      Mc[n * 7 + y] = Mc[y * 7 + n] = s;
      bad = !isfinite(s);
    } else if (lane < 27) {
      Mc[(lane - 21) * 7 + 6] = -s;  // -(div sigma_i, 1)
      Mc[6 * 7 + lane - 21] = s;     // (1, div sigma_i)
      bc[lane - 21] = 0.0;
      bad = !isfinite(s);
    } else {
      Mc[6 * 7 + 6] = 0.0;           // (R u, v) with R = 0
      bc[6] = s;
    }
  }
  bad = __any(bad);
  if (lane == 0) {
    int st = MSFEC_CELL_OK;
    for (int n = 0; n < 6; ++n) {
      const int f = g.flg[(size_t)cell * 6 + n];
      if (f != MSFEC_CELL_OK && st == MSFEC_CELL_OK) st = f;
    }
    g.status[cell] = st == MSFEC_CELL_OK && bad ? MSFEC_CELL_NONFINITE : st;
  }
}

template <int M>
hipError_t masses(const Rt3Proj& g, hipStream_t s) {
  hipLaunchKernelGGL(rt3_proj_mass_kernel<M>, dim3(g.n_cells * Cfg<M>::BLOCKS), dim3(Cfg<M>::CT), 0, s, g);
  return hipGetLastError();
}

template <int M>
hipError_t solve(const Rt3Proj& g, hipStream_t s) {
  typedef Cfg<M> C;
  const size_t lds = (3 * C::S3 + C::M3 + C::NS * C::M2 + 2 * C::NW + 4 * M) * sizeof(double);
  if (lds > 48 * 1024) {
    const hipError_t e = hipFuncSetAttribute((const void*)rt3_proj_cg_kernel<M>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(rt3_proj_cg_kernel<M>, dim3((g.n_cells + 7) / 8 * 8 * 6), dim3(C::NT), lds, s, g);
  return hipGetLastError();
}

template <int M>
hipError_t element(const Rt3Proj& g, hipStream_t s) {
  hipLaunchKernelGGL(rt3_proj_element_kernel<M>, dim3(g.n_cells * Cfg<M>::BLOCKS), dim3(Cfg<M>::CT), 0, s, g);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(rt3_proj_finish_kernel, dim3((g.n_cells + 3) / 4), dim3(256), 0, s, g, Cfg<M>::BLOCKS);
  return hipGetLastError();
}

}  // namespace

namespace msfec_detail {

int rt3_proj_blocks(int l) { return l < 4 ? (l == 3 ? Cfg<8>::BLOCKS : 1) : Cfg<16>::BLOCKS; }

#define RT3_PROJ(fn)                                            \
  hipError_t rt3_proj_##fn(int l, const Rt3Proj& g, hipStream_t s) { \
    switch (l) {                                                \
      case 1: return fn<2>(g, s);                               \
      case 2: return fn<4>(g, s);                               \
      case 3: return fn<8>(g, s);                               \
      default: return fn<16>(g, s);                             \
    }                                                           \
  }
RT3_PROJ(masses)
RT3_PROJ(solve)
RT3_PROJ(element)

}  // namespace msfec_detail
