// Q1 problems with a tensor coefficient per Gauss point on one refined box
// (see msfec_q1t.hpp): assembly of the interior rows and their solution.
#include "msfec_q1t.hpp"

#include <algorithm>

namespace {

using msfec_detail::Q1tCg;
using msfec_detail::Q1tRows;

constexpr double kGp[2] = {0.21132486540518711775, 0.78867513459481288225};

// deal.II's line order on the unit cube: axis, and the fixed values of the
// two other coordinates (lower axis first)
constexpr int kLnAx[12] = {1, 1, 0, 0, 1, 1, 0, 0, 2, 2, 2, 2};
constexpr int kLnF1[12] = {0, 1, 0, 1, 0, 1, 0, 1, 0, 1, 0, 1};
constexpr int kLnF2[12] = {0, 0, 0, 0, 1, 1, 1, 1, 0, 0, 1, 1};

// The nodes of one workgroup of the assembly: whole rows in x, TY x TZ of
// them.  The tensors of the cells around them are staged in LDS two Gauss
// points at a time (42 KB for M = 16, three workgroups per CU).
template <int M>
struct RowTile {
  static constexpr int TY = M >= 16 ? 4 : M, TZ = M >= 8 ? 4 : M;
  static constexpr int NT = M * TY * TZ < 64 ? 64 : M * TY * TZ;
  static constexpr int CELLS = M * (TY + 1) * (TZ + 1);
  static constexpr int TILES = (M / TY) * (M / TZ);
};

// One thread per interior node: its 27 matrix entries and the 12 right-hand
// sides, summed over its 8 cells and their 8 Gauss points.  Every cell's
// products are formed by each of its nodes: 3.7 kFMA a node, against 130
// doubles a node through memory for element matrices formed once.
template <int M>
__global__ __launch_bounds__(RowTile<M>::NT, 2) void q1t_rows_kernel(Q1tRows g) {
  typedef RowTile<M> T;
  constexpr int M3 = M * M * M;
  __shared__ double A[T::CELLS * 13];
  const int cell = blockIdx.x / T::TILES, tile = blockIdx.x % T::TILES, tid = threadIdx.x;
  const int y0 = (tile % (M / T::TY)) * T::TY, z0 = (tile / (M / T::TY)) * T::TZ;
  const double* v = g.verts + (size_t)cell * 24;
  const double H[3] = {v[3] - v[0], v[7] - v[1], v[14] - v[2]};
  const double ih[3] = {M / H[0], M / H[1], M / H[2]};
  const double w = H[0] * H[1] * H[2] / M3 * 0.125;
  const double* src = g.a + (size_t)cell * M3 * 48;
  const int ni = tid % M, nj = y0 + (tid / M) % T::TY, nk = z0 + tid / (M * T::TY);
  const bool own = tid < M * T::TY * T::TZ;
  const bool act = own && ni > 0 && nj > 0 && nk > 0;
  double st[27], rh[12];
#pragma unroll
  for (int e = 0; e < 27; ++e) st[e] = 0.0;
#pragma unroll
  for (int n = 0; n < 12; ++n) rh[n] = 0.0;
  bool bad = false;
#pragma unroll 1
  for (int qp = 0; qp < 4; ++qp) {
    __syncthreads();
    for (int idx = tid; idx < T::CELLS * 12; idx += T::NT) {
      const int c = idx / 12, e = idx - c * 12;
      const int cx = c % M, cy = y0 - 1 + (c / M) % (T::TY + 1), cz = z0 - 1 + c / (M * (T::TY + 1));
      A[c * 13 + e] = (cy < 0 || cz < 0) ? 1.0 : src[((size_t)((cz * M + cy) * M + cx) * 8 + 2 * qp) * 6 + e];
    }
    __syncthreads();
    for (int idx = tid; idx < T::CELLS * 2; idx += T::NT) {
      const int c = idx >> 1;
      if ((c / M) % (T::TY + 1) + y0 == 0 || c / (M * (T::TY + 1)) + z0 == 0) continue;
      const double* t = A + c * 13 + (idx & 1) * 6;
      const double m2 = t[0] * t[3] - t[1] * t[1];
      const double m3 = t[0] * (t[3] * t[5] - t[4] * t[4]) - t[1] * (t[1] * t[5] - t[4] * t[2]) +
                        t[2] * (t[1] * t[4] - t[3] * t[2]);
      if (!(t[0] > 0.0 && m2 > 0.0 && m3 > 0.0 && isfinite(m3))) bad = true;
    }
    if (!act) continue;
    const double Xy = kGp[0] + (qp & 1) * (kGp[1] - kGp[0]), Xz = kGp[0] + (qp >> 1) * (kGp[1] - kGp[0]);
    const double ly[2] = {1.0 - Xy, Xy}, lz[2] = {1.0 - Xz, Xz};
#pragma unroll 1
    for (int qq = 0; qq < 2; ++qq) {
      const double Xx = kGp[0] + qq * (kGp[1] - kGp[0]);
      const double lx[2] = {1.0 - Xx, Xx};
#pragma unroll
      for (int al = 0; al < 8; ++al) {
        asm volatile("" ::: "memory");  // one cell's tensor in registers at a time
        const int ax = al & 1, ay = (al >> 1) & 1, az = al >> 2;
        const int cx = ni - ax, cy = nj - ay, cz = nk - az;
        const double* t = A + (((cz - z0 + 1) * (T::TY + 1) + cy - y0 + 1) * M + cx) * 13 + qq * 6;
        const double gx = (ax ? w : -w) * ih[0] * ly[ay] * lz[az];
        const double gy = (ay ? w : -w) * ih[1] * lx[ax] * lz[az];
        const double gz = (az ? w : -w) * ih[2] * lx[ax] * ly[ay];
        const double ux = t[0] * gx + t[1] * gy + t[2] * gz;
        const double uy = t[1] * gx + t[3] * gy + t[4] * gz;
        const double uz = t[2] * gx + t[4] * gy + t[5] * gz;
        const double vx = ux * ih[0], vy = uy * ih[1], vz = uz * ih[2];
#pragma unroll
        for (int b = 0; b < 8; ++b) {
          const int bx = b & 1, by = (b >> 1) & 1, bz = b >> 2;
          const int e = ((bz - az + 1) * 3 + by - ay + 1) * 3 + bx - ax + 1;
          double s = (bx ? vx : -vx) * (ly[by] * lz[bz]);
          s += (by ? vy : -vy) * (lx[bx] * lz[bz]);
          s += (bz ? vz : -vz) * (lx[bx] * ly[by]);
          st[e] += s;
        }
        // N_n = l_f1 l_f2 e_axis / H_axis at the point, in the coarse coordinates
        double Cx = (cx + lx[1]) / M, Cy = (cy + ly[1]) / M, Cz = (cz + lz[1]) / M;
        asm volatile("" : "+v"(Cx), "+v"(Cy), "+v"(Cz));  // not formed for all cells ahead
        const double Lx[2] = {1.0 - Cx, Cx}, Ly[2] = {1.0 - Cy, Cy}, Lz[2] = {1.0 - Cz, Cz};
#pragma unroll
        for (int n = 0; n < 12; ++n) {
          const int f1 = kLnF1[n], f2 = kLnF2[n];
          if (kLnAx[n] == 0) rh[n] -= ux * (Ly[f1] * Lz[f2]);
          else if (kLnAx[n] == 1) rh[n] -= uy * (Lx[f1] * Lz[f2]);
          else rh[n] -= uz * (Lx[f1] * Ly[f2]);
        }
      }
    }
  }
  if (bad) g.bad[cell] = 1;
  if (!own) return;
  const size_t node = (size_t)(nk * M + nj) * M + ni;
#pragma unroll
  for (int e = 0; e < 27; ++e) g.st[((size_t)cell * 27 + e) * M3 + node] = st[e];
#pragma unroll
  for (int n = 0; n < 12; ++n)
    g.rhs[((size_t)cell * 12 + n) * M3 + node] = rh[n] / H[kLnAx[n]];
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// Jacobi-preconditioned conjugate gradients, NB right-hand sides of one
// coarse cell per workgroup in step, LZ nodes of a column in z per thread.
// The vectors x, r and p stay in registers and p in LDS as well (a flat copy
// padded with zeros, so that all 26 neighbours are constant offsets); an
// iteration reads the 27 entries of every row once for the NB vectors, and
// each plane of 9 neighbour values serves the three nodes above, in and
// below it.  The bound is the L2 rate of the rows, 885 KB an iteration at
// M = 16: 14 us an iteration with 96 workgroups.  Workgroups of one coarse
// cell share an XCD (block index mod 8).
template <int M, int LZ, int NB>
__global__ __launch_bounds__(M * M * M / LZ) void q1t_cg_kernel(Q1tCg g) {
  constexpr int M2 = M * M, M3 = M2 * M, NT = M3 / LZ, PAD = M2 + M + 1;
  constexpr int NW = (NT + 63) / 64;
  __shared__ double P[NB][M3 + 2 * PAD];
  __shared__ double redA[NW][NB], redB[NW][2 * NB];
  const int groups = (g.nr + NB - 1) / NB;
  const int slot = blockIdx.x >> 3, cell = (slot / groups) * 8 + (blockIdx.x & 7);
  const int n0 = (slot % groups) * NB;
  if (cell >= g.n_cells || (g.skip && g.skip[cell])) return;
  const int tid = threadIdx.x, col = tid % M2, k0 = (tid / M2) * LZ, wv = tid >> 6;
  const double* st = g.st + (size_t)cell * 27 * M3;
  const int row0 = k0 * M2 + col;
  for (int i = tid; i < NB * (M3 + 2 * PAD); i += NT) P[0][i] = 0.0;
  const bool inner = col % M > 0 && col / M > 0;
  double x[NB][LZ], r[NB][LZ], p[NB][LZ], dinv[LZ];
  double rz[NB], rr[NB], stop[NB];
  int it[NB], state[NB];
  bool live[NB];
#pragma unroll
  for (int z = 0; z < LZ; ++z)
    dinv[z] = (inner && k0 + z > 0) ? 1.0 / st[(size_t)13 * M3 + row0 + z * M2] : 0.0;
#pragma unroll
  for (int n = 0; n < NB; ++n) {
    double a = 0.0, b = 0.0;
#pragma unroll
    for (int z = 0; z < LZ; ++z) {
      x[n][z] = 0.0;
      r[n][z] = n0 + n < g.nr ? g.rhs[((size_t)cell * g.nr + n0 + n) * M3 + row0 + z * M2] : 0.0;
      p[n][z] = dinv[z] * r[n][z];
      a = fma(r[n][z], p[n][z], a);
      b = fma(r[n][z], r[n][z], b);
    }
    a = wave_sum(a);
    b = wave_sum(b);
    if ((tid & 63) == 0) {
      redB[wv][2 * n] = a;
      redB[wv][2 * n + 1] = b;
    }
  }
  __syncthreads();  // also: P is zeroed
  bool any = false;
#pragma unroll
  for (int n = 0; n < NB; ++n) {
    rz[n] = rr[n] = 0.0;
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      rz[n] += redB[i][2 * n];
      rr[n] += redB[i][2 * n + 1];
    }
    stop[n] = g.tol * g.tol * rr[n];
    it[n] = 0;
    state[n] = 0;
    live[n] = rr[n] > stop[n];
    any = any || live[n];
#pragma unroll
    for (int z = 0; z < LZ; ++z) P[n][PAD + row0 + z * M2] = p[n][z];
  }
  while (any) {
    __syncthreads();  // p of every thread is in LDS
    // entries are read from a uniform base plus one 32-bit offset, opaque so
    // that no per-lane 64-bit addresses are formed ahead of the loop
    const char* stb = reinterpret_cast<const char*>(st);
    unsigned ro = (unsigned)row0 * 8u;
    asm volatile("" : "+v"(ro));
    double q[NB][LZ];
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
      for (int z = 0; z < LZ; ++z) q[n][z] = 0.0;
#pragma unroll
    for (int pz = -1; pz <= LZ; ++pz) {
      // one plane's entries in flight at a time: more would spill
      asm volatile("" ::: "memory");
      double v[NB][9];
#pragma unroll
      for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int t = 0; t < 9; ++t)
          v[n][t] = P[n][PAD + row0 + pz * M2 + (t / 3 - 1) * M + t % 3 - 1];
#pragma unroll
      for (int dz = -1; dz <= 1; ++dz) {
        const int z = pz - dz;
        if (z < 0 || z >= LZ) continue;
        const unsigned at0 = ro + z * M2 * 8;
#pragma unroll
        for (int t = 0; t < 9; ++t) {
          const double at = *reinterpret_cast<const double*>(stb + ((dz + 1) * 9 + t) * M3 * 8 + at0);
#pragma unroll
          for (int n = 0; n < NB; ++n) q[n][z] = fma(at, v[n][t], q[n][z]);
        }
      }
    }
#pragma unroll
    for (int n = 0; n < NB; ++n) {
      double s = 0.0;
#pragma unroll
      for (int z = 0; z < LZ; ++z) s = fma(p[n][z], q[n][z], s);
      s = wave_sum(s);
      if ((tid & 63) == 0) redA[wv][n] = s;
    }
    __syncthreads();  // also: every thread is done reading p
#pragma unroll
    for (int n = 0; n < NB; ++n) {
      double pq = 0.0;
#pragma unroll
      for (int i = 0; i < NW; ++i) pq += redA[i][n];
      if (live[n] && !(pq > 0.0)) {
        state[n] = 2;
        live[n] = false;
      }
      const double alpha = live[n] ? rz[n] / pq : 0.0;
      double a = 0.0, b = 0.0;
#pragma unroll
      for (int z = 0; z < LZ; ++z) {
        x[n][z] = fma(alpha, p[n][z], x[n][z]);
        r[n][z] = fma(-alpha, q[n][z], r[n][z]);
        a = fma(r[n][z], dinv[z] * r[n][z], a);
        b = fma(r[n][z], r[n][z], b);
      }
      a = wave_sum(a);
      b = wave_sum(b);
      if ((tid & 63) == 0) {
        redB[wv][2 * n] = a;
        redB[wv][2 * n + 1] = b;
      }
    }
    __syncthreads();
    any = false;
#pragma unroll
    for (int n = 0; n < NB; ++n) {
      double rz1 = 0.0, rr1 = 0.0;
#pragma unroll
      for (int i = 0; i < NW; ++i) {
        rz1 += redB[i][2 * n];
        rr1 += redB[i][2 * n + 1];
      }
      if (!live[n]) continue;
      const double beta = rz1 / rz[n];
      rz[n] = rz1;
      rr[n] = rr1;
      ++it[n];
#pragma unroll
      for (int z = 0; z < LZ; ++z) {
        p[n][z] = fma(beta, p[n][z], dinv[z] * r[n][z]);
        P[n][PAD + row0 + z * M2] = p[n][z];
      }
      if (!(rr1 > stop[n])) live[n] = false;
      else if (it[n] >= g.max_iter) {
        state[n] = 1;
        live[n] = false;
      }
      any = any || live[n];
    }
  }
#pragma unroll
  for (int n = 0; n < NB; ++n) {
    if (n0 + n >= g.nr) continue;
#pragma unroll
    for (int z = 0; z < LZ; ++z)
      g.x[((size_t)cell * g.nr + n0 + n) * M3 + row0 + z * M2] = x[n][z];
    if (tid == 0) {
      int* o = g.iters + ((size_t)cell * g.nr + n0 + n) * 2;
      o[0] = it[n];
      o[1] = isfinite(rr[n]) ? state[n] : 3;
    }
  }
}

// l <= 2: one wave per coarse cell eliminates the (M - 1)^3 interior unknowns
// with its right-hand sides (Gauss-Jordan without pivoting on the positive
// definite rows), one column of [K | rhs] per lane in registers: the
// multipliers of a step are one lane's column, read by v_readlane.
template <int M>
__global__ __launch_bounds__(64) void q1t_direct_kernel(Q1tCg g) {
  constexpr int M3 = M * M * M, ni = M - 1, n = ni * ni * ni;
  const int cell = blockIdx.x, lane = threadIdx.x;
  if (g.skip && g.skip[cell]) return;
  const double* st = g.st + (size_t)cell * 27 * M3;
  auto flat = [](int r) { return ((r / (ni * ni) + 1) * M + (r / ni) % ni + 1) * M + r % ni + 1; };
  const int cx = lane % ni, cy = (lane / ni) % ni, cz = lane / (ni * ni);
  double a[n];
#pragma unroll
  for (int i = 0; i < n; ++i) {
    const int dx = cx - i % ni, dy = cy - (i / ni) % ni, dz = cz - i / (ni * ni);
    a[i] = 0.0;
    if (lane < n) {
      if (dx >= -1 && dx <= 1 && dy >= -1 && dy <= 1 && dz >= -1 && dz <= 1)
        a[i] = st[(size_t)(((dz + 1) * 3 + dy + 1) * 3 + dx + 1) * M3 + flat(i)];
    } else if (lane - n < g.nr) {
      a[i] = g.rhs[((size_t)cell * g.nr + lane - n) * M3 + flat(i)];
    }
  }
  auto bcast = [](double v, int l) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
    return __hiloint2double(hi, lo);
  };
  bool ok = true, fin = true;
#pragma unroll
  for (int k = 0; k < n; ++k) {
    const double piv = bcast(a[k], k);
    ok = ok && piv > 0.0;
    fin = fin && isfinite(piv);
    const double t = a[k] * (1.0 / piv);
#pragma unroll
    for (int i = 0; i < n; ++i)
      if (i != k) a[i] = fma(-bcast(a[i], k), t, a[i]);
    a[k] = t;
  }
  if (lane >= n && lane - n < g.nr) {
    double* x = g.x + ((size_t)cell * g.nr + lane - n) * M3;
    for (int i = 0; i < M3; ++i)
      if (i % M == 0 || (i / M) % M == 0 || i < M * M) x[i] = 0.0;
#pragma unroll
    for (int i = 0; i < n; ++i) x[flat(i)] = a[i];
    int* o = g.iters + ((size_t)cell * g.nr + lane - n) * 2;
    o[0] = 0;
    o[1] = !fin ? 3 : (ok ? 0 : 2);
  }
}

template <int M>
hipError_t rows(const Q1tRows& g, hipStream_t s) {
  hipLaunchKernelGGL(q1t_rows_kernel<M>, dim3(g.n_cells * RowTile<M>::TILES), dim3(RowTile<M>::NT), 0,
                     s, g);
  return hipGetLastError();
}

template <int M, int LZ, int NB>
hipError_t cg(const Q1tCg& g, hipStream_t s) {
  const int blocks = (g.n_cells + 7) / 8 * 8 * ((g.nr + NB - 1) / NB);
  hipLaunchKernelGGL((q1t_cg_kernel<M, LZ, NB>), dim3(blocks), dim3(M * M * M / LZ), 0, s, g);
  return hipGetLastError();
}

}  // namespace

namespace msfec_detail {

hipError_t q1t_rows(int l, const Q1tRows& g, hipStream_t s) {
  switch (l) {
    case 1: return rows<2>(g, s);
    case 2: return rows<4>(g, s);
    case 3: return rows<8>(g, s);
    default: return rows<16>(g, s);
  }
}

hipError_t q1t_solve(int l, const Q1tCg& g, hipStream_t s) {
  if (l == 1) hipLaunchKernelGGL(q1t_direct_kernel<2>, dim3(g.n_cells), dim3(64), 0, s, g);
  else if (l == 2) hipLaunchKernelGGL(q1t_direct_kernel<4>, dim3(g.n_cells), dim3(64), 0, s, g);
  else if (l == 3) return cg<8, 2, 1>(g, s);
  else return cg<16, 4, 1>(g, s);
  return hipGetLastError();
}

}  // namespace msfec_detail
