// Q1 problems with a tensor coefficient per Gauss point on one refined box
// (see msfec_q1t.hpp): assembly of the interior rows and their solution.
#include "msfec_q1t.hpp"

#include "msfec.h"
#include "msfec_cell.hpp"
#include "msfec_wave.hpp"

#include <algorithm>

namespace {

using msfec_detail::Q1tBasis;
using msfec_detail::Q1tCg;
using msfec_detail::Q1tRows;
using namespace msfec_cell;
using msfec_wave::block_sums;
using msfec_wave::buffer_f64;
using msfec_wave::buffer_of;
using msfec_wave::from_left;
using msfec_wave::from_right;
using msfec_wave::wave_sum;


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

// One thread per interior node: its 27 matrix entries and the right-hand
// sides, summed over its 8 cells and their 8 Gauss points.  Every cell's
// products are formed by each of its nodes: 3.7 kFMA a node, against 130
// doubles a node through memory for element matrices formed once.  95 us for
// 64 cells at M = 16 (8 right-hand sides), bound by the FP64 rate.
template <int M, bool Edge>
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
  const double* src = g.a + (size_t)cell * M3 * (!Edge && g.scalar ? 1 : 48);
  const int ni = tid % M, nj = y0 + (tid / M) % T::TY, nk = z0 + tid / (M * T::TY);
  const bool own = tid < M * T::TY * T::TZ;
  const bool act = own && ni > 0 && nj > 0 && nk > 0;
  constexpr int NR = Edge ? 12 : 8;
  double st[27], rh[NR];
#pragma unroll
  for (int e = 0; e < 27; ++e) st[e] = 0.0;
#pragma unroll
  for (int n = 0; n < NR; ++n) rh[n] = 0.0;
  bool bad = false;
#pragma unroll 1
  for (int qp = 0; qp < 4; ++qp) {
    __syncthreads();
    for (int idx = tid; idx < T::CELLS * 12; idx += T::NT) {
      const int c = idx / 12, e = idx - c * 12;
      const int cx = c % M, cy = y0 - 1 + (c / M) % (T::TY + 1), cz = z0 - 1 + c / (M * (T::TY + 1));
      const int z = (cz * M + cy) * M + cx;
      double val = 1.0;
      if (cy >= 0 && cz >= 0) {
        if (!Edge && g.scalar) val = (e % 6 == 0 || e % 6 == 3 || e % 6 == 5) ? src[z] : 0.0;
        else val = src[((size_t)z * 8 + 2 * qp) * 6 + e];
      }
      A[c * 13 + e] = val;
    }
    __syncthreads();
    if constexpr (Edge) for (int idx = tid; idx < T::CELLS * 2; idx += T::NT) {
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
        if constexpr (!Edge) continue;
        // N_n = l_f1 l_f2 e_axis / H_axis at the point, in the coarse coordinates
        double Cx = (cx + lx[1]) / M, Cy = (cy + ly[1]) / M, Cz = (cz + lz[1]) / M;
        asm volatile("" : "+v"(Cx), "+v"(Cy), "+v"(Cz));  // not formed for all cells ahead
        const double Lx[2] = {1.0 - Cx, Cx}, Ly[2] = {1.0 - Cy, Cy}, Lz[2] = {1.0 - Cz, Cz};
#pragma unroll
        for (int n = 0; n < (Edge ? 12 : 0); ++n) {
          const int f1 = kLnF1[n], f2 = kLnF2[n];
          if (kLnAx[n] == 0) rh[n] -= ux * (Ly[f1] * Lz[f2]);
          else if (kLnAx[n] == 1) rh[n] -= uy * (Lx[f1] * Lz[f2]);
          else rh[n] -= uz * (Lx[f1] * Ly[f2]);
        }
      }
    }
  }
  if (Edge && bad) g.bad[cell] = 1;
  if (!own) return;
  const size_t node = (size_t)(nk * M + nj) * M + ni;
  if constexpr (Edge) {
#pragma unroll
    for (int n = 0; n < 12; ++n) rh[n] /= H[kLnAx[n]];
  } else if (act) {
    if (g.reac || g.reac0 != 0.0) {
      // the mass on a box: 1/3 for the node with itself, 1/6 with a neighbour, per direction
#pragma unroll
      for (int al = 0; al < 8; ++al) {
        const int ax = al & 1, ay = (al >> 1) & 1, az = al >> 2;
        const double r =
            (g.reac ? g.reac[(size_t)cell * M3 + ((nk - az) * M + nj - ay) * M + ni - ax] : g.reac0) *
            w * (8.0 / 216.0);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
          const int bx = b & 1, by = (b >> 1) & 1, bz = b >> 2;
          st[((bz - az + 1) * 3 + by - ay + 1) * 3 + bx - ax + 1] +=
              r * ((bx == ax ? 2.0 : 1.0) * (by == ay ? 2.0 : 1.0) * (bz == az ? 2.0 : 1.0));
        }
      }
    }
  }
  if (act && (ni == 1 || nj == 1 || nk == 1 || ni == M - 1 || nj == M - 1 || nk == M - 1)) {
    // the entries to boundary nodes go to the right-hand sides and are dropped
#pragma unroll
    for (int e = 0; e < 27; ++e) {
      const int mx = ni + e % 3 - 1, my = nj + (e / 3) % 3 - 1, mz = nk + e / 9 - 1;
      if (!(mx == 0 || my == 0 || mz == 0 || mx == M || my == M || mz == M)) continue;
      if constexpr (!Edge) {
        const double X = mx * (1.0 / M), Y = my * (1.0 / M), Z = mz * (1.0 / M);
#pragma unroll
        for (int n = 0; n < 8; ++n)
          rh[n] -= st[e] * ((n & 1 ? X : 1.0 - X) * (n & 2 ? Y : 1.0 - Y) * (n & 4 ? Z : 1.0 - Z));
      }
      st[e] = 0.0;
    }
  }
#pragma unroll
  for (int e = 0; e < 14; ++e) g.st[((size_t)cell * 15 + e) * M3 + node] = st[e];
  g.st[((size_t)cell * 15 + 14) * M3 + node] = act ? 1.0 / st[13] : 0.0;
#pragma unroll
  for (int n = 0; n < NR; ++n)
    if (n < g.nr) g.rhs[((size_t)cell * g.nr + n) * M3 + node] = rh[n];
}

// Jacobi-preconditioned conjugate gradients, one right-hand side of one
// coarse cell per workgroup, LZ nodes of a column in z per thread.  x, r and p
// stay in registers; p is in LDS as well, flat and padded with zeros, so that
// every neighbour is a constant offset.
//
// An iteration reads the 14 entries of every row (the diagonal and the lower
// neighbours) once: entry e of node n serves row n with p of n + e and row
// n + e with p of n.  The second product goes to its row by lane shifts along
// x, through LDS along y, and stays in the column along z.  Reading all 27
// entries of every row instead was bound by the L2 (885 KB an iteration and
// workgroup at M = 16, 14.6 us), and 8 cells of rows an XCD then exceed its
// L2 (64 cells x 7 bases: 2.4 ms with one vector per workgroup, 8.5 ms with
// two sharing the rows, which keeps all 8 cells in use at once).  Here 9.7 us
// an iteration: 1.41 ms for those, 0.68 ms for 8 cells x 12 potentials.
// Workgroups of one coarse cell share an XCD (block index mod 8).
template <int M, int LZ>
__global__ __launch_bounds__(M * M * M / LZ < 64 ? 64 : M * M * M / LZ) void q1t_cg_kernel(Q1tCg g) {
  constexpr int M2 = M * M, M3 = M2 * M, NT = M3 / LZ < 64 ? 64 : M3 / LZ, PAD = M2 + M + 1;
  constexpr int NW = NT / 64, NS = M / LZ;
  __shared__ double P[M3 + 2 * PAD];
  // products on their way to the rows y - 1 and y + 1 (the latter shifted by
  // M), and to the last plane of the segment of columns below
  __shared__ double UM[M3 + M], UP[M3 + M], B0[NS * M2], BM[NS * M2 + M], BP[NS * M2 + M];
  __shared__ double redA[NW], redB[NW][2];
  const int slot = blockIdx.x >> 3, cell = (slot / g.nr) * 8 + (blockIdx.x & 7), n = slot % g.nr;
  if (cell >= g.n_cells || (g.skip && g.skip[cell])) return;
  // (M = 2: the threads beyond the nodes repeat node 0, where all is zero)
  const int tid = threadIdx.x, own = tid < M3 / LZ ? tid : 0;
  const int col = own % M2, seg = own / M2, k0 = seg * LZ, wv = tid >> 6;
  const int row0 = k0 * M2 + col;
  const double* st = g.st + (size_t)cell * 15 * M3;
  const __amdgpu_buffer_rsrc_t rsrc =
      buffer_of(st, 15 * M3 * 8);
  for (int i = tid; i < M3 + 2 * PAD; i += NT) P[i] = 0.0;
  for (int i = tid; i < M3 + M; i += NT) UM[i] = UP[i] = 0.0;
  for (int i = tid; i < NS * M2 + M; i += NT) BM[i] = BP[i] = 0.0;
  double x[LZ], r[LZ], p[LZ];
  double rz = 0.0, rr = 0.0;
#pragma unroll
  for (int z = 0; z < LZ; ++z) {
    x[z] = 0.0;
    r[z] = g.rhs[((size_t)cell * g.nr + n) * M3 + row0 + z * M2];
    p[z] = buffer_f64(rsrc, row0 * 8, (14 * M3 + z * M2) * 8) * r[z];
    rz = fma(r[z], p[z], rz);
    rr = fma(r[z], r[z], rr);
  }
  rz = wave_sum(rz);
  rr = wave_sum(rr);
  if ((tid & 63) == 0) {
    redB[wv][0] = rz;
    redB[wv][1] = rr;
  }
  __syncthreads();  // also: the buffers are zeroed
  rz = rr = 0.0;
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    rz += redB[i][0];
    rr += redB[i][1];
  }
#pragma unroll
  for (int z = 0; z < LZ; ++z) P[PAD + row0 + z * M2] = p[z];
  const double stop = g.tol * g.tol * rr;
  int it = 0, state = 0;
  while (rr > stop) {
    if (it >= g.max_iter) {
      state = 1;
      break;
    }
    __syncthreads();  // p of every thread is in LDS
    double q[LZ], low = 0.0, pq = 0.0;
#pragma unroll
    for (int z = 0; z < LZ; ++z) q[z] = 0.0;
    // the entries to the plane below (9) and in the plane (5) of one node in
    // turn, three groups in flight; left alone the scheduler waits for every
    // load by itself
    double at[3][9], v[9], toM = 0.0;
    auto fetch = [&](int gr) {
#pragma unroll
      for (int t = 0; t < (gr & 1 ? 5 : 9); ++t)
        at[gr % 3][t] = buffer_f64(rsrc, row0 * 8, (((gr & 1 ? 9 : 0) + t) * M3 + (gr >> 1) * M2) * 8);
    };
    fetch(0);
    fetch(1);
#pragma unroll
    for (int gr = 0; gr < 2 * LZ; ++gr) {
      const int z = gr >> 1;
      const double* a = at[gr % 3];
      if (gr + 2 < 2 * LZ) fetch(gr + 2);
      const int at0 = PAD + row0 + (gr & 1 ? z : z - 1) * M2;
#pragma unroll
      for (int t = 0; t < (gr & 1 ? 4 : 9); ++t) v[t] = P[at0 + (t / 3 - 1) * M + t % 3 - 1];
      __builtin_amdgcn_sched_barrier(0);
      if ((gr & 1) == 0) {
        // lower half of the row: the plane below
        low = 0.0;
#pragma unroll
        for (int t = 0; t < 9; ++t) low = fma(a[t], v[t], low);
        const double cm = fma(a[1], p[z], from_right(a[0] * p[z]) + from_left(a[2] * p[z]));
        const double c0 = fma(a[4], p[z], from_right(a[3] * p[z]) + from_left(a[5] * p[z]));
        const double cp = fma(a[7], p[z], from_right(a[6] * p[z]) + from_left(a[8] * p[z]));
        if (z == 0) {
          B0[seg * M2 + col] = c0;
          BM[seg * M2 + col] = cm;
          BP[seg * M2 + col + M] = cp;
        } else {
          q[z - 1] += c0;
          UM[row0 + (z - 1) * M2] = toM + cm;
          UP[row0 + (z - 1) * M2 + M] = cp;
        }
      } else {
#pragma unroll
        for (int t = 0; t < 4; ++t) low = fma(a[t], v[t], low);
        const double d = a[4] * p[z];
        pq = fma(p[z], fma(2.0, low, d), pq);
        toM = fma(a[1], p[z], from_right(a[0] * p[z]) + from_left(a[2] * p[z]));
        q[z] += low + d + from_right(a[3] * p[z]);
        if (z == LZ - 1) UM[row0 + z * M2] = toM;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    pq = wave_sum(pq);
    if ((tid & 63) == 0) redA[wv] = pq;
    __syncthreads();  // products exchanged; every thread is done reading p
    pq = 0.0;
#pragma unroll
    for (int i = 0; i < NW; ++i) pq += redA[i];
    if (!(pq > 0.0)) {
      state = 2;
      break;
    }
#pragma unroll
    for (int z = 0; z < LZ; ++z) {
      q[z] += UM[row0 + z * M2 + M];
      if (z < LZ - 1) q[z] += UP[row0 + z * M2];
    }
    if (seg < NS - 1)
      q[LZ - 1] += B0[(seg + 1) * M2 + col] + BM[(seg + 1) * M2 + col + M] + BP[(seg + 1) * M2 + col];
    const double alpha = rz / pq;
    double rz1 = 0.0, dv[LZ];
    rr = 0.0;
#pragma unroll
    for (int z = 0; z < LZ; ++z) dv[z] = buffer_f64(rsrc, row0 * 8, (14 * M3 + z * M2) * 8);
#pragma unroll
    for (int z = 0; z < LZ; ++z) {
      x[z] = fma(alpha, p[z], x[z]);
      r[z] = fma(-alpha, q[z], r[z]);
      dv[z] *= r[z];
      rz1 = fma(r[z], dv[z], rz1);
      rr = fma(r[z], r[z], rr);
    }
    rz1 = wave_sum(rz1);
    rr = wave_sum(rr);
    if ((tid & 63) == 0) {
      redB[wv][0] = rz1;
      redB[wv][1] = rr;
    }
    __syncthreads();
    rz1 = rr = 0.0;
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      rz1 += redB[i][0];
      rr += redB[i][1];
    }
    const double beta = rz1 / rz;
    rz = rz1;
#pragma unroll
    for (int z = 0; z < LZ; ++z) {
      p[z] = fma(beta, p[z], dv[z]);
      P[PAD + row0 + z * M2] = p[z];
    }
    ++it;
  }
#pragma unroll
  for (int z = 0; z < LZ; ++z) g.x[((size_t)cell * g.nr + n) * M3 + row0 + z * M2] = x[z];
  if (tid == 0) {
    int* o = g.iters + ((size_t)cell * g.nr + n) * 2;
    o[0] = it;
    o[1] = isfinite(rr) ? state : 3;
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
  const double* st = g.st + (size_t)cell * 15 * M3;
  auto flat = [](int r) { return ((r / (ni * ni) + 1) * M + (r / ni) % ni + 1) * M + r % ni + 1; };
  const int cx = lane % ni, cy = (lane / ni) % ni, cz = lane / (ni * ni);
  double a[n];
#pragma unroll
  for (int i = 0; i < n; ++i) {
    const int dx = cx - i % ni, dy = cy - (i / ni) % ni, dz = cz - i / (ni * ni);
    a[i] = 0.0;
    if (lane < n) {
      if (dx >= -1 && dx <= 1 && dy >= -1 && dy <= 1 && dz >= -1 && dz <= 1)
        {
          const int e = ((dz + 1) * 3 + dy + 1) * 3 + dx + 1;  // column lane seen from row i
          a[i] = e < 14 ? st[(size_t)e * M3 + flat(i)] : st[(size_t)(26 - e) * M3 + flat(lane)];
        }
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

// Psi of a slab of fine cells and its part of the element matrix and load: one
// fine cell per thread, the energy psi_i . K psi_j by quadrature from the 8
// bases at its 8 nodes (second order in the error of the interior values).
// The 64 nodal values and 44 sums of a thread need one wave per SIMD.
template <int M>
struct Slab {
  static constexpr int L = M >= 16 ? 2 : (M >= 8 ? 4 : M);  // layers of cells
  static constexpr int COUNT = M / L;
  static constexpr int NT = M * M * L < 64 ? 64 : (M * M * L > 256 ? 256 : M * M * L);
};

template <int M>
__global__ __launch_bounds__(Slab<M>::NT) void q1t_basis_kernel(Q1tBasis g) {
  typedef Slab<M> B;
  constexpr int M2 = M * M, M3 = M2 * M, S = M + 1, S3 = S * S * S, NT = B::NT, NW = NT / 64;
  __shared__ double red[NW][16];
  const int cell = blockIdx.x / B::COUNT, slab = blockIdx.x % B::COUNT, tid = threadIdx.x;
  const int z0 = slab * B::L;
  const double* v = g.verts + (size_t)cell * 24;
  const double H[3] = {v[3] - v[0], v[7] - v[1], v[14] - v[2]};
  const double ih[3] = {M / H[0], M / H[1], M / H[2]};
  const double w = H[0] * H[1] * H[2] / M3 * 0.125;
  const double* x = g.x + (size_t)cell * g.nr * M3;
  auto values = [&](int i, int j, int k, double* p) {
    const bool in = i > 0 && j > 0 && k > 0 && i < M && j < M && k < M;
    if (in) {
      const double* y = x + (k * M + j) * M + i;
      double s = 0.0;
#pragma unroll
      for (int n = 0; n < 7; ++n) {
        p[n] = y[(size_t)n * M3];
        s += p[n];
      }
      p[7] = g.nr == 8 ? y[(size_t)7 * M3] : 1.0 - s;
    } else {
      const double X = i * (1.0 / M), Y = j * (1.0 / M), Z = k * (1.0 / M);
#pragma unroll
      for (int n = 0; n < 8; ++n)
        p[n] = (n & 1 ? X : 1.0 - X) * (n & 2 ? Y : 1.0 - Y) * (n & 4 ? Z : 1.0 - Z);
    }
  };
  const int planes = slab == B::COUNT - 1 ? B::L + 1 : B::L;
  for (int n = tid; n < planes * S * S; n += NT) {
    double p[8];
    values(n % S, (n / S) % S, z0 + n / (S * S), p);
#pragma unroll
    for (int k = 0; k < 8; ++k) g.Psi[((size_t)cell * 8 + k) * S3 + (size_t)z0 * S * S + n] = p[k];
  }
  double acc[48];
#pragma unroll
  for (int t = 0; t < 48; ++t) acc[t] = 0.0;
  const bool reac = g.reac || g.reac0 != 0.0;
#pragma unroll 1
  for (int c = tid; c < B::L * M2; c += NT) {
    const int i = c % M, j = (c / M) % M, k = z0 + c / M2;
    const size_t z = (size_t)cell * M3 + (size_t)k * M2 + j * M + i;
    double p[8][8];  // node, basis
#pragma unroll
    for (int t = 0; t < 8; ++t) values(i + (t & 1), j + ((t >> 1) & 1), k + (t >> 2), p[t]);
    const double rc = (g.reac ? g.reac[z] : g.reac0) * w;
#pragma unroll 1
    for (int q = 0; q < 8; ++q) {
      const double qx = q & 1 ? kGp[1] : kGp[0], qy = q & 2 ? kGp[1] : kGp[0], qz = q & 4 ? kGp[1] : kGp[0];
      double t[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
      if (g.scalar) {
        t[0] = t[3] = t[5] = g.a[z] * w;
      } else {
#pragma unroll
        for (int e = 0; e < 6; ++e) t[e] = g.a[(z * 8 + q) * 6 + e] * w;
      }
      const double fq = (g.f ? g.f[z * g.per_point + (g.per_point == 8 ? q : 0)] : g.f0) * w;
      const double lx[2] = {1.0 - qx, qx}, ly[2] = {1.0 - qy, qy}, lz[2] = {1.0 - qz, qz};
      double gx[8], gy[8], gz[8], pv[8];
#pragma unroll
      for (int n = 0; n < 8; ++n) {
        double sx = 0.0, sy = 0.0, sz = 0.0, sv = 0.0;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const int u = b & 1, y = b >> 1;
          sx = fma(ly[u] * lz[y], p[2 * u + 4 * y + 1][n] - p[2 * u + 4 * y][n], sx);
          sy = fma(lx[u] * lz[y], p[u + 4 * y + 2][n] - p[u + 4 * y][n], sy);
          sz = fma(lx[u] * ly[y], p[u + 2 * y + 4][n] - p[u + 2 * y][n], sz);
          sv = fma(lx[u] * ly[y], fma(qz, p[u + 2 * y + 4][n] - p[u + 2 * y][n], p[u + 2 * y][n]), sv);
        }
        gx[n] = sx * ih[0];
        gy[n] = sy * ih[1];
        gz[n] = sz * ih[2];
        pv[n] = sv;
        acc[36 + n] = fma(fq, sv, acc[36 + n]);
      }
      int e = 0;
#pragma unroll
      for (int n = 0; n < 8; ++n) {
        const double ux = t[0] * gx[n] + t[1] * gy[n] + t[2] * gz[n];
        const double uy = t[1] * gx[n] + t[3] * gy[n] + t[4] * gz[n];
        const double uz = t[2] * gx[n] + t[4] * gy[n] + t[5] * gz[n];
#pragma unroll
        for (int y = 0; y <= n; ++y, ++e)
          acc[e] = fma(ux, gx[y], fma(uy, gy[y], fma(uz, gz[y], acc[e])));
      }
      if (reac) {
        e = 0;
#pragma unroll
        for (int n = 0; n < 8; ++n)
#pragma unroll
          for (int y = 0; y <= n; ++y, ++e) acc[e] = fma(rc * pv[n], pv[y], acc[e]);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < 48; t += 16) {
    const double s = block_sums<NW>(acc + t, red);
    if (tid < 16) g.part[((size_t)cell * B::COUNT + slab) * 48 + t + tid] = s;
  }
}

// The slabs' sums, the symmetric matrix, and the status of one cell per wave.
__global__ __launch_bounds__(256) void q1t_finish_kernel(Q1tBasis g, int slabs) {
  const int cell = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (cell >= g.n_cells) return;
  if (lane < 44) {
    double s = 0.0;
    for (int t = 0; t < slabs; ++t) s += g.part[((size_t)cell * slabs + t) * 48 + lane];
    if (lane < 36) {
      int i = 0;
      while ((i + 1) * (i + 2) / 2 <= lane) ++i;
      const int j = lane - i * (i + 1) / 2;
      g.Mat[(size_t)cell * 64 + i * 8 + j] = s;
      g.Mat[(size_t)cell * 64 + j * 8 + i] = s;
    } else {
      g.b[(size_t)cell * 8 + lane - 36] = s;
    }
  }
  int it = 0, state = 0;
  if (lane < g.nr) {
    it = g.iters[((size_t)cell * g.nr + lane) * 2];
    state = g.iters[((size_t)cell * g.nr + lane) * 2 + 1];
  }
  int most = it;  // a basis that was not iterated repeats the largest count
#pragma unroll
  for (int off = 1; off < 8; off <<= 1) most = max(most, __shfl_xor(most, off));
  const int st = __any(state == 3)   ? MSFEC_CELL_NONFINITE
                 : __any(state == 2) ? MSFEC_CELL_NOT_SPD
                 : __any(state == 1) ? MSFEC_CELL_NOT_CONVERGED
                                     : MSFEC_CELL_OK;
  if (lane < 8) {
    g.cgit[((size_t)cell * 8 + lane) * 2] = lane < g.nr ? it : most;
    g.cgit[((size_t)cell * 8 + lane) * 2 + 1] = state;
  }
  if (lane == 0) g.status[cell] = st;
}

template <int M>
hipError_t rows(const Q1tRows& g, hipStream_t s) {
  const dim3 grid(g.n_cells * RowTile<M>::TILES), block(RowTile<M>::NT);
  if (g.edge) hipLaunchKernelGGL((q1t_rows_kernel<M, true>), grid, block, 0, s, g);
  else hipLaunchKernelGGL((q1t_rows_kernel<M, false>), grid, block, 0, s, g);
  return hipGetLastError();
}

template <int M, int LZ>
hipError_t cg(const Q1tCg& g, hipStream_t s) {
  const int blocks = (g.n_cells + 7) / 8 * 8 * g.nr;
  hipLaunchKernelGGL((q1t_cg_kernel<M, LZ>), dim3(blocks), dim3(std::max(64, M * M * M / LZ)), 0, s, g);
  return hipGetLastError();
}

template <int M>
hipError_t basis(const Q1tBasis& g, hipStream_t s) {
  hipLaunchKernelGGL(q1t_basis_kernel<M>, dim3(g.n_cells * Slab<M>::COUNT), dim3(Slab<M>::NT), 0, s, g);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(q1t_finish_kernel, dim3((g.n_cells + 3) / 4), dim3(256), 0, s, g, Slab<M>::COUNT);
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
  switch (l) {
    case 1:
      if (!g.direct) return cg<2, 1>(g, s);
      hipLaunchKernelGGL(q1t_direct_kernel<2>, dim3(g.n_cells), dim3(64), 0, s, g);
      break;
    case 2:
      if (!g.direct) return cg<4, 1>(g, s);
      hipLaunchKernelGGL(q1t_direct_kernel<4>, dim3(g.n_cells), dim3(64), 0, s, g);
      break;
    case 3: return cg<8, 2>(g, s);
    default: return cg<16, 4>(g, s);
  }
  return hipGetLastError();
}

int q1t_slabs(int l) {
  return l == 1 ? Slab<2>::COUNT : l == 2 ? Slab<4>::COUNT : l == 3 ? Slab<8>::COUNT : Slab<16>::COUNT;
}

hipError_t q1t_basis(int l, const Q1tBasis& g, hipStream_t s) {
  switch (l) {
    case 1: return basis<2>(g, s);
    case 2: return basis<4>(g, s);
    case 3: return basis<8>(g, s);
    default: return basis<16>(g, s);
  }
}

}  // namespace msfec_detail
