// Sine and cosine transforms of edge, face and cell fields of the refined box:
// three components on a lattice of (M + 1)^3 points in LDS, index
// (k (M + 1) + j) (M + 1) + i, M = 2, 4, 8 or 16.
//
// A cell value sits at half points (cosines, modes 0 .. M-1), a node value
// that vanishes at both ends at the points 1 .. M-1 (sines, modes 1 .. M-1).
// With kappa = 2 sin(k pi / 2M) the difference of two nodes takes the sine of
// mode k to kappa times its cosine.  The transforms are not normalised: both
// ways together multiply by M / 2 per direction, by M for mode 0.
#pragma once
#include <hip/hip_runtime.h>

namespace msfec_trig {

// cos(t pi / 32)
__host__ __device__ constexpr double cos32(int t) {
  t = ((t % 64) + 64) % 64;
  if (t > 32) t = 64 - t;
  const int u = t > 16 ? 32 - t : t;
  const double c = u == 0    ? 1.0
                   : u == 1  ? 0.99518472667219692873
                   : u == 2  ? 0.98078528040323043058
                   : u == 3  ? 0.95694033573220882438
                   : u == 4  ? 0.92387953251128673848
                   : u == 5  ? 0.88192126434835504956
                   : u == 6  ? 0.83146961230254523567
                   : u == 7  ? 0.77301045336273699338
                   : u == 8  ? 0.70710678118654757274
                   : u == 9  ? 0.63439328416364548779
                   : u == 10 ? 0.55557023301960228867
                   : u == 11 ? 0.47139673682599780857
                   : u == 12 ? 0.38268343236508983729
                   : u == 13 ? 0.29028467725446233105
                   : u == 14 ? 0.19509032201612833135
                   : u == 15 ? 0.098017140329560770162
                             : 0.0;
  return t > 16 ? -c : c;
}
// cos(t pi / 2M)
template <int M>
__host__ __device__ constexpr double cosm(int t) {
  return cos32(t * (16 / M));
}

// One line of M values, in place; the even and the odd modes use the sums
// and the differences of mirrored points, half the products of the full
// matrix.
//   sine: points and modes 1 .. M-1 (index 0 is not read, and zero after)
template <int M>
__device__ __forceinline__ void sine_line(double* v) {
  constexpr int H = M / 2;
  double s[H], d[H];
#pragma unroll
  for (int j = 1; j < H; ++j) {
    s[j] = v[j] + v[M - j];
    d[j] = v[j] - v[M - j];
  }
  const double mid = v[H];
  v[0] = 0.0;
#pragma unroll
  for (int k = 1; k < M; ++k) {
    double a = k & 1 ? mid * cosm<M>(M - 2 * H * k) : 0.0;
#pragma unroll
    for (int j = 1; j < H; ++j) a = fma(cosm<M>(M - 2 * j * k), k & 1 ? s[j] : d[j], a);
    v[k] = a;
  }
}
//   cosine: M cell values to modes 0 .. M-1
template <int M>
__device__ __forceinline__ void cos_line(double* v) {
  constexpr int H = M / 2;
  double s[H], d[H];
#pragma unroll
  for (int c = 0; c < H; ++c) {
    s[c] = v[c] + v[M - 1 - c];
    d[c] = v[c] - v[M - 1 - c];
  }
#pragma unroll
  for (int k = 0; k < M; ++k) {
    double a = 0.0;
#pragma unroll
    for (int c = 0; c < H; ++c) a = fma(cosm<M>((2 * c + 1) * k), k & 1 ? d[c] : s[c], a);
    v[k] = a;
  }
}
//   and back
template <int M>
__device__ __forceinline__ void cos_line_t(double* v) {
  constexpr int H = M / 2;
  double e[H], o[H];
#pragma unroll
  for (int c = 0; c < H; ++c) {
    e[c] = o[c] = 0.0;
#pragma unroll
    for (int k = 0; k < M; k += 2) e[c] = fma(cosm<M>((2 * c + 1) * k), v[k], e[c]);
#pragma unroll
    for (int k = 1; k < M; k += 2) o[c] = fma(cosm<M>((2 * c + 1) * k), v[k], o[c]);
  }
#pragma unroll
  for (int c = 0; c < H; ++c) {
    v[c] = e[c] + o[c];
    v[M - 1 - c] = e[c] - o[c];
  }
}

// An edge field is a cosine along its axis and a sine across it, a face field
// the other way round.
enum Kind { EdgeToModes, CellToModes, FaceToModes, ModesToFace };

// All `comps` components, in place, NT threads; ends with a barrier.
template <int M, int NT, int K>
__device__ __forceinline__ void transform(double* E, int comps) {
  constexpr int S = M + 1, S3 = S * S * S, M2 = M * M;
#pragma unroll 1
  for (int d = 0; d < 3; ++d) {
    const int step = d == 0 ? 1 : (d == 1 ? S : S * S);
    for (int ln = threadIdx.x; ln < comps * M2; ln += NT) {
      const int a = ln / M2, u = ln % M, w = (ln / M) % M;
      // lines along x: neighbouring lanes S values apart (no bank conflict,
      // S is odd); along y and z: neighbouring values
      double* p = E + a * S3 + (d == 0 ? (w * S + u) * S : (d == 1 ? w * S * S + u : w * S + u));
      double v[M];
#pragma unroll
      for (int t = 0; t < M; ++t) v[t] = p[t * step];
      if constexpr (K == EdgeToModes) {
        if (a == d) cos_line<M>(v);
        else sine_line<M>(v);
      } else if constexpr (K == CellToModes) {
        cos_line<M>(v);
      } else if constexpr (K == FaceToModes) {
        if (a == d) sine_line<M>(v);
        else cos_line<M>(v);
      } else {
        if (a == d) sine_line<M>(v);
        else cos_line_t<M>(v);
      }
#pragma unroll
      for (int t = 0; t < M; ++t) p[t * step] = v[t];
    }
    __syncthreads();
  }
}

}  // namespace msfec_trig
