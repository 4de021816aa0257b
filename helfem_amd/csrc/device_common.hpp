// Device helpers shared by the atomic and diatomic kernels (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>

namespace hfg {
namespace dev {

constexpr int NT = 256;  // threads per workgroup (4 wave64)

__device__ inline double wave_sum(double v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  return v;
}

// Reduce two values over the 256-thread block; result valid in thread 0.
__device__ inline void block_sum2(double &x, double &y, double *red) {
  x = wave_sum(x);
  y = wave_sum(y);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) {
    red[w] = x;
    red[4 + w] = y;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    x = red[0] + red[1] + red[2] + red[3];
    y = red[4] + red[5] + red[6] + red[7];
  }
}

typedef double v4d __attribute__((ext_vector_type(4)));

// D(16x16) += X(16x16) * Y(16x16), one wave, four v_mfma_f64_16x16x4f64.
// Lane l (g = l/16, c = l%16) supplies X(c, k) and Y(k, c) for the inner
// index k = g + 4s of step s, and holds the result D(g + 4r, c) in component
// r (the layout measured on gfx950).  With this choice of k a result tile is
// already in Y-operand layout, so products chain without a shuffle.
__device__ inline v4d mfma_16x16x16(const double xs[4], const double ys[4], v4d d) {
#pragma unroll
  for (int s = 0; s < 4; ++s) d = __builtin_amdgcn_mfma_f64_16x16x4f64(xs[s], ys[s], d, 0, 0, 0);
  return d;
}

__device__ inline v4d mfma_16x16x16(const double xs[4], v4d y, v4d d) {
  const double ys[4] = {y[0], y[1], y[2], y[3]};
  return mfma_16x16x16(xs, ys, d);
}

typedef float v4f __attribute__((ext_vector_type(4)));

// Operand/result layout of the 16x16x4 matrix instructions, per precision.
// Both take X(c, k) and Y(k, c) from lane l (g = l/16, c = l%16) with the
// instruction's inner index g; the result row held in accumulator component
// r differs (measured on gfx950 with one-hot probes):
//   v_mfma_f64_16x16x4f64: D(g + 4r, c)      v_mfma_f32_16x16x4f32: D(4g + r, c)
// Choosing the global inner index of step s as row(g, s) makes a result tile
// the next product's Y operand without a shuffle, in either precision.
template <typename T> struct Mma;
template <> struct Mma<double> {
  typedef v4d acc_t;
  __device__ static int row(int g, int s) { return g + 4 * s; }
  __device__ static acc_t step(double x, double y, acc_t d) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(x, y, d, 0, 0, 0);
  }
};
template <> struct Mma<float> {
  typedef v4f acc_t;
  __device__ static int row(int g, int s) { return 4 * g + s; }
  __device__ static acc_t step(float x, float y, acc_t d) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, d, 0, 0, 0);
  }
};

// D(16x16) += X Y over the 16-long inner index, four instructions.
template <typename T>
__device__ inline typename Mma<T>::acc_t mma16(const T xs[4], const T ys[4], typename Mma<T>::acc_t d) {
#pragma unroll
  for (int s = 0; s < 4; ++s) d = Mma<T>::step(xs[s], ys[s], d);
  return d;
}
template <typename T>
__device__ inline typename Mma<T>::acc_t mma16(const T xs[4], typename Mma<T>::acc_t y,
                                               typename Mma<T>::acc_t d) {
#pragma unroll
  for (int s = 0; s < 4; ++s) d = Mma<T>::step(xs[s], y[s], d);
  return d;
}

// Index s of the system owning workgroup b of a launch that concatenates
// the grids of n systems: the largest s with start[s] <= b (systems with no
// workgroups have start[s] == start[s+1] and are skipped).
__device__ inline int batch_find(const int *start, int n, int b) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (start[mid] <= b)
      lo = mid;
    else
      hi = mid - 1;
  }
  // the same for every lane: kept in a scalar register, so the system's
  // argument struct is read with scalar loads
  return __builtin_amdgcn_readfirstlane(lo);
}

// Whole columns b0 .. ni-1 of one element of a Coulomb shell block, zeros
// included: tile T(a,b) = T[a + 16 b] in rows f0 + a, and in the last column the
// next element's first column N[0 .. nn) (nn = 0 without one; N[0] is in T).
// Block rows start at J, its first column at J; the shells leave out their first
// roff and coff functions, and may then have none (one element of two nodes: a
// shell of m != 0).  A wave per column, lanes along rows in 16-byte pairs from the
// first aligned address on.
__device__ inline void j_store_columns(double *J, int64_t ldj, int nrow, int roff, int coff, int f0, int ni, int nn,
                                       int b0, const double *T, const double *N) {
  if (nrow <= 0) return;
  const int lane = threadIdx.x & 63;
  for (int b = b0 + (int)(threadIdx.x >> 6); b < ni; b += (int)(blockDim.x >> 6)) {
    const int c = f0 + b - coff;
    if (c < 0) continue;
    double *col = J + (int64_t)c * ldj;
    const int nx = b == ni - 1 ? nn : 0;
    auto at = [&](int r) {
      const int a = r + roff - f0;
      if (a >= 0 && a < ni) return T[a + TILE * b];
      return a >= ni && a - (ni - 1) < nx ? N[a - (ni - 1)] : 0.0;
    };
    const int odd = (int)((reinterpret_cast<uintptr_t>(col) >> 3) & 1);
    for (int r = 2 * lane - odd; r < nrow; r += 128) {
      if (r >= 0 && r + 1 < nrow)
        *reinterpret_cast<double2 *>(col + r) = make_double2(at(r), at(r + 1));
      else if (r >= 0)
        col[r] = at(r);
      else
        col[0] = at(0);  // r = -1: nrow >= 1
    }
  }
}

// Workgroup w of a grid of 8 * xcd_share(n) places -> work item: each XCD (w & 7)
// takes a contiguous share, so that neighbours meet in one L2; items from n on are
// empty.
__host__ __device__ inline int xcd_share(int n) { return (n + 7) / 8; }
__device__ inline int xcd_item(int w, int n) {
  const int i = (w & 7) * xcd_share(n) + (w >> 3);
  return i < n ? i : -1;
}

// v[k] = sum_p pair_c[nc p + k] P-tile(pair p) over the pair list [p0, p1): the
// waves deal the pairs in runs of JG_RUN, a lane holds entries lane + 64 u, and the
// waves' sums meet in part [4][NC][TILE2].  at(kl, a, b) is the entry of P.
constexpr int JG_RUN = 4;
template <int NC, typename At>
__device__ inline void j_pair_sums(const int *pair_kl, const double *pair_c, int p0, int p1, At at, double *part,
                                   double *out) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, a = lane & 15, b = lane >> 4;
  double v[NC][4];
#pragma unroll
  for (int k = 0; k < NC; ++k)
#pragma unroll
    for (int u = 0; u < 4; ++u) v[k][u] = 0.0;
  const int w0 = __builtin_amdgcn_readfirstlane(w);
  for (int p = p0 + w0 * JG_RUN; p < p1; p += 4 * JG_RUN) {
    double x[JG_RUN][4];
#pragma unroll
    for (int i = 0; i < JG_RUN; ++i) {
      const int kl = pair_kl[min(p + i, p1 - 1)];
#pragma unroll
      for (int u = 0; u < 4; ++u) x[i][u] = at(kl, a, b + 4 * u);
    }
#pragma unroll
    for (int i = 0; i < JG_RUN; ++i)
      if (p + i < p1)
#pragma unroll
        for (int k = 0; k < NC; ++k) {
          const double c = pair_c[NC * (p + i) + k];
#pragma unroll
          for (int u = 0; u < 4; ++u) v[k][u] += c * x[i][u];
        }
  }
#pragma unroll
  for (int k = 0; k < NC; ++k)
#pragma unroll
    for (int u = 0; u < 4; ++u) part[(w * NC + k) * TILE2 + lane + 64 * u] = v[k][u];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NC; ++k)
    out[k] = part[k * TILE2 + t] + part[(NC + k) * TILE2 + t] + part[(2 * NC + k) * TILE2 + t] +
             part[(3 * NC + k) * TILE2 + t];
}

}  // namespace dev
}  // namespace hfg
