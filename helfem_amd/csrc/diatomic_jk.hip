// Diatomic (prolate spheroidal) Coulomb and exchange kernels (FP64), gfx950.
//
// Data layout (device):
//   P, J, K   dense Nbf x Nbf column-major in the pure basis; shell a's
//             radial function r is row poff[a] + r - skip[a] (r >= skip[a]).
//   pq        per ((L,|M|), element) four 16x16 zero-padded tiles: the
//             disjoint integrals P0, P2, Q0, Q2 (basis.cpp:352-394).
//   chol      per ((L,|M|), element) and Cholesky vector p the two channel
//             blocks M0_p(a,b) = B(a + b Ni, p), M2_p(a,b) = B(Ni^2 + a + b Ni, p)
//             of W = B diag(sigma) B' (basis.cpp:1492-1537), and sigma.
//
// Coulomb (basis.cpp:1627-1816): two density channels per (L,M),
// Paux0 = sum mod_coeff * P_kl and Paux2 = sum coeff * P_kl, of which only
// the element-diagonal bands matter.  Kernel 1 gathers both bands, reduces
// the P/Q traces and applies the in-element kernel through the Cholesky
// factor; kernel 2 adds the other elements' traces times P and Q, the whole
// band; kernel 3 expands the bands into the shell blocks of J.
// Exchange (basis.cpp:1818-2089), one-step form: one workgroup per (output block
// (j,k), element pair (e,f)); for each coupled (L,|M|) the four Gaunt-weighted
// density tiles R00, R02, R20, R22 are formed in registers and contracted on
// the matrix cores with the disjoint P/Q factors (e != f) or the four-channel
// Cholesky factor (e == f).  The density tiles are first copied out of P into
// a tiled array (k_dia_ptile: one contiguous, aligned 2 KB tile per (element
// pair, density block) in operand order), so a term's gather is one aligned
// 32-byte read per lane.
#include "hfgpu_internal.hpp"
#include "device_common.hpp"
#include <algorithm>
#include <type_traits>

// terms in flight per lane in the cross-element gathers, and that launch's
// waves per SIMD
#ifndef HFG_DIA_OFF_UNROLL
#define HFG_DIA_OFF_UNROLL 4
#endif
#ifndef HFG_DIA_OFF_WAVES
#define HFG_DIA_OFF_WAVES 5
#endif

namespace hfg {
namespace {

using namespace dev;

__device__ inline long long pure_row(const int *skip, const long long *poff, int shell, int r) {
  const int s = skip[shell];
  return r >= s ? poff[shell] + (r - s) : -1;
}

// --- Coulomb -----------------------------------------------------------------

struct DJArgs {
  const double *P;
  int64_t ldp;
  int Nel, Nang;
  const int *first, *ni, *skip;
  const long long *poff;
  const double *pq, *chol, *sigma;
  const int *chol_off, *chol_rank;
  const int *LM_ilm;
  const double *LM_fac;
  const int *pstart, *pair_kl;
  const double *pair_c;
  double *Jin, *ds, *db;
  int n_LM;
};

// One workgroup per ((L,M), element), items e n_LM + q in shares per XCD: the L of
// one M read the same tiles of P.  The waves deal the pairs: a chain of dependent
// loads a quarter as long (N2, 16 shells per |m| <= 2: 410 -> 269 us).
__global__ void __launch_bounds__(NT) k_dia_j_gather(DJArgs A) {
  const int item = xcd_item(blockIdx.x, A.n_LM * A.Nel);
  if (item < 0) return;
  const int e = item / A.n_LM, q = item - e * A.n_LM;
  const int t = threadIdx.x, a = t & 15, b = t >> 4;
  const int ni = A.ni[e], f0 = A.first[e], ilm = A.LM_ilm[q];
  const double fac = A.LM_fac[q];
  __shared__ double part[8 * TILE2];
  __shared__ double s0[TILE2], s2[TILE2];
  __shared__ double red[8];
  double *sc = part;  // 2 TILE2 channel weights, once the partial sums are added
  auto at = [&](int kl, int i, int j) {
    const int k = kl / A.Nang, l = kl - k * A.Nang;
    const long long r = pure_row(A.skip, A.poff, k, f0 + i), c = pure_row(A.skip, A.poff, l, f0 + j);
    return i < ni && j < ni && r >= 0 && c >= 0 ? A.P[r + c * A.ldp] : 0.0;
  };
  double v[2];
  j_pair_sums<2>(A.pair_kl, A.pair_c, A.pstart[q], A.pstart[q + 1], at, part, v);
  s0[t] = v[0];
  s2[t] = v[1];
  __syncthreads();
  // traces tr(X s) = sum_ab X(a,b) s(b,a)
  const size_t tb = ((size_t)ilm * A.Nel + e) * 4 * TILE2;
  const double x0 = s0[b + TILE * a], x2 = s2[b + TILE * a];
  double dsv = A.pq[tb + t] * x0 - A.pq[tb + TILE2 + t] * x2;
  double dbv = A.pq[tb + 2 * TILE2 + t] * x0 - A.pq[tb + 3 * TILE2 + t] * x2;
  block_sum2(dsv, dbv, red);
  if (t == 0) {
    A.ds[(size_t)q * A.Nel + e] = fac * dsv;
    A.db[(size_t)q * A.Nel + e] = fac * dbv;
  }
  // c_p = sigma_p <[M0_p; M2_p], [s0; s2]>, wave w handles p = w, w+4, ...
  const int rank = A.chol_rank[ilm * A.Nel + e], off = A.chol_off[ilm * A.Nel + e];
  const double *M = A.chol + (size_t)off * 2 * TILE2;
  const int lane = t & 63, w = t >> 6;
  for (int p = w; p < rank; p += 4) {
    const double *M0 = M + (size_t)p * 2 * TILE2, *M2 = M0 + TILE2;
    double s = 0.0;
#pragma unroll
    for (int u = 0; u < 4; ++u) s += M0[lane + 64 * u] * s0[lane + 64 * u] + M2[lane + 64 * u] * s2[lane + 64 * u];
    s = wave_sum(s);
    if (lane == 0) sc[p] = s * A.sigma[off + p];
  }
  __syncthreads();
  double j0 = 0.0, j2 = 0.0;
#pragma unroll 4
  for (int p = 0; p < rank; ++p) {
    const double cp = sc[p];
    j0 += M[(size_t)p * 2 * TILE2 + t] * cp;
    j2 += M[(size_t)p * 2 * TILE2 + TILE2 + t] * cp;
  }
  double *out = A.Jin + ((size_t)q * A.Nel + e) * 2 * TILE2;
  out[t] = j0 * fac;
  out[TILE2 + t] = j2 * fac;
}

struct DJBandArgs {
  int Nel;
  const int *LM_ilm;
  const double *pq, *ds, *db;
  double *Jin;
};

// The whole potential of (L,M) in element e, in place, one workgroup per (q, e):
// Ja0 = Jin0 + preA P0 + preB Q0, Ja2 = Jin2 - preA P2 - preB Q2 with preA =
// sum_{j>e} db(q,j), preB = sum_{j<e} ds(q,j).  Formed once here, an output block
// reads two tiles per (L,M) instead of six.
__global__ void __launch_bounds__(NT) k_dia_j_band(DJBandArgs A) {
  const int q = blockIdx.x / A.Nel, e = blockIdx.x - q * A.Nel, t = threadIdx.x;
  const double *ds = A.ds + (size_t)q * A.Nel, *db = A.db + (size_t)q * A.Nel;
  double pa = 0.0, pb = 0.0;
  for (int j = A.Nel - 1; j > e; --j) pa += db[j];
  for (int j = 0; j < e; ++j) pb += ds[j];
  const double *pq = A.pq + ((size_t)A.LM_ilm[q] * A.Nel + e) * 4 * TILE2;
  double *jin = A.Jin + (size_t)blockIdx.x * 2 * TILE2;
  jin[t] = jin[t] + pa * pq[t] + pb * pq[2 * TILE2 + t];
  jin[TILE2 + t] = jin[TILE2 + t] - pa * pq[TILE2 + t] - pb * pq[3 * TILE2 + t];
}

struct DJOutArgs {
  double *J;
  int64_t ldj;
  int Nel, Nang;
  const int *first, *ni, *skip;
  const long long *poff;
  const double *Jin;
  const int *out_start, *out_q;
  const double *out_c;
};

// One workgroup per (output shell block (i,j), element): the element's columns of
// the block from top to bottom, zeros included, so that J is written in one pass
// of whole columns.  A column shared with element e-1 is e-1's.  The blocks i of
// one column run on one XCD, whose L2 joins their partial lines.  Bound by the
// latency of the tile reads: fill + expand of N2 (16 shells per |m| <= 2) 72 + 276
// -> 197 us (and 8 for the band tiles).
__global__ void __launch_bounds__(NT) k_dia_j_expand(DJOutArgs A) {
  const int item = xcd_item(blockIdx.x, A.Nang * A.Nang * A.Nel);
  if (item < 0) return;
  const int je = item / A.Nang, i = item - je * A.Nang, j = je / A.Nel, e = je - j * A.Nel, ij = i * A.Nang + j;
  const int o0 = A.out_start[ij], o1 = A.out_start[ij + 1];
  const int t = threadIdx.x, a = t & 15, b = t >> 4;
  const int ni = A.ni[e], f0 = A.first[e], nn = e + 1 < A.Nel ? A.ni[e + 1] : 0;
  __shared__ double sT[TILE2], sN[TILE];
  double v = 0.0, w = 0.0;
#pragma unroll 4
  for (int o = o0; o < o1; ++o) {
    const double *x = A.Jin + ((size_t)A.out_q[o] * A.Nel + e) * 2 * TILE2;
    v += A.out_c[2 * o] * x[t] + A.out_c[2 * o + 1] * x[TILE2 + t];
  }
  if (nn && t < TILE)
#pragma unroll 4
    for (int o = o0; o < o1; ++o) {
      const double *x = A.Jin + ((size_t)A.out_q[o] * A.Nel + e + 1) * 2 * TILE2;
      w += A.out_c[2 * o] * x[t] + A.out_c[2 * o + 1] * x[TILE2 + t];
    }
  if (t < TILE) sN[t] = w;
  sT[t] = v;
  __syncthreads();
  if (nn && a == ni - 1 && b == ni - 1) sT[t] = v + sN[0];
  __syncthreads();
  double *J = A.J + A.poff[i] + A.poff[j] * A.ldj;
  j_store_columns(J, A.ldj, (int)(A.poff[i + 1] - A.poff[i]), A.skip[i], A.skip[j], f0, ni, nn, e > 0, sT, sN);
}

// --- Exchange ----------------------------------------------------------------

// One pass over P per shell block pair i <= l and 32-row chunk ch of P_il:
// partial sums for the Frobenius norms of P_il and P_li (the reference's
// screen) and partial maxima for the symmetry test, part[(il * nch + ch) *
// 4 + {0..3}] = (sum P_il^2, sum P_li^2, max |P_il - P_li'|, max |P_il|),
// reduced on the host.  32x32 sub-tiles of both blocks are read coalesced
// into LDS and compared transposed.  Shell a spans rows poff[a] .. poff[a] +
// Nrad - skip[a] (a Nrad, no skip when the tables are null: atomic basis).
__device__ inline void block_stats_body(const double *P, int64_t ldp, int Nrad, int Nang, const int *skip,
                                        const long long *poff, double *part, int il, int ch, int nch) {
  const int i = il / Nang, l = il - i * Nang;
  if (i > l) return;  // covered by the workgroups of (l, i)
  __shared__ double A[32][33], B[32][33];
  __shared__ double red[16];
  double amax = 0.0, pmax = 0.0, ssa = 0.0, ssb = 0.0;
  const int ri = Nrad - (skip ? skip[i] : 0), rl = Nrad - (skip ? skip[l] : 0);
  const long long oi = poff ? poff[i] : (long long)i * Nrad, ol = poff ? poff[l] : (long long)l * Nrad;
  const int t = threadIdx.x, x = t & 31, y0 = t >> 5;
  for (int tr = 32 * ch; tr < ri; tr += 32 * nch)
    for (int tc = 0; tc < rl; tc += 32) {
      __syncthreads();
      // A[x][y] = P_il(tr + x, tc + y), B[x][y] = P_li(tc + x, tr + y)
      for (int y = y0; y < 32; y += NT / 32) {
        const bool va = tr + x < ri && tc + y < rl, vb = tc + x < rl && tr + y < ri;
        const double pa = va ? P[(oi + tr + x) + (ol + tc + y) * ldp] : 0.0;
        const double pb = vb ? P[(ol + tc + x) + (oi + tr + y) * ldp] : 0.0;
        A[x][y] = pa;
        B[x][y] = pb;
        ssa += pa * pa;
        ssb += pb * pb;
      }
      __syncthreads();
      for (int y = y0; y < 32; y += NT / 32) {
        const double dlt = fabs(A[x][y] - B[y][x]);
        amax = isnan(dlt) ? HUGE_VAL : fmax(amax, dlt);  // a NaN counts as asymmetric
        pmax = fmax(pmax, fabs(A[x][y]));
      }
    }
  for (int o = 32; o > 0; o >>= 1) {
    amax = fmax(amax, __shfl_xor(amax, o));
    pmax = fmax(pmax, __shfl_xor(pmax, o));
    ssa += __shfl_xor(ssa, o);
    ssb += __shfl_xor(ssb, o);
  }
  const int w = t >> 6;
  if ((t & 63) == 0) {
    red[w] = amax;
    red[4 + w] = pmax;
    red[8 + w] = ssa;
    red[12 + w] = ssb;
  }
  __syncthreads();
  if (t == 0) {
    double *o = part + ((size_t)il * nch + ch) * 4;
    o[0] = (red[8] + red[9]) + (red[10] + red[11]);
    o[1] = (red[12] + red[13]) + (red[14] + red[15]);
    o[2] = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
    o[3] = fmax(fmax(red[4], red[5]), fmax(red[6], red[7]));
  }
}

__global__ void __launch_bounds__(NT) k_block_stats(const double *P, int64_t ldp, int Nrad, int Nang,
                                                    const int *skip, const long long *poff, double *part) {
  block_stats_body(P, ldp, Nrad, Nang, skip, poff, part, blockIdx.x, blockIdx.y, gridDim.y);
}

// Many matrices in one launch: workgroup b of system s (start[s] <= b <
// start[s+1]) takes shell pair il = local / nch and chunk local % nch.
__global__ void __launch_bounds__(NT) k_block_stats_batch(const StatsArgs *args, const int *start, int n) {
  const int s = batch_find(start, n, blockIdx.x);
  const StatsArgs &a = args[s];
  const int loc = blockIdx.x - start[s], nch = a.nch;
  block_stats_body(a.P, a.ldp, a.Nrad, a.Nang, a.skip, a.poff, a.part, loc / nch, loc - (loc / nch) * nch, nch);
}

// Two products sharing the Y operand, issued interleaved so the two
// accumulation chains overlap: da += Xa Y, db += Xb Y (16x16x16 each).
template <typename T>
__device__ inline void mma_pair(const T xa[4], const T xb[4], const T ys[4], typename Mma<T>::acc_t &da,
                                typename Mma<T>::acc_t &db) {
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    da = Mma<T>::step(xa[s], ys[s], da);
    db = Mma<T>::step(xb[s], ys[s], db);
  }
}

// da += Xa Ya, db += Xb Yb with Ya, Yb result tiles, interleaved.
template <typename T>
__device__ inline void mma_pair2(const T xa[4], typename Mma<T>::acc_t ya, typename Mma<T>::acc_t &da,
                                 const T xb[4], typename Mma<T>::acc_t yb, typename Mma<T>::acc_t &db) {
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    da = Mma<T>::step(xa[s], ya[s], da);
    db = Mma<T>::step(xb[s], yb[s], db);
  }
}

// Cholesky channel tiles of vector p in both operand layouts:
// y = M(c, k) (M' as Y operand), x = M(k, c) (M' as X operand), k = row(g, s).
template <typename T>
__device__ inline void load_chol(const T *M, int p, const int kk[4], int c, T y0[4], T y2[4], T x0[4], T x2[4]) {
  const T *M0 = M + (size_t)p * 2 * TILE2, *M2 = M0 + TILE2;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    y0[s] = M0[c + TILE * kk[s]];
    y2[s] = M2[c + TILE * kk[s]];
    x0[s] = M0[kk[s] + TILE * c];
    x2[s] = M2[kk[s] + TILE * c];
  }
}

// Gaunt-weighted density tiles of one run, four channels, in matrix-operand
// layout (lane (g,c) holds R(c, row(g,s)) in entry s).  Lanes outside the
// element pair read a clamped entry (rloc, cloc) and are masked by cmask; the
// dropped radial function 0 of an m != 0 shell (only at the first radial
// index) is masked per term.  No branches, two terms' loads in flight.
template <typename T, int U = 2>
__device__ inline void gather_terms(const T *P, int64_t ldp, const int4 *tpos, const T *term_f, int q0, int q1,
                                    int rloc, const int cloc[4], const T cmask[4], T r00[4], T r02[4], T r20[4],
                                    T r22[4]) {
#pragma unroll
  for (int s = 0; s < 4; ++s) r00[s] = r02[s] = r20[s] = r22[s] = T(0);
  int q = q0;
  for (; q + U <= q1; q += U) {
    T x[U][4];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // (poff[i], poff[l] - skip[l], skip[i], skip[l]) of the term's density block
      const int4 tp = tpos[q + u];
      const long long row = tp.x + max(rloc - tp.z, 0), cb = tp.y;
      const bool rv = rloc >= tp.z;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const T v = P[row + (cb + max(cloc[s], tp.w)) * ldp];
        x[u][s] = (rv && cloc[s] >= tp.w) ? v : T(0);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const T f00 = term_f[4 * (q + u)], f02 = term_f[4 * (q + u) + 1], f20 = term_f[4 * (q + u) + 2],
              f22 = term_f[4 * (q + u) + 3];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        r00[s] += f00 * x[u][s];
        r02[s] += f02 * x[u][s];
        r20[s] += f20 * x[u][s];
        r22[s] += f22 * x[u][s];
      }
    }
  }
  for (; q < q1; ++q) {
    const int4 tp = tpos[q];
    const long long row = tp.x + max(rloc - tp.z, 0), cb = tp.y;
    const bool rv = rloc >= tp.z;
    const T f00 = term_f[4 * q], f02 = term_f[4 * q + 1], f20 = term_f[4 * q + 2], f22 = term_f[4 * q + 3];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const T v = P[row + (cb + max(cloc[s], tp.w)) * ldp];
      const T x = (rv && cloc[s] >= tp.w) ? v : T(0);
      r00[s] += f00 * x;
      r02[s] += f02 * x;
      r20[s] += f20 * x;
      r22[s] += f22 * x;
    }
  }
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    r00[s] *= cmask[s];
    r02[s] *= cmask[s];
    r20[s] *= cmask[s];
    r22[s] *= cmask[s];
  }
}

// Density tiles in gather order: tile (ef = e*Nel+f, src) holds the 16x16
// block of P between element e's radial functions of shell i and element f's
// of shell l (src = i*Nang+l from the source list), stored lane-major in the
// matrix-core operand order: entry lane*4 + s is R(c, row(g,s)) for lane
// (g,c), zero where a radial index is outside the element or is the dropped
// radial function 0 of an m != 0 shell.  One wave per tile.
template <typename T>
__global__ void __launch_bounds__(NT) k_dia_ptile(const double *P, int64_t ldp, int Nel, const int *first,
                                                  const int *ni, const int *skip, const long long *poff,
                                                  int Nang, const int *src_blk, int n_src, T *out) {
  const int64_t tile = (int64_t)blockIdx.x * (NT / 64) + (threadIdx.x >> 6);
  const int64_t n_tiles = (int64_t)Nel * Nel * n_src;
  if (tile >= n_tiles) return;
  const int ef = (int)(tile / n_src), src = (int)(tile - (int64_t)ef * n_src);
  const int e = ef / Nel, f = ef - e * Nel;
  const int blk = src_blk[src], i = blk / Nang, l = blk - i * Nang;
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const int rr = first[e] + c, si = skip[i], sl = skip[l];
  const bool rv = c < ni[e] && rr >= si;
  typename Mma<T>::acc_t v;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int kk = Mma<T>::row(g, s), cc = first[f] + kk;
    const bool ok = rv && kk < ni[f] && cc >= sl;
    v[s] = ok ? (T)P[(poff[i] + rr - si) + (poff[l] + cc - sl) * ldp] : T(0);
  }
  *reinterpret_cast<typename Mma<T>::acc_t *>(out + tile * TILE2 + lane * 4) = v;
}

// gather_terms over the tiled density: term q reads tile tt[q] of the
// element pair's slice pt (one 4-vector per lane), masks already applied.
template <typename T, int U = 2>
__device__ inline void gather_tiles(const T *pt, const int *tt, const T *term_f, int q0, int q1, T r00[4],
                                    T r02[4], T r20[4], T r22[4]) {
  typedef typename Mma<T>::acc_t vec;
#pragma unroll
  for (int s = 0; s < 4; ++s) r00[s] = r02[s] = r20[s] = r22[s] = T(0);
  int q = q0;
  for (; q + U <= q1; q += U) {
    vec x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = *reinterpret_cast<const vec *>(pt + (size_t)tt[q + u] * TILE2);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const T f00 = term_f[4 * (q + u)], f02 = term_f[4 * (q + u) + 1], f20 = term_f[4 * (q + u) + 2],
              f22 = term_f[4 * (q + u) + 3];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        r00[s] += f00 * x[u][s];
        r02[s] += f02 * x[u][s];
        r20[s] += f20 * x[u][s];
        r22[s] += f22 * x[u][s];
      }
    }
  }
  for (; q < q1; ++q) {
    const vec x = *reinterpret_cast<const vec *>(pt + (size_t)tt[q] * TILE2);
    const T f00 = term_f[4 * q], f02 = term_f[4 * q + 1], f20 = term_f[4 * q + 2], f22 = term_f[4 * q + 3];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      r00[s] += f00 * x[s];
      r02[s] += f02 * x[s];
      r20[s] += f20 * x[s];
      r22[s] += f22 * x[s];
    }
  }
}

template <typename T>
struct DKArgs {
  const T *P;
  int64_t ldp;
  double *K;
  int64_t ldk;
  int Nel, Nang, n_act;
  const int *first, *ni, *skip;
  const long long *poff;
  const T *pq, *chol, *sigma;
  const int *chol_off, *chol_rank;
  const int *act_jk, *act_lstart, *lrun_ilm, *lrun_tstart;
  const int4 *tpos;
  const T *term_f;
  const int *efl;  // element pairs e*Nel+f of this launch
  int n_ef;
  const double *lsig;  // FP32 only: log scale of the (ilm, element) P/Q tiles
  const T *pt;         // tiled density (k_dia_ptile) or null: gather from P
  const int *ttile;    // per term: its tile in an element pair's slice
  int n_src;
  int sym;  // symmetric density: e > f pairs (e == f: j <= k) also written to the mirror
};

// One workgroup per (active output block (j,k), element pair (e,f)), the
// four waves splitting the block's coupled (L,|M|) runs.  Workgroups sharing
// (e,f) are mapped to one XCD so the (e,f) slice of the density tiles (or of
// P, when the tiles do not fit) stays in its L2.
// T = double is the reference's arithmetic; T = float gathers and multiplies
// in FP32 and sums the waves' tiles in FP64.
template <bool INSIDE, bool TILED, typename T>
__device__ inline void dia_k_body(const DKArgs<T> &A) {
  typedef Mma<T> MM;
  typedef typename MM::acc_t acc_t;
  const int w = blockIdx.x;
  const int xcd = w & 7, loc = w >> 3;
  const int efi = (loc / A.n_act) * 8 + xcd;
  const int act = loc - (loc / A.n_act) * A.n_act;
  if (efi >= A.n_ef) return;
  const int ef = A.efl[efi], e = ef / A.Nel, f = ef - e * A.Nel;
  const int jk = A.act_jk[act], j = jk / A.Nang, k = jk - j * A.Nang;
  if (INSIDE && A.sym && j > k) return;  // the mirror of block (k, j) covers it
  const int t = threadIdx.x, lane = t & 63, g = lane >> 4, c = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int ni = A.ni[e], nj = A.ni[f], fi = A.first[e], fj = A.first[f];
  __shared__ double red[4 * TILE2];
  acc_t acc = {0, 0, 0, 0}, acc2 = {0, 0, 0, 0};
  // Lanes outside the element pair read a clamped entry and are masked once
  // per tile; the dropped radial function 0 of an m != 0 shell (only at the
  // first radial index) is masked per term.  The term loop has no branches.
  const int rloc = fi + min(c, ni - 1);
  int cloc[4], kk[4];
  T cmask[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    kk[s] = MM::row(g, s);
    cloc[s] = fj + min(kk[s], nj - 1);
    cmask[s] = (c < ni && kk[s] < nj) ? T(1) : T(0);
  }
  const int r0 = A.act_lstart[act], r1 = A.act_lstart[act + 1];
  const T *pt = TILED ? A.pt + (size_t)ef * A.n_src * TILE2 + lane * 4 : nullptr;
  for (int run = r0 + wv; run < r1; run += 4) {
    const int ilm = A.lrun_ilm[run];
    T r00[4], r02[4], r20[4], r22[4];
    if constexpr (TILED)
      gather_tiles<T, INSIDE ? 2 : HFG_DIA_OFF_UNROLL>(pt, A.ttile, A.term_f, A.lrun_tstart[run],
                                                       A.lrun_tstart[run + 1], r00, r02, r20, r22);
    else
      gather_terms<T>(A.P, A.ldp, A.tpos, A.term_f, A.lrun_tstart[run], A.lrun_tstart[run + 1], rloc, cloc, cmask,
                      r00, r02, r20, r22);
    const T *te = A.pq + ((size_t)ilm * A.Nel + e) * 4 * TILE2;
    if (!INSIDE) {
      const T *tf = A.pq + ((size_t)ilm * A.Nel + f) * 4 * TILE2;
      const bool up = e > f;
      // row side: Q of e if e > f else P of e; column side the other kind
      const T *i0 = te + (up ? 2 : 0) * TILE2, *i2 = te + (up ? 3 : 1) * TILE2;
      const T *j0 = tf + (up ? 0 : 2) * TILE2, *j2 = tf + (up ? 1 : 3) * TILE2;
      T a0[4], a2[4], b0[4], b2[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int x = c + TILE * kk[s];
        a0[s] = i0[x];
        a2[s] = i2[x];
        b0[s] = j0[x];
        b2[s] = j2[x];
      }
      // two independent chains: ya = R00 j0' + R02 j2', yb = R20 j0' + R22 j2'
      acc_t ya = {0, 0, 0, 0}, yb = {0, 0, 0, 0};
      mma_pair<T>(r00, r20, b0, ya, yb);
      mma_pair<T>(r02, r22, b2, ya, yb);
      if constexpr (sizeof(T) == 4) {
        // FP32 tiles hold P / s and Q * s per (ilm, element): restore the
        // pair's Q(e) P(f) or P(e) Q(f) scale, s_f / s_e or s_e / s_f
        const double le = A.lsig[ilm * A.Nel + e], lf = A.lsig[ilm * A.Nel + f];
        const T rho = (T)exp(up ? lf - le : le - lf);
        ya *= rho;
        yb *= rho;
      }
      mma_pair2<T>(a0, ya, acc, a2, yb, acc2);  // acc += i0 ya, acc2 += i2 yb
    } else {
      const int rank = A.chol_rank[ilm * A.Nel + e], off = A.chol_off[ilm * A.Nel + e];
      const T *M = A.chol + (size_t)off * 2 * TILE2;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        r02[s] = -r02[s];
        r20[s] = -r20[s];
      }
      // M0', M2' as Y operands (y0, y2) and as X operands (x0, x2); the next
      // vector's tiles are loaded while the current one is on the matrix cores
      T y0[4], y2[4], x0[4], x2[4];
      load_chol<T>(M, 0, kk, c, y0, y2, x0, x2);
      T sg = rank > 0 ? A.sigma[off] : T(0);
      for (int p = 0; p < rank; ++p) {
        T ny0[4], ny2[4], nx0[4], nx2[4];
        T nsg = 0;
        if (p + 1 < rank) {
          load_chol<T>(M, p + 1, kk, c, ny0, ny2, nx0, nx2);
          nsg = A.sigma[off + p + 1];
        }
        // ya = R00 M0' - R02 M2', yb = -R20 M0' + R22 M2' (signs folded into
        // r02, r20); sigma_p = +-1 goes on the X operands, off the MFMA chain
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          x0[s] *= sg;
          x2[s] *= sg;
        }
        acc_t ya = {0, 0, 0, 0}, yb = {0, 0, 0, 0};
        mma_pair<T>(r00, r20, y0, ya, yb);
        mma_pair<T>(r02, r22, y2, ya, yb);
        mma_pair2<T>(x0, ya, acc, x2, yb, acc2);  // acc += sigma M0' ya, acc2 += sigma M2' yb
        if (p + 1 < rank) {
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            y0[s] = ny0[s];
            y2[s] = ny2[s];
            x0[s] = nx0[s];
            x2[s] = nx2[s];
          }
          sg = nsg;
        }
      }
    }
  }
  // combine the four waves' partial tiles (lane holds acc(row(g,r), c)) in FP64
  acc += acc2;
#pragma unroll
  for (int rr = 0; rr < 4; ++rr) red[wv * TILE2 + kk[rr] + TILE * c] = (double)acc[rr];
  __syncthreads();
  const int a = t & 15, b = t >> 4;
  if (a >= ni || b >= nj) return;
  const long long row = pure_row(A.skip, A.poff, j, fi + a), col = pure_row(A.skip, A.poff, k, fj + b);
  if (row < 0 || col < 0) return;
  const double v = red[t] + red[TILE2 + t] + red[2 * TILE2 + t] + red[3 * TILE2 + t];
  const bool srow = (a == 0 && e > 0) || (a == ni - 1 && e + 1 < A.Nel);
  const bool scol = (b == 0 && f > 0) || (b == nj - 1 && f + 1 < A.Nel);
  double *dst = A.K + row + col * A.ldk;
  if (srow || scol)
    atomicAdd(dst, -v);
  else
    *dst = -v;
  if (A.sym && (!INSIDE || j != k)) {
    // mirror tile (k, j, f, e) = this tile transposed
    double *mdst = A.K + col + row * A.ldk;
    if (srow || scol)
      atomicAdd(mdst, -v);
    else
      *mdst = -v;
  }
}

// Cross-element launch held to 5 waves per SIMD (96 registers), which the
// two-term gather fits; the in-element fallback keeps the compiler's choice.
template <typename T, bool TILED>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(HFG_DIA_OFF_WAVES))) k_dia_k_off(DKArgs<T> A) {
  dia_k_body<false, TILED, T>(A);
}
template <typename T, bool TILED>
__global__ void __launch_bounds__(NT) k_dia_k_in(DKArgs<T> A) {
  dia_k_body<true, TILED, T>(A);
}

// --- Cross-element exchange in two steps ----------------------------------------
//
// One workgroup per (column shell k, element pair (e,f)); each wave owns up to
// three rows j of the column (of one m and parity of l, which share their
// slots) and keeps their output tiles in registers over all coupled (L,|M|)
// groups of k.  Per group: the slot tiles V_b(i) = sum_l v_b(k,l) P(i,l) of
// the pair are gathered (waves split the slots) and multiplied by the column
// side's disjoint factors at once, H(i) = V0 j0' - V1 j2', which goes to LDS;
// then each wave sums G0 = sum c0 H, G1 = -sum c1 H of its rows from LDS and
// adds i0 G0 + i2 G1 (the four channel tiles R00 = sum c0 V0, R02 = -sum c0 V1,
// R20 = -sum c1 V0, R22 = sum c1 V1 of k_dia_k_off never exist).  The rows
// share each H tile, so the L2 gathers drop from |S_j| |S_k| per row and group
// to |S_k| per slot, and a row costs two 16x16x16 products and one LDS tile
// per slot and wave.  FP32 adds each group's products to the rows in FP64 (in
// FP32 the sum over all groups lost a quarter of a digit).
// N2 (lmax 16, 8 elements): 5.1 ms, 9.5 ms with the four channel tiles formed
// per row; the matrix pipe is busy 28% of it (1.4 ms), the rest is
// latency: tile gathers (2.2 ms of it), list loads and the two barriers per
// group.  Two 512-thread workgroups per CU (16 waves) measured fastest: 384
// threads 7.3, 256 threads 6.8, one of 1024 over two element pairs 5.4 ms;
// the lists staged in LDS 5.4, eight gathers in flight 5.2 ms.

template <typename T>
struct DK2Args {
  const T *pt;  // tiled density
  int n_src;
  double *K;
  int64_t ldk;
  int Nel, Nang;
  const int *first, *ni, *skip;
  const long long *poff;
  const T *pqo;        // P/Q tiles in operand order
  const double *lsig;  // FP32 only: log scale of the (ilm, element) P/Q tiles
  const int *wg, *kshell, *rows, *kg, *gilm, *gslot, *sl, *lt, *jo, *js;
  const T *ltv, *jtc;
  int sym;
};

// Slot tiles sit in LDS as two halves [half][lane][2], so that a wave's
// 16-byte accesses are contiguous (no bank conflicts).
template <typename T>
__device__ inline typename Mma<T>::acc_t h_load(const T *H, int lane) {
  typedef T v2 __attribute__((ext_vector_type(2)));
  const v2 a = *reinterpret_cast<const v2 *>(H + 2 * lane), b = *reinterpret_cast<const v2 *>(H + 128 + 2 * lane);
  return typename Mma<T>::acc_t{a[0], a[1], b[0], b[1]};
}
template <typename T>
__device__ inline void h_store(T *H, int lane, typename Mma<T>::acc_t v) {
  typedef T v2 __attribute__((ext_vector_type(2)));
  *reinterpret_cast<v2 *>(H + 2 * lane) = v2{v[0], v[1]};
  *reinterpret_cast<v2 *>(H + 128 + 2 * lane) = v2{v[2], v[3]};
}

template <typename T>
__global__ void __launch_bounds__(K2_THREADS) __attribute__((amdgpu_waves_per_eu(4))) k_dia_k2_off(DK2Args<T> A) {
  typedef Mma<T> MM;
  typedef typename MM::acc_t acc_t;
  typedef acc_t vec;
  __shared__ T Hs[K2_SLOTS * TILE2];  // slot tiles H in result order (the next product's Y operand)
  const int w = blockIdx.x;
  const int kq = A.wg[2 * w], ef = A.wg[2 * w + 1];
  if (kq < 0) return;
  const int e = ef / A.Nel, f = ef - e * A.Nel;
  const int k = A.kshell[kq];
  const int t = threadIdx.x, lane = t & 63, g = lane >> 4, c = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int *wrow = A.rows + (kq * K2_WAVES + wv) * K2_ROWS;
  static_assert(K2_ROWS == 3, "row counts dispatched below");
  const int nrow = wrow[2] >= 0 ? 3 : wrow[1] >= 0 ? 2 : 1;
  v4d acc[K2_ROWS];  // one accumulator per owned row
#pragma unroll
  for (int r = 0; r < K2_ROWS; ++r) acc[r] = v4d{0, 0, 0, 0};
  const T *pt = A.pt + (size_t)ef * A.n_src * TILE2;
  const bool up = e > f;
  for (int gi = A.kg[kq]; gi < A.kg[kq + 1]; ++gi) {
    const int ilm = A.gilm[gi], s0 = A.gslot[gi], ns = A.gslot[gi + 1] - s0;
    // the group's factor operands: row side Q of e if e > f else P of e,
    // column side the other kind
    const T *te = A.pqo + ((size_t)ilm * A.Nel + e) * 4 * TILE2 + (up ? 2 : 0) * TILE2;
    const T *tf = A.pqo + ((size_t)ilm * A.Nel + f) * 4 * TILE2 + (up ? 0 : 2) * TILE2;
    const vec b0 = *reinterpret_cast<const vec *>(tf + lane * 4);
    const vec b2 = *reinterpret_cast<const vec *>(tf + TILE2 + lane * 4);
    T rho = T(1);
    if constexpr (sizeof(T) == 4) {
      // FP32 tiles hold P / s and Q * s per (ilm, element): restore the
      // pair's Q(e) P(f) or P(e) Q(f) scale, s_f / s_e or s_e / s_f
      const double le = A.lsig[ilm * A.Nel + e], lf = A.lsig[ilm * A.Nel + f];
      rho = (T)exp(up ? lf - le : le - lf);
    }
    __syncthreads();  // the previous group's LDS tiles are no longer read
    for (int sq = wv; sq < ns; sq += K2_WAVES) {
      vec v0 = {0, 0, 0, 0}, v1 = {0, 0, 0, 0};
      const int x1 = A.sl[s0 + sq + 1];
      int x = A.sl[s0 + sq];
      for (; x < x1; x += 4) {  // lists come in fours, padded with zero weights
        vec tv[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) tv[u] = *reinterpret_cast<const vec *>(pt + (unsigned)(A.lt[x + u] * TILE2) + lane * 4);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          v0 += A.ltv[2 * (x + u)] * tv[u];
          v1 -= A.ltv[2 * (x + u) + 1] * tv[u];
        }
      }
      acc_t hh = {0, 0, 0, 0};
#pragma unroll
      for (int s = 0; s < 4; ++s) hh = MM::step(v0[s], b0[s], hh);
#pragma unroll
      for (int s = 0; s < 4; ++s) hh = MM::step(v1[s], b2[s], hh);
      if constexpr (sizeof(T) == 4) hh *= rho;
      h_store<T>(Hs + sq * TILE2, lane, hh);
    }
    const vec a0 = *reinterpret_cast<const vec *>(te + lane * 4);
    const vec a2 = *reinterpret_cast<const vec *>(te + TILE2 + lane * 4);
    __syncthreads();
    const int y1 = A.jo[gi * K2_WAVES + wv + 1];
    const int y = A.jo[gi * K2_WAVES + wv];
    if (y == y1) continue;
    // the wave's rows, 1 to 3: one instantiation each, so no idle row is summed
    auto rows = [&](auto count) {
      constexpr int N = decltype(count)::value;
      vec g0[N], g1[N];
#pragma unroll
      for (int r = 0; r < N; ++r) g0[r] = g1[r] = vec{0, 0, 0, 0};
      for (int q = y; q < y1; q += 2) {  // lists come in twos
        vec hv[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) hv[u] = h_load<T>(Hs + A.js[q + u] * TILE2, lane);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const T *cf = A.jtc + 2 * K2_ROWS * (q + u);
#pragma unroll
          for (int r = 0; r < N; ++r) {
            g0[r] += cf[2 * r] * hv[u];
            g1[r] += cf[2 * r + 1] * hv[u];
          }
        }
      }
#pragma unroll
      for (int r = 0; r < N; ++r) {
        acc_t x = {0, 0, 0, 0};
        if constexpr (sizeof(T) == 8) x = acc[r];
#pragma unroll
        for (int s = 0; s < 4; ++s) x = MM::step(a0[s], g0[r][s], x);  // += i0 G0
#pragma unroll
        for (int s = 0; s < 4; ++s) x = MM::step(a2[s], g1[r][s], x);  // += i2 G1
        if constexpr (sizeof(T) == 8)
          acc[r] = x;
        else
#pragma unroll
          for (int s = 0; s < 4; ++s) acc[r][s] += (double)x[s];
      }
    };
    if (nrow == 3)
      rows(std::integral_constant<int, 3>());
    else if (nrow == 2)
      rows(std::integral_constant<int, 2>());
    else
      rows(std::integral_constant<int, 1>());
  }
  // the owned rows' tiles (lane holds entry (row(g,s), c)) and their mirrors
  const int ni = A.ni[e], nj = A.ni[f], fi = A.first[e], fj = A.first[f];
  const int b = c;
  const long long col = pure_row(A.skip, A.poff, k, fj + min(b, nj - 1));
  const bool scol = (b == 0 && f > 0) || (b == nj - 1 && f + 1 < A.Nel);
#pragma unroll
  for (int r = 0; r < K2_ROWS; ++r) {
    const int j = wrow[r];
    if (j < 0) break;
    const v4d v = acc[r];
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
      const int a = MM::row(g, rr);
      if (a >= ni || b >= nj || col < 0) continue;
      const long long row = pure_row(A.skip, A.poff, j, fi + a);
      if (row < 0) continue;
      const bool srow = (a == 0 && e > 0) || (a == ni - 1 && e + 1 < A.Nel);
      double *dst = A.K + row + col * A.ldk;
      if (srow || scol)
        atomicAdd(dst, -v[rr]);
      else
        *dst = -v[rr];
      if (A.sym) {
        double *mdst = A.K + col + row * A.ldk;
        if (srow || scol)
          atomicAdd(mdst, -v[rr]);
        else
          *mdst = -v[rr];
      }
    }
  }
}

// --- In-element exchange with the Cholesky factors resident in LDS -------------
//
// One 1024-thread workgroup per ((L,|M|), element e, batch of runs of that
// (L,|M|)): the rank x {M0_p, M2_p} channel tiles of (ilm, e) are read once
// into LDS (rows padded to 17 so both the M and M' operand reads are free of
// bank conflicts), then each of the 16 waves takes runs of the batch, gathers
// their density tiles and applies sum_p sigma_p [M0'(R00 M0' - R02 M2') +
// M2'(-R20 M0' + R22 M2')] from LDS.  Runs of one output block sit in
// different workgroups, so the tiles are added to K atomically.  Compared
// with k_dia_k_in (one workgroup per (block, element), factors re-read
// from L2 for every run) this moves the factor traffic from ~100 GB to a few
// GB per N2 build.

constexpr int KL_THREADS = 1024, KL_WAVES = 16, KL_RMAX = KL_RANK_MAX, KL_LD = 17;

template <typename T>
struct DKLArgs {
  const T *P;
  int64_t ldp;
  double *K;
  int64_t ldk;
  int Nel, Nang;
  const int *first, *ni, *skip;
  const long long *poff;
  const T *chol, *sigma;
  const int *chol_off, *chol_rank;
  const int *act_jk, *lrun_tstart;
  const int4 *tpos;
  const T *term_f;
  const int *wg;       // per workgroup: ilm, e, first entry in runs, count (or ilm = -1)
  const int *runs;     // runs grouped by ilm
  const int *run_act;  // output block of each run
  const T *pt;         // tiled density (k_dia_ptile) or null: gather from P
  const int *ttile;
  int n_src;
  int sym;  // symmetric density: runs of blocks j < k also written to the mirror
};

template <typename T, bool TILED>
__global__ void __launch_bounds__(KL_THREADS) k_dia_kin_lds(DKLArgs<T> A) {
  typedef Mma<T> MM;
  typedef typename MM::acc_t acc_t;
  constexpr int TL = TILE * KL_LD;  // one padded 16x16 tile
  __shared__ T Mt[KL_RMAX * 2 * TL];
  __shared__ T sg[KL_RMAX];
  const int w = blockIdx.x;
  const int ilm = A.wg[4 * w], e = A.wg[4 * w + 1], b0 = A.wg[4 * w + 2], nb = A.wg[4 * w + 3];
  if (ilm < 0) return;
  const int rank = A.chol_rank[ilm * A.Nel + e], off = A.chol_off[ilm * A.Nel + e];
  const T *M = A.chol + (size_t)off * 2 * TILE2;
  for (int q = threadIdx.x; q < rank * 2 * TILE2; q += KL_THREADS) {
    const int pc = q / TILE2, u = q - pc * TILE2;  // pc = 2 p + channel
    Mt[pc * TL + (u & 15) + KL_LD * (u >> 4)] = M[q];
  }
  for (int q = threadIdx.x; q < rank; q += KL_THREADS) sg[q] = A.sigma[off + q];
  __syncthreads();
  const int t = threadIdx.x, lane = t & 63, g = lane >> 4, c = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int n = A.ni[e], fe = A.first[e];
  const int rloc = fe + min(c, n - 1);
  int cloc[4], kk[4];
  T cmask[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    kk[s] = MM::row(g, s);
    cloc[s] = fe + min(kk[s], n - 1);
    cmask[s] = (c < n && kk[s] < n) ? T(1) : T(0);
  }
  const T *pt = TILED ? A.pt + (size_t)(e * A.Nel + e) * A.n_src * TILE2 + lane * 4 : nullptr;
  for (int i = wv; i < nb; i += KL_WAVES) {
    const int run = A.runs[b0 + i], act = A.run_act[run];
    T r00[4], r02[4], r20[4], r22[4];
    if constexpr (TILED)
      gather_tiles<T>(pt, A.ttile, A.term_f, A.lrun_tstart[run], A.lrun_tstart[run + 1], r00, r02, r20, r22);
    else
      gather_terms<T>(A.P, A.ldp, A.tpos, A.term_f, A.lrun_tstart[run], A.lrun_tstart[run + 1], rloc, cloc, cmask,
                      r00, r02, r20, r22);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      r02[s] = -r02[s];
      r20[s] = -r20[s];
    }
    acc_t acc = {0, 0, 0, 0}, acc2 = {0, 0, 0, 0};
    // sigma_p = +-1 is applied to the X operands (exact).  The loop stays
    // rolled: the 16 waves of the workgroup keep the matrix pipe busy, and
    // two vectors per step measured no faster.
    for (int p = 0; p < rank; ++p) {
      const T *M0 = Mt + 2 * p * TL, *M2 = M0 + TL;
      const T sp = sg[p];
      T y0[4], y2[4], x0[4], x2[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        y0[s] = M0[c + KL_LD * kk[s]];
        y2[s] = M2[c + KL_LD * kk[s]];
        x0[s] = sp * M0[kk[s] + KL_LD * c];
        x2[s] = sp * M2[kk[s] + KL_LD * c];
      }
      acc_t ya = {0, 0, 0, 0}, yb = {0, 0, 0, 0};
      mma_pair<T>(r00, r20, y0, ya, yb);
      mma_pair<T>(r02, r22, y2, ya, yb);
      mma_pair2<T>(x0, ya, acc, x2, yb, acc2);
    }
    acc += acc2;
    const int jk = A.act_jk[act], j = jk / A.Nang, k = jk - j * A.Nang;
    const long long col = pure_row(A.skip, A.poff, k, fe + c);
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
      const int a = kk[rr];
      if (a >= n || c >= n) continue;
      const long long row = pure_row(A.skip, A.poff, j, fe + a);
      if (row >= 0 && col >= 0) {
        atomicAdd(A.K + row + col * A.ldk, -(double)acc[rr]);
        if (A.sym && j != k) atomicAdd(A.K + col + row * A.ldk, -(double)acc[rr]);
      }
    }
  }
}

// --- In-element exchange with folded dense operators ---------------------------
//
// For one ((L,|M|), element e) the in-element tile of every coupled output
// block is Y(a,b) = sum_xy sum_cd W_xy(ca, bd) R_xy(c,d), x, y the two channels,
// W = B diag(sigma) B' (basis.cpp:1992-2033 contracts the factor) and R_xy =
// sum_i u_x(j,i) V_y(i) the Gaunt-weighted density sums.  W is symmetric under
// c <-> a, under b <-> d and as a matrix, so with tau the transposition of a
// tile the diagonal channels commute with tau and W_20 = tau W_02 tau: the
// symmetric and antisymmetric parts of Y separate,
//   Y_s (a <= b) = Ts [S_00; S_22; R_02 + R_20'],   S = R + R' (R on the diagonal)
//   Y_a (a <  b) = Ta [A_00; A_22; R_02 - R_20'],   A = R - R'
// 120 x 465 and 105 x 435 for 15 functions: 0.20 MFLOP per (block, element)
// against 0.41 of the plain operators and 12 r n^3 = 1.2 of the Cholesky form
// (rank r ~ 30).  k_dia_fold_build writes Ts, Ta once per basis in operand order
// (row tile, four k-steps, lane, step).
// k_dia_kin_fold: one 1024-thread workgroup per ((L,|M|), e, 16 units of two
// rows), a GEMM with 32 columns.  Each wave gathers its unit's R tiles (the two
// rows share the slots' V tiles), folds them in registers (lanes c <= d keep
// the symmetric entries, the others the antisymmetric ones) and stores the
// symmetric, then the antisymmetric columns in LDS (120 KB); the waves split
// row tiles and, beyond those, the inner extent; the operator streams from L2
// one quad of k-steps ahead.  Column c of inner index k sits at (c + k/2) & 15,
// which keeps stores (many k, one column) and reads (four k, all columns) free
// of bank conflicts.  The tiles are added to K atomically (boundary entries are
// shared with the cross-element launch, the (L,|M|) of a block with other
// workgroups).
// N2 (lmax 16, 8 elements, 60 k rows x 8 elements): 4.2 ms against 13.0 of
// k_dia_kin_lds, FP32 (lmax 12, 6 elements) 1.0 against 2.1; 1.6 ms of it the
// matrix pipe's, the gathers 0.65, the output 0.55, the folding the rest (one
// workgroup per CU, its phases one after another).

template <typename T>
struct DFoldBuildArgs {
  const double *chol, *sigma;
  const int *chol_off, *chol_rank, *ni, *fexp;
  int Nel;
  size_t size, x0;  // x0: first ilm*Nel + e of the launch
  T *out;           // [ilm*Nel + e][size]
  double *scale;    // [ilm*Nel + e]
};

// q-th pair a <= b (anti: a < b) in the order b (b + 1) / 2 + a (b (b - 1) / 2 + a)
__device__ inline void fold_pair(int q, bool anti, int &a, int &b) {
  b = anti ? 1 : 0;
  for (int first = 0, w = 1; q >= first + w; ++b) {
    first += w;
    ++w;
  }
  a = q - (anti ? b * (b - 1) / 2 : b * (b + 1) / 2);
}

// Workgroups ((ilm, e), one of FB_PARTS shares of the row tiles); the channel
// tiles sit in LDS when the rank allows (LDS), else they are read in place.
// |W(ca,bd)| <= max sum_p B_p^2 over the channels' entries (Cauchy-Schwarz), so
// T is stored divided by that bound's power of two.  Bound by LDS reads (two per product and vector); N2: 1792 operators of 0.9 MB
// in 3 ms (21 ms with the tiles read from L2).
constexpr int FB_THREADS = 1024, FB_PARTS = 4;

template <bool LDS, typename T>
__global__ void __launch_bounds__(FB_THREADS) k_dia_fold_build(DFoldBuildArgs<T> A) {
  __shared__ double Ml[LDS ? KL_RANK_MAX * 2 * TILE2 : 1];
  __shared__ double sgl[LDS ? KL_RANK_MAX : 1];
  __shared__ int2 pairs[2][TILE * (TILE + 1) / 2];
  const size_t x = A.x0 + blockIdx.y;
  const int e = (int)(x % A.Nel), n = A.ni[e];
  const int rank = A.chol_rank[x], off = A.chol_off[x];
  const double *Mg = A.chol + (size_t)off * 2 * TILE2, *sg = A.sigma + off;
  if (LDS) {
    for (int q = threadIdx.x; q < rank * 2 * TILE2; q += FB_THREADS) Ml[q] = Mg[q];
    for (int q = threadIdx.x; q < rank; q += FB_THREADS) sgl[q] = sg[q];
  }
  for (int q = threadIdx.x; q < 2 * kf_pairs(n, false); q += FB_THREADS) {
    const bool anti = q >= kf_pairs(n, false);
    const int r = anti ? q - kf_pairs(n, false) : q;
    int a, b;
    if (!anti || r < kf_pairs(n, true)) {
      fold_pair(r, anti, a, b);
      pairs[anti][r] = make_int2(a, b);
    }
  }
  __syncthreads();
  const double *M = LDS ? Ml : Mg, *sv = LDS ? sgl : sg;
  double top = 0.0;
  for (int q = threadIdx.x; q < 2 * TILE2; q += FB_THREADS) {  // zero outside the element
    double v = 0.0;
    for (int p = 0; p < rank; ++p) v += M[p * 2 * TILE2 + q] * M[p * 2 * TILE2 + q];
    top = fmax(top, v);
  }
  __shared__ double red[FB_THREADS / 64];
  for (int o = 32; o > 0; o >>= 1) top = fmax(top, __shfl_xor(top, o));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = top;
  __syncthreads();
  for (int w = 0; w < FB_THREADS / 64; ++w) top = fmax(top, red[w]);
  const int ex = top > 0.0 && top < HUGE_VAL ? ilogb(top) : 0;
  const double down = ldexp(1.0, -ex);
  if (blockIdx.x == 0 && threadIdx.x == 0) A.scale[x] = ldexp(1.0, ex - A.fexp[x / A.Nel]);
  // sum_p sigma_p Mx(c,a) My(b,d) + sn sum_p sigma_p Mx(c2,a2) My(b2,d2)
  auto two = [&](int cx, int cy, int o1, int o2, int o3, int o4, double sn) {
    const double *p1 = M + cx * TILE2 + o1, *p2 = M + cy * TILE2 + o2, *p3 = M + cx * TILE2 + o3,
                 *p4 = M + cy * TILE2 + o4;
    double v = 0.0, w = 0.0;
    for (int p = 0; p < rank; ++p) {
      const int q = p * 2 * TILE2;
      v += sv[p] * p1[q] * p2[q];
      w += sv[p] * p3[q] * p4[q];
    }
    return v + sn * w;
  };
  auto at = [](int r, int c) { return r + TILE * c; };
  const int rs = kf_tiles(n, false), ra = kf_tiles(n, true);
  for (int tile = blockIdx.x; tile < rs + ra; tile += FB_PARTS) {
    const bool anti = tile >= rs;
    const int rt = anti ? tile - rs : tile;
    const int np = kf_pairs(n, anti), K = kf_inner(n, anti);
    const double sn = anti ? -1.0 : 1.0;
    T *out = A.out + x * A.size + (anti ? (size_t)16 * rs * kf_inner(n, false) : 0) + (size_t)16 * rt * K;
    for (int q = threadIdx.x; q < 16 * K; q += FB_THREADS) {
      const int quad = q >> 8, lane = (q >> 2) & 63, st = q & 3;
      const int row = 16 * rt + (lane & 15), k = 16 * quad + 4 * st + (lane >> 4);
      double v = 0.0;
      if (row < np && k < 2 * np + n * n) {
        const int a = pairs[anti][row].x, b = pairs[anti][row].y;
        if (k < 2 * np) {
          const int ch = k >= np;
          const int c = pairs[anti][k - ch * np].x, d = pairs[anti][k - ch * np].y;
          v = two(ch, ch, at(c, a), at(b, d), at(d, a), at(b, c), sn);
          // c == d (symmetric half only): one entry, and both sums are it
          v *= 0.5;
        } else {
          const int c = (k - 2 * np) % n, d = (k - 2 * np) / n;
          v = 0.5 * two(0, 1, at(c, a), at(b, d), at(c, b), at(a, d), sn);
        }
      }
      out[q] = (T)(v * down);
    }
  }
}

template <typename T>
struct DFoldArgs {
  double *K;
  int64_t ldk;
  int Nel, Nang;
  const int *first, *ni, *skip;
  const long long *poff;
  const T *Top;
  size_t size;
  const double *scale;
  const int4 *wg;
  const int *jk, *ent;
  const int4 *rec, *more;
  const T *u, *v;
  const T *pt;  // tiled density
  int n_src;
  int sym;
};

// V0, V1 of one slot: sources in runs of consecutive tiles, four loads in
// flight (a run's weights are padded with zeros; the padding rereads its last tile).
template <typename T>
__device__ inline void slot_sums(const T *pt, int4 r, const int4 *more, const T *v, int lane,
                                 typename Mma<T>::acc_t &v0, typename Mma<T>::acc_t &v1) {
  typedef typename Mma<T>::acc_t vec;
  v0 = v1 = vec{0, 0, 0, 0};
  for (;;) {
    for (int x = 0; x < r.y; x += 4) {
      vec tv[4];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        tv[u] = *reinterpret_cast<const vec *>(pt + (size_t)(r.x + min(x + u, r.y - 1)) * TILE2 + lane * 4);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        v0 += v[2 * (r.z + x + u)] * tv[u];
        v1 += v[2 * (r.z + x + u) + 1] * tv[u];
      }
    }
    if (r.w < 0) break;
    r = more[r.w];
  }
}

// One half (symmetric or antisymmetric) of the GEMM: the wave's row tile rt
// over the quads [q0, q1) and both column tiles.  Every quad's 16 products are a
// sum of their own.  One chain of matrix instructions over up to 480 products, whose
// two channels cancel, was further off than the Cholesky form: R = 6, l <= 3, 6
// elements of 15 functions, FP32 1.6 times its error (now 0.69), FP64 against 64-bit
// sums 1.9e-15 (now 1.65e-15, Cholesky form 1.7e-15).  N2 10.58 -> 10.74 ms, FP32
// (lmax 12, 6 elements) 2.08 -> 2.11 ms; the FP32 parts added in FP64 0.56 times, but
// 2.15 ms.
template <typename T>
__device__ inline void fold_gemm(const T *top, const T *X, int rt, int nq, int q0, int q1, int lane,
                                 typename Mma<T>::acc_t sum[2]) {
  typedef Mma<T> MM;
  typedef typename MM::acc_t vec;
  const int g = lane >> 4, c = lane & 15;
  const T *tp = top + (size_t)rt * nq * 256 + lane * 4;
  const T *Xg = X + g * 16;
  vec cur = *reinterpret_cast<const vec *>(tp + (size_t)q0 * 256);
  for (int q = q0; q < q1; ++q) {
    const vec nxt = *reinterpret_cast<const vec *>(tp + (size_t)min(q + 1, q1 - 1) * 256);
    vec acc[2] = {vec{0, 0, 0, 0}, vec{0, 0, 0, 0}};
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      const int k = 16 * q + 4 * st;  // + g
      const int pos = k * 16 + ((c + ((k + g) >> 1)) & 15);
      const T b0 = Xg[pos], b1 = Xg[nq * 256 + pos];
      acc[0] = MM::step(cur[st], b0, acc[0]);
      acc[1] = MM::step(cur[st], b1, acc[1]);
    }
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) sum[ct] += acc[ct];
    cur = nxt;
  }
}

template <typename T>
__global__ void __launch_bounds__(KF_THREADS) k_dia_kin_fold(DFoldArgs<T> A) {
  typedef Mma<T> MM;
  typedef typename MM::acc_t vec;
  extern __shared__ char fold_lds[];
  T *X = reinterpret_cast<T *>(fold_lds);
  const int4 wg = A.wg[blockIdx.x];
  const int ilm = wg.x, e = wg.y, u0 = wg.z, nu = wg.w;
  if (ilm < 0) return;
  const int t = threadIdx.x, lane = t & 63, g = lane >> 4, c = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int n = A.ni[e], fe = A.first[e];
  const int nS = kf_pairs(n, false), nA = kf_pairs(n, true);
  const int qS = kf_inner(n, false) / 16, qA = kf_inner(n, true) / 16;
  const int rS = kf_tiles(n, false), rA = kf_tiles(n, true);
  int kk[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) kk[s] = MM::row(g, s);
  // 1. the unit's tiles R_xy(c, kk) = sum u_x V_y of its two rows
  vec r00[KF_ROWS], r02[KF_ROWS], r20[KF_ROWS], r22[KF_ROWS];
#pragma unroll
  for (int r = 0; r < KF_ROWS; ++r) r00[r] = r02[r] = r20[r] = r22[r] = vec{0, 0, 0, 0};
  if (wv < nu) {
    const T *pt = A.pt + (size_t)(e * A.Nel + e) * A.n_src * TILE2;
    for (int q = A.ent[u0 + wv]; q < A.ent[u0 + wv + 1]; ++q) {
      vec v0, v1;
      slot_sums<T>(pt, A.rec[q], A.more, A.v, lane, v0, v1);
#pragma unroll
      for (int r = 0; r < KF_ROWS; ++r) {
        const T c0 = A.u[2 * KF_ROWS * q + 2 * r], c1 = A.u[2 * KF_ROWS * q + 2 * r + 1];
        r00[r] += c0 * v0;
        r02[r] += c0 * v1;
        r20[r] += c1 * v0;
        r22[r] += c1 * v1;
      }
    }
    // 2. fold: transposes through the wave's own 16 x 17 scratch
    T *sc = X + wv * (TILE * 17);
    auto transposed = [&](const vec &r) {
      vec o;
#pragma unroll
      for (int s = 0; s < 4; ++s) sc[kk[s] * 17 + c] = r[s];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int s = 0; s < 4; ++s) o[s] = sc[c * 17 + kk[s]];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      return o;
    };
#pragma unroll
    for (int r = 0; r < KF_ROWS; ++r) {
      const vec t00 = transposed(r00[r]), t22 = transposed(r22[r]), t20 = transposed(r20[r]);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        // c < kk: S(c, kk); c == kk: R; c > kk: A(kk, c)
        const T d00 = c < kk[s] ? t00[s] : T(0), d22 = c < kk[s] ? t22[s] : T(0);
        r00[r][s] = c > kk[s] ? t00[s] - r00[r][s] : r00[r][s] + d00;
        r22[r][s] = c > kk[s] ? t22[s] - r22[r][s] : r22[r][s] + d22;
        const T up = r02[r][s] + t20[s], um = r02[r][s] - t20[s];
        r02[r][s] = up;
        r20[r][s] = um;
      }
    }
  }
  __syncthreads();
  // 3. columns of one half in LDS: X[column tile][k][16]
  auto columns = [&](bool anti) {
    const int np = anti ? nA : nS, nq = anti ? qA : qS;
    if (wv < nu)
#pragma unroll
      for (int r = 0; r < KF_ROWS; ++r) {
        const int col = KF_ROWS * wv + r, cc = col & 15;
        T *Xc = X + (col >> 4) * nq * 256;
        auto put = [&](int k, T x) { Xc[k * 16 + ((cc + (k >> 1)) & 15)] = x; };
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          if (c >= n || kk[s] >= n) continue;
          const int lo = min(c, kk[s]), hi = max(c, kk[s]);
          if (anti ? c > kk[s] : c <= kk[s]) {
            const int p = (anti ? hi * (hi - 1) / 2 : hi * (hi + 1) / 2) + lo;
            put(p, r00[r][s]);
            put(np + p, r22[r][s]);
          }
          put(2 * np + c + n * kk[s], anti ? r20[r][s] : r02[r][s]);
        }
      }
    // the padding of the inner extent meets zero operator entries: keep it finite
    const int k0 = 2 * np + n * n;
    for (int q = t; q < (16 * nq - k0) * 32; q += KF_THREADS)
      X[(q & 1) * nq * 256 + (k0 + (q >> 5)) * 16 + ((q >> 1) & 15)] = T(0);
  };
  const T *top = A.Top + (size_t)(ilm * A.Nel + e) * A.size;
  vec aS[2] = {vec{0, 0, 0, 0}, vec{0, 0, 0, 0}}, aA[2] = {vec{0, 0, 0, 0}, vec{0, 0, 0, 0}};
  // waves: row tile, and a share of the inner extent
  const int kS = KF_WAVES / rS, kA = rA > 0 ? KF_WAVES / rA : 1;
  columns(false);
  __syncthreads();
  const int hS = wv / rS, hA = rA > 0 ? wv / rA : 1;
  if (hS < kS) fold_gemm<T>(top, X, wv - hS * rS, qS, qS * hS / kS, qS * (hS + 1) / kS, lane, aS);
  __syncthreads();
  columns(true);
  __syncthreads();
  if (rA > 0 && hA < kA)
    fold_gemm<T>(top + (size_t)16 * rS * 16 * qS, X, wv - hA * rA, qA, qA * hA / kA, qA * (hA + 1) / kA, lane, aA);
  __syncthreads();
  // 4. partial tiles to LDS (rows rotated as the columns above), then the
  // blocks' entries: Y(a,b) = Y_s + Y_a, Y(b,a) = Y_s - Y_a, scaled back
  const double scale = A.scale[ilm * A.Nel + e];
  T *Ys = X, *Ya = X + kS * rS * 512;
  auto partial = [&](T *Y, int h, int rt, int nr, const vec acc[2]) {
#pragma unroll
    for (int ct = 0; ct < 2; ++ct)
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int row = kk[s];
        Y[((h * nr + rt) * 2 + ct) * 256 + row * 16 + ((c + (row >> 1)) & 15)] = acc[ct][s];
      }
  };
  if (hS < kS) partial(Ys, hS, wv - hS * rS, rS, aS);
  if (rA > 0 && hA < kA) partial(Ya, hA, wv - hA * rA, rA, aA);
  __syncthreads();
  // a wave adds its own rows' blocks; entry x = lo + n hi of the tile, four per
  // lane, the same places for every row, written consecutively in lo both as
  // K(j lo, k hi) and as the mirror K(k lo, j hi) = Y(hi, lo)
  if (wv >= nu) return;
  int lo[4], hi[4], ps[4], pa[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int x = min(lane + 64 * i, n * n - 1);
    hi[i] = x / n;
    lo[i] = lane + 64 * i < n * n ? x - hi[i] * n : -1;
    const int mn = min(max(lo[i], 0), hi[i]), mx = max(lo[i], hi[i]);
    const int p = mx * (mx + 1) / 2 + mn, q = max(mx * (mx - 1) / 2 + mn, 0);
    ps[i] = ((p >> 4) * 512 + (p & 15) * 16) | ((p & 15) >> 1) << 24;  // offset of the row, rotation
    pa[i] = mn == mx ? -1 : (((q >> 4) * 512 + (q & 15) * 16) | ((q & 15) >> 1) << 24);
  }
#pragma unroll
  for (int r = 0; r < KF_ROWS; ++r) {
    const int jk = A.jk[KF_ROWS * (u0 + wv) + r];
    if (jk < 0) break;
    const int j = jk / A.Nang, k = jk - j * A.Nang;
    const int col = KF_ROWS * wv + r, ct = (col >> 4) * 256, cc = col & 15;
    const int sj = A.skip[j], sk = A.skip[k];
    const long long oj = A.poff[j] + fe - sj, ok = A.poff[k] + fe - sk;
    const bool both = A.sym && j != k;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (lo[i] < 0) continue;
      const int os = (ps[i] & 0xffffff) + ct + ((cc + (ps[i] >> 24)) & 15);
      double vs = 0.0, va = 0.0;
      for (int h = 0; h < kS; ++h) vs += (double)Ys[os + h * rS * 512];
      if (pa[i] >= 0) {
        const int oa = (pa[i] & 0xffffff) + ct + ((cc + (pa[i] >> 24)) & 15);
        for (int h = 0; h < kA; ++h) va += (double)Ya[oa + h * rA * 512];
      }
      if (lo[i] > hi[i]) va = -va;  // Y(lo, hi) = Y_s + Y_a for lo < hi
      vs *= scale;
      va *= scale;
      if (fe + lo[i] >= sj && fe + hi[i] >= sk) atomicAdd(A.K + (oj + lo[i]) + (ok + hi[i]) * A.ldk, -(vs + va));
      if (both && fe + lo[i] >= sk && fe + hi[i] >= sj)
        atomicAdd(A.K + (ok + lo[i]) + (oj + hi[i]) * A.ldk, -(vs - va));
    }
  }
}

// --- In-element exchange as a dense operator on the matrix cores ---------------
//
// For one ((L,|M|), element e) every coupled output block's in-element tile
// is Y(a,b) = sum_ch sum_cd T_ch((a,b),(c,d)) R_ch(c,d), the four channel
// tiles R_ch the run's Gaunt-weighted density sums and T_ch = sign_ch W~_ch
// with W~ = B diag(sigma) B' (basis.cpp:1992-2033 contracts the same
// factor).  Applied as a GEMM Y (225 x runs) = T (225 x 912) X (912 x runs) it
// costs 2 n^4 per channel and run against 12 r n^3 / 4 of the Cholesky form
// (r ~ 30: 3.4x fewer matrix operations).
//
// k_dia_op_build (before the first exchange) writes T in the matrix-core operand order: for
// k-step ks (inner indices kappa = 4 ks + g, kappa = ch * 228 + c + 15 d) and
// row tile rt (rows rho = 16 rt + c, rho = a + 15 b), lane (g, c) holds
// T(rho, kappa); one aligned 512-byte read per wave and (ks, rt).
// k_dia_kin_op: one 256-thread workgroup per ((L,|M|), e, up to 16 runs):
// the waves gather the runs' four channel tiles from the tiled density into
// LDS (X[kappa][run], rows padded to 17), then each wave multiplies its row
// tiles of T (streamed from L2: the workgroups of one (L,|M|), e) run on one
// XCD) by X on the FP64 matrix cores and adds the tiles into K atomically
// (boundary rows shared with other launches; other (L,|M|) of the block in
// other workgroups), with the mirror of a symmetric density as k_dia_kin_lds.

constexpr int OP_NC = 16, OP_KC = 228, OP_K = 4 * OP_KC, OP_KS = OP_K / 4, OP_RT = 15, OP_XLD = 17;
constexpr size_t OP_TSIZE = (size_t)OP_KS * OP_RT * 64;  // doubles of one (ilm, element) operator

struct DOpBuildArgs {
  const double *chol, *sigma;
  const int *chol_off, *chol_rank, *ni;
  int Nel;
  double *T;  // [ilm*Nel + e][OP_TSIZE]
};

__global__ void __launch_bounds__(NT) k_dia_op_build(DOpBuildArgs A) {
  const int x = blockIdx.x / OP_KS, ks = blockIdx.x - x * OP_KS;
  const int e = x % A.Nel, n = A.ni[e];
  const int rank = A.chol_rank[x], off = A.chol_off[x];
  const double *M = A.chol + (size_t)off * 2 * TILE2;
  double *out = A.T + (size_t)x * OP_TSIZE + (size_t)ks * OP_RT * 64;
  for (int q = threadIdx.x; q < OP_RT * 64; q += NT) {
    const int rt = q >> 6, lane = q & 63, g = lane >> 4, c = lane & 15;
    const int rho = 16 * rt + c, kap = 4 * ks + g;
    const int ch = kap / OP_KC, kc = kap - ch * OP_KC;
    const int cc = kc % 15, dd = kc / 15, a = rho % 15, b = rho / 15;
    double v = 0.0;
    if (rho < 225 && kc < 225 && a < n && b < n && cc < n && dd < n) {
      // B(xo + cc + a n, p) B(yo + b + dd n, p): channel block x of M_p at (cc, a), y at (b, dd)
      const int xo = ch >> 1, yo = ch & 1;
      for (int p = 0; p < rank; ++p) {
        const double *Mp = M + (size_t)p * 2 * TILE2;
        v += A.sigma[off + p] * Mp[xo * TILE2 + cc + TILE * a] * Mp[yo * TILE2 + b + TILE * dd];
      }
      if (ch == 1 || ch == 2) v = -v;
    }
    out[q] = v;
  }
}

struct DOpArgs {
  double *K;
  int64_t ldk;
  int Nel, Nang;
  const int *first, *ni, *skip;
  const long long *poff;
  const double *T;
  const int *act_jk, *lrun_tstart;
  const double *term_f;
  const int *wg;       // per workgroup: ilm, e, first entry in runs, count (or ilm = -1)
  const int *runs, *run_act;
  const double *pt;    // tiled density
  const int *ttile;
  int n_src;
  int sym;
};

__global__ void __launch_bounds__(NT) k_dia_kin_op(DOpArgs A) {
  __shared__ double X[OP_K * OP_XLD];
  const int w = blockIdx.x;
  const int ilm = A.wg[4 * w], e = A.wg[4 * w + 1], b0 = A.wg[4 * w + 2], nb = A.wg[4 * w + 3];
  if (ilm < 0) return;
  const int t = threadIdx.x, lane = t & 63, g = lane >> 4, c = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int n = A.ni[e], fe = A.first[e];
  for (int q = t; q < OP_K * OP_XLD; q += NT) X[q] = 0.0;
  __syncthreads();
  const double *pt = A.pt + (size_t)(e * A.Nel + e) * A.n_src * TILE2 + lane * 4;
  for (int i = wv; i < nb; i += NT / 64) {
    const int run = A.runs[b0 + i];
    double r[4][4];
    gather_tiles<double>(pt, A.ttile, A.term_f, A.lrun_tstart[run], A.lrun_tstart[run + 1], r[0], r[1], r[2],
                         r[3]);
    // lane (g, c) holds R_ch(c, kk) in entry s, kk = row(g, s): kappa = ch * 228 + c + 15 kk
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int kk = Mma<double>::row(g, s);
      if (c < n && kk < n)
#pragma unroll
        for (int ch = 0; ch < 4; ++ch) X[(ch * OP_KC + c + 15 * kk) * OP_XLD + i] = r[ch][s];
    }
  }
  __syncthreads();
  // row tiles wv, wv + 4, wv + 8, wv + 12 (< 15)
  const int nrt = wv < 3 ? 4 : 3;
  v4d acc[4] = {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}};
  // One wave per SIMD (the X tile takes the LDS): the operator reads are
  // issued OP_PF k-steps ahead so their L2 latency hides behind the matrix work.
  constexpr int OP_PF = 4;
  static_assert(OP_KS % OP_PF == 0, "k-steps in whole prefetch rounds");
  const double *Tx = A.T + (size_t)(ilm * A.Nel + e) * OP_TSIZE + lane + (size_t)wv * 64;
  double abuf[OP_PF][4];
#pragma unroll
  for (int u = 0; u < OP_PF; ++u)
#pragma unroll
    for (int j = 0; j < 4; ++j) abuf[u][j] = j < nrt ? Tx[(size_t)u * OP_RT * 64 + 4 * j * 64] : 0.0;
  for (int ks0 = 0; ks0 < OP_KS; ks0 += OP_PF) {
#pragma unroll
    for (int u = 0; u < OP_PF; ++u) {
      const int ks = ks0 + u;
      const double bv = X[(4 * ks + g) * OP_XLD + c];
      double av[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) av[j] = abuf[u][j];
      if (ks + OP_PF < OP_KS) {
        const double *Tn = Tx + (size_t)(ks + OP_PF) * OP_RT * 64;
#pragma unroll
        for (int j = 0; j < 4; ++j) abuf[u][j] = j < nrt ? Tn[4 * j * 64] : 0.0;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (j < nrt) acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[j], bv, acc[j], 0, 0, 0);
    }
  }
  // lane (g, c) holds Y(rho = 16 rt + g + 4 r, run c) in acc[j][r]
  if (c >= nb) return;
  const int run = A.runs[b0 + c], act = A.run_act[run];
  const int jk = A.act_jk[act], j = jk / A.Nang, k = jk - j * A.Nang;
#pragma unroll
  for (int jj = 0; jj < 4; ++jj) {
    if (jj >= nrt) break;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int rho = 16 * (wv + 4 * jj) + g + 4 * r;
      const int a = rho % 15, b = rho / 15;
      if (rho >= 225 || a >= n || b >= n) continue;
      const long long row = pure_row(A.skip, A.poff, j, fe + a), col = pure_row(A.skip, A.poff, k, fe + b);
      if (row < 0 || col < 0) continue;
      atomicAdd(A.K + row + col * A.ldk, -acc[jj][r]);
      if (A.sym && j != k) atomicAdd(A.K + col + row * A.ldk, -acc[jj][r]);
    }
  }
}

// --- In-element exchange as a dense operator ----------------------------------
//
// For one ((L,|M|), element e) the in-element exchange of every output block
// coupled to it is Y(a,b) = sum_ch sum_cd T_ch((a,b),(c,d)) R_ch(c,d), R_ch the
// Gaunt-weighted density tiles of that block: a GEMM Y (256 x runs) =
// T (256 x 4 KC) X (4 KC x runs), run on the f64 matrix cores.  X is formed in
// LDS one channel at a time from the screened terms.  Partial tiles go to
// Ypart[run][e]; k_dia_kin_reduce sums them per output block.

constexpr int NCOL = 32;  // runs (GEMM columns) per workgroup

struct DKInArgs {
  const double *P;
  int64_t ldp;
  int Nel, Nang;
  const int *first, *ni, *skip;
  const long long *poff;
  const double *T;
  const int *wg, *ilm_rstart, *ilm_runs, *lrun_tstart, *term_il;
  const double *term_f;
  double *Y;
};

__global__ void __launch_bounds__(NT) k_dia_kin_gemm(DKInArgs A) {
  const int w = blockIdx.x;
  const int ilm = A.wg[3 * w], e = A.wg[3 * w + 1], c0 = A.wg[3 * w + 2];
  if (ilm < 0) return;
  const int r0 = A.ilm_rstart[ilm] + c0, r1 = min(A.ilm_rstart[ilm + 1], r0 + NCOL);
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6, g = lane >> 4, c = lane & 15;
  const int n = A.ni[e], fe = A.first[e];
  __shared__ double X[KC * NCOL];
  __shared__ int srun[NCOL];
  if (t < NCOL) srun[t] = r0 + t < r1 ? A.ilm_runs[r0 + t] : -1;
  v4d acc[4][2];
#pragma unroll
  for (int rt = 0; rt < 4; ++rt) acc[rt][0] = acc[rt][1] = v4d{0.0, 0.0, 0.0, 0.0};
  const double *Tb = A.T + (size_t)(ilm * A.Nel + e) * 4 * KC * TILE2;
  const int cc = t % 15, dd = t / 15;
  const bool cdok = t < 225 && cc < n && dd < n;
  for (int ch = 0; ch < 4; ++ch) {
    __syncthreads();
    if (t < KC)
      for (int j = 0; j < NCOL; ++j) {
        const int run = srun[j];
        double v = 0.0;
        if (run >= 0 && cdok)
          for (int q = A.lrun_tstart[run]; q < A.lrun_tstart[run + 1]; ++q) {
            const int il = A.term_il[q], i = il / A.Nang, l = il - i * A.Nang;
            const long long row = pure_row(A.skip, A.poff, i, fe + cc), col = pure_row(A.skip, A.poff, l, fe + dd);
            if (row >= 0 && col >= 0) v += A.term_f[4 * q + ch] * A.P[row + col * A.ldp];
          }
        X[t * NCOL + j] = v;
      }
    __syncthreads();
    const double *Tc = Tb + (size_t)ch * KC * TILE2 + 64 * wv + c;
    for (int ks = 0; ks < KC / 4; ++ks) {
      const int k = 4 * ks + g;
      const double b0 = X[k * NCOL + c], b1 = X[k * NCOL + 16 + c];
      const double *Tk = Tc + (size_t)k * TILE2;
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        const double a = Tk[16 * rt];
        acc[rt][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b0, acc[rt][0], 0, 0, 0);
        acc[rt][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b1, acc[rt][1], 0, 0, 0);
      }
    }
  }
  // lane (g, c) holds Y(64 wv + 16 rt + g + 4 r, 16 ct + c) in component r
#pragma unroll
  for (int ct = 0; ct < 2; ++ct) {
    const int run = srun[16 * ct + c];
    if (run < 0) continue;
    double *out = A.Y + ((size_t)run * A.Nel + e) * TILE2 + 64 * wv + g;
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int r = 0; r < 4; ++r) out[16 * rt + 4 * r] = acc[rt][ct][r];
  }
}

struct DKRedArgs {
  double *K;
  int64_t ldk;
  int Nel, Nang;
  const int *first, *ni, *skip;
  const long long *poff;
  const int *act_jk, *act_lstart;
  const double *Y;
};

// One workgroup per (active output block, element): K tile = -sum over the
// block's runs of the partial tiles, shared boundary rows/cols accumulated
// atomically (the cross-element launch adds into the same entries).
__global__ void __launch_bounds__(NT) k_dia_kin_reduce(DKRedArgs A) {
  const int act = blockIdx.x / A.Nel, e = blockIdx.x - act * A.Nel;
  const int t = threadIdx.x, a = t & 15, b = t >> 4;
  const int n = A.ni[e], fe = A.first[e];
  if (a >= n || b >= n) return;
  const int jk = A.act_jk[act], j = jk / A.Nang, k = jk - j * A.Nang;
  const long long row = pure_row(A.skip, A.poff, j, fe + a), col = pure_row(A.skip, A.poff, k, fe + b);
  if (row < 0 || col < 0) return;
  double v = 0.0;
  for (int run = A.act_lstart[act]; run < A.act_lstart[act + 1]; ++run)
    v += A.Y[((size_t)run * A.Nel + e) * TILE2 + t];
  const bool srow = (a == 0 && e > 0) || (a == n - 1 && e + 1 < A.Nel);
  const bool scol = (b == 0 && e > 0) || (b == n - 1 && e + 1 < A.Nel);
  double *dst = A.K + row + col * A.ldk;
  if (srow || scol)
    atomicAdd(dst, -v);
  else
    *dst = -v;
}

// K(-mj,-mk) = K(mj,mk) for a +-m symmetric density (basis.cpp:2067-2086):
// one workgroup per mirrored shell block; m != 0 on both sides, so both
// blocks hold (Nrad-1) x (Nrad-1) pure entries.
__global__ void __launch_bounds__(NT) k_dia_mirror(double *K, int64_t ldk, int Nrad, const long long *poff,
                                                    const int *mirror, int Nang) {
  const int dst = mirror[2 * blockIdx.x], src = mirror[2 * blockIdx.x + 1];
  const int jd = dst / Nang, kd = dst - jd * Nang, js = src / Nang, ks = src - js * Nang;
  const int n = Nrad - 1;
  for (int q = threadIdx.x; q < n * n; q += NT) {
    const int cc = q / n, rr = q - cc * n;
    K[(poff[jd] + rr) + (poff[kd] + cc) * ldk] = K[(poff[js] + rr) + (poff[ks] + cc) * ldk];
  }
}

}  // namespace

namespace {
// P/Q tiles in matrix-core operand order (FP64 lanes), each with its half of the
// power of two that the lists' coupling factors carry.
__global__ void __launch_bounds__(NT) k_pq_operands(const double *pq, const int *fexp, double *pqo, int Nel) {
  const size_t o = (size_t)blockIdx.x * TILE2;
  const int u = threadIdx.x, lane = u >> 2;
  const double f = ldexp(1.0, -fexp[blockIdx.x / (4 * Nel)] / 2);
  pqo[o + u] = f * pq[o + (lane & 15) + TILE * Mma<double>::row(lane >> 4, u & 3)];
}
}  // namespace

namespace {
template <typename T>
void fold_build(DiatomicDevice &d, DevArray<T> &out, hipStream_t s) {
  const size_t nx = (size_t)d.n_lm * d.Nel, size = kf_size(d.fold_n);
  out.alloc(nx * size);
  d.kf_scale.alloc(nx);
  const size_t step = (size_t)(65535 / d.Nel) * d.Nel;  // whole (L,|M|) within the grid's y limit
  for (size_t x = 0; x < nx; x += step) {
    const unsigned cnt = (unsigned)std::min(step, nx - x);
    DFoldBuildArgs<T> a{d.chol.p, d.sigma.p, d.chol_off.p, d.chol_rank.p, d.ni.p, d.fexp.p, d.Nel, size, x,
                        out.p, d.kf_scale.p};
    if (d.max_rank <= KL_RANK_MAX)
      hipLaunchKernelGGL((k_dia_fold_build<true, T>), dim3(FB_PARTS, cnt), dim3(FB_THREADS), 0, s, a);
    else
      hipLaunchKernelGGL((k_dia_fold_build<false, T>), dim3(FB_PARTS, cnt), dim3(FB_THREADS), 0, s, a);
    hip_check(hipGetLastError(), "diatomic_fold_build");
  }
}
}  // namespace

bool diatomic_fold_ready(DiatomicDevice &d, bool fp32, bool allowed, hipStream_t s) {
  int &state = d.fold_state[fp32];
  if (state == 0) {
    state = -1;
    if (d.fold_form && allowed) {
      size_t fr = 0, tot = 0;
      hip_check(hipMemGetInfo(&fr, &tot), "hipMemGetInfo");
      double budget = fr / 4;  // keep three quarters of the free memory for densities and tiles
      if (const char *env = std::getenv("HFGPU_EXCHANGE_FOLD_GIB")) budget = std::atof(env) * (1ull << 30);
      const double bytes =
          (double)d.n_lm * d.Nel * kf_size(d.fold_n) * (fp32 ? sizeof(float) : sizeof(double));
      if (bytes <= budget) try {
          if (fp32)
            fold_build(d, d.Tfold32, s);
          else
            fold_build(d, d.Tfold, s);
          state = 1;
        } catch (const Error &e) {
          if (e.code != -4) throw;  // no room after all: the Cholesky form needs none
          (void)hipGetLastError();
          (void)(fp32 ? d.Tfold32.release() : d.Tfold.release());
        }
    }
  }
  return state == 1;
}

void diatomic_op_build(DiatomicDevice &d, const std::vector<int> &ni, hipStream_t s) {
  d.pqo.alloc(d.pq.n);
  static_assert(NT == TILE2, "one thread per tile entry");
  const size_t nx = (size_t)d.n_lm * d.Nel;
  if (nx) {
    hipLaunchKernelGGL(k_pq_operands, dim3((unsigned)(4 * nx)), dim3(NT), 0, s, d.pq.p, d.fexp.p, d.pqo.p, d.Nel);
    hip_check(hipGetLastError(), "pq_operands");
  }
  d.op_in = d.fold_form = d.fold_in = false;
  d.fold_state[0] = d.fold_state[1] = 0;
  d.Top2.release();
  d.Tfold.release();
  d.Tfold32.release();
  if (nx == 0 || d.max_rank > 2 * TILE2) return;
  const char *env = std::getenv("HFGPU_EXCHANGE_OP");
  if (env && std::atoi(env) == 0) return;
  if (env) {
    size_t fr = 0, tot = 0;
    hip_check(hipMemGetInfo(&fr, &tot), "hipMemGetInfo");
    // on N2 (lmax 16) slower than the Cholesky-form kernel (16.2 against 13.1
    // ms): each workgroup streams its 1.75 MB operator for 16 runs
    if (nx * OP_TSIZE * sizeof(double) > fr / 4) return;  // keep three quarters of the free memory
    d.Top2.alloc(nx * OP_TSIZE);
    DOpBuildArgs a{d.chol.p, d.sigma.p, d.chol_off.p, d.chol_rank.p, d.ni.p, d.Nel, d.Top2.p};
    hipLaunchKernelGGL(k_dia_op_build, dim3((unsigned)(nx * OP_KS)), dim3(NT), 0, s, a);
    hip_check(hipGetLastError(), "diatomic_op_build");
    d.op_in = true;
    return;
  }
  d.fold_n = *std::max_element(ni.begin(), ni.end());
  d.fold_form = true;
}

void diatomic_coulomb_launch(const DiatomicDevice &d, const double *P, int64_t ldp, double *J, int64_t ldj,
                             hipStream_t s, KernelTimer *timer) {
  if (d.n_LM == 0) {
    fill_zero_launch(J, d.Nbf, d.Nbf, ldj, s);
    return;
  }
  DJArgs a{P, ldp, d.Nel, d.Nang, d.first.p, d.ni.p, d.skip.p, d.poff.p, d.pq.p, d.chol.p, d.sigma.p,
           d.chol_off.p, d.chol_rank.p, d.LM_ilm.p, d.LM_fac.p, d.pstart.p, d.pair_kl.p, d.pair_c.p,
           d.Jin.p, d.ds.p, d.db.p, d.n_LM};
  {
    TimedLaunch tl(timer, "diatomic_j_gather", s);
    hipLaunchKernelGGL(k_dia_j_gather, dim3(8 * xcd_share(d.n_LM * d.Nel)), dim3(NT), 0, s, a);
    hip_check(hipGetLastError(), "diatomic_j_gather");
  }
  DJBandArgs w{d.Nel, d.LM_ilm.p, d.pq.p, d.ds.p, d.db.p, d.Jin.p};
  hipLaunchKernelGGL(k_dia_j_band, dim3(d.n_LM * d.Nel), dim3(NT), 0, s, w);
  hip_check(hipGetLastError(), "diatomic_j_band");
  DJOutArgs o{J, ldj, d.Nel, d.Nang, d.first.p, d.ni.p, d.skip.p, d.poff.p, d.Jin.p, d.out_start.p, d.out_q.p,
              d.out_c.p};
  {
    TimedLaunch tl(timer, "diatomic_j_expand", s);
    hipLaunchKernelGGL(k_dia_j_expand, dim3(8 * xcd_share(d.Nang * d.Nang * d.Nel)), dim3(NT), 0, s, o);
    hip_check(hipGetLastError(), "diatomic_j_expand");
  }
}

int block_stats_chunks(int Nrad) { return (Nrad + 31) / 32; }

void block_stats_batch_launch(const StatsArgs *d_args, const int *d_start, int n, int total_wg, hipStream_t s) {
  if (total_wg <= 0) return;
  hipLaunchKernelGGL(k_block_stats_batch, dim3(total_wg), dim3(NT), 0, s, d_args, d_start, n);
  hip_check(hipGetLastError(), "block_stats_batch");
}

void block_stats_launch(const double *P, int64_t ldp, int Nrad, int Nang, const int *skip, const long long *poff,
                        double *d_part, double *h_part, hipStream_t s) {
  const int nch = block_stats_chunks(Nrad);
  hipLaunchKernelGGL(k_block_stats, dim3(Nang * Nang, nch), dim3(NT), 0, s, P, ldp, Nrad, Nang, skip, poff, d_part);
  hip_check(hipGetLastError(), "block_stats");
  hip_check(hipMemcpyAsync(h_part, d_part, sizeof(double) * 4 * nch * Nang * Nang, hipMemcpyDeviceToHost, s),
            "copy block statistics");
}

bool block_stats_reduce(const double *h_part, int Nrad, int Nang, double *bnorm) {
  const int nch = block_stats_chunks(Nrad);
  double amax = 0.0, pmax = 0.0;
  for (int i = 0; i < Nang; ++i)
    for (int l = i; l < Nang; ++l) {  // only the pairs i <= l are written
      const double *o = h_part + (size_t)(i * Nang + l) * nch * 4;
      double sa = 0.0, sb = 0.0;
      for (int c = 0; c < nch; ++c) {
        sa += o[4 * c];
        sb += o[4 * c + 1];
        amax = std::max(amax, o[4 * c + 2]);
        pmax = std::max(pmax, o[4 * c + 3]);
      }
      bnorm[i * Nang + l] = std::sqrt(sa);
      if (i != l) bnorm[l * Nang + i] = std::sqrt(sb);
    }
  return amax <= 1e-14 * pmax;
}

bool symmetric_exchange_allowed() {
  const char *env = std::getenv("HFGPU_EXCHANGE_SYMMETRIC");
  return !(env && std::atoi(env) == 0);
}

namespace {
template <typename T>
void launch_dia_k(int part, bool tiled, int64_t grid, hipStream_t s, const DKArgs<T> &a) {
  const dim3 gd((unsigned)grid), bd(NT);
  if (part == 0 && tiled)
    hipLaunchKernelGGL((k_dia_k_off<T, true>), gd, bd, 0, s, a);
  else if (part == 0)
    hipLaunchKernelGGL((k_dia_k_off<T, false>), gd, bd, 0, s, a);
  else if (tiled)
    hipLaunchKernelGGL((k_dia_k_in<T, true>), gd, bd, 0, s, a);
  else
    hipLaunchKernelGGL((k_dia_k_in<T, false>), gd, bd, 0, s, a);
}

template <typename T>
void launch_fold(const DiatomicDevice &d, const T *top, const T *u, const T *v, const T *pt, double *K, int64_t ldk,
                 hipStream_t s) {
  const int n = d.fold_n;
  // the columns of one half, or all partial tiles of both, or the transposes' scratch
  size_t lds = (size_t)32 * std::max(kf_inner(n, false), kf_inner(n, true));
  for (int m = 1; m <= n; ++m) {  // elements of any size up to n
    const int a = kf_tiles(m, false), b = kf_tiles(m, true);
    lds = std::max(lds, (size_t)512 * (a * (KF_WAVES / a) + (b ? b * (KF_WAVES / b) : 0)));
  }
  lds = std::max(lds, (size_t)KF_WAVES * TILE * 17) * sizeof(T);
  const void *f = reinterpret_cast<const void *>(&k_dia_kin_fold<T>);
  if (lds > 64 * 1024)
    hip_check(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds), "fold LDS size");
  DFoldArgs<T> a{K, ldk, d.Nel, d.Nang, d.first.p, d.ni.p, d.skip.p, d.poff.p, top, kf_size(n), d.kf_scale.p, d.wg_kf.p, d.kf_jk.p,
                 d.kf_ent.p, d.kf_rec.p, d.kf_more.p, u, v, pt, d.n_src, (int)d.sym};
  hipLaunchKernelGGL(k_dia_kin_fold<T>, dim3(d.n_wg_kf), dim3(KF_THREADS), lds, s, a);
  hip_check(hipGetLastError(), "diatomic_kin_fold");
}

// FP32 copy of the P/Q tiles with P kinds divided and Q kinds multiplied by
// exp(lsig) of their (ilm, element), in storage order and, with their share of the
// coupling factor's power of two, in operand order.
__global__ void k_scale_pq_f32(const double *pq, const double *lsig, const int *fexp, float *pq32, float *pqo32,
                               int n_x, int Nel) {
  const int x = blockIdx.x;
  if (x >= n_x) return;
  const double up = exp(-lsig[x]), dn = exp(lsig[x]), h = ldexp(1.0, -fexp[x / Nel] / 2);
  for (int u = threadIdx.x; u < 4 * TILE2; u += NT) {
    const int kind = u / TILE2, lane = (u & 255) >> 2;
    const size_t o = ((size_t)x * 4 + kind) * TILE2;
    const double f = kind < 2 ? up : dn;
    pq32[(size_t)x * 4 * TILE2 + u] = (float)(pq[(size_t)x * 4 * TILE2 + u] * f);
    pqo32[o + (u & 255)] = (float)(pq[o + (lane & 15) + TILE * Mma<float>::row(lane >> 4, u & 3)] * f * h);
  }
}
}  // namespace

void diatomic_exchange_kernels(DiatomicDevice &d, const double *P, int64_t ldp, double *K, int64_t ldk,
                               hipStream_t s, KernelTimer *timer, bool fp32) {
  fill_zero_launch(K, d.Nbf, d.Nbf, ldk, s);
  if (d.n_act == 0) return;
  if (fp32) {
    if (!d.f32_tables) {
      d.pq32.alloc(d.pq.n);
      d.pqo32.alloc(d.pq.n);
      d.chol32.alloc(d.chol.n);
      d.sigma32.alloc(d.sigma.n);
      const int n_x = d.n_lm * d.Nel;
      hipLaunchKernelGGL(k_scale_pq_f32, dim3(n_x), dim3(NT), 0, s, d.pq.p, d.lsig.p, d.fexp.p, d.pq32.p,
                         d.pqo32.p, n_x, d.Nel);
      hip_check(hipGetLastError(), "scale_pq_f32");
      to_f32_launch(d.chol.p, d.chol32.p, d.chol.n, s);
      to_f32_launch(d.sigma.p, d.sigma32.p, d.sigma.n, s);
      d.f32_tables = true;
    }
    if (d.term_f32_gen != d.list_gen) {
      d.term_f32.alloc(d.term_f.n);
      to_f32_launch(d.term_f.p, d.term_f32.p, d.term_f.n, s);
      if (d.k2) {
        d.k2_ltv32.alloc(d.k2_ltv.n);
        d.k2_jtc32.alloc(d.k2_jtc.n);
        to_f32_launch(d.k2_ltv.p, d.k2_ltv32.p, d.k2_ltv.n, s);
        to_f32_launch(d.k2_jtc.p, d.k2_jtc32.p, d.k2_jtc.n, s);
      }
      if (d.fold_in && d.n_wg_kf > 0) {
        d.kf_u32.alloc(d.kf_u.n);
        d.kf_v32.alloc(d.kf_v.n);
        to_f32_launch(d.kf_u.p, d.kf_u32.p, d.kf_u.n, s);
        to_f32_launch(d.kf_v.p, d.kf_v32.p, d.kf_v.n, s);
      }
      d.term_f32_gen = d.list_gen;
    }
    if (!d.tiled) {
      d.P32.alloc((size_t)d.Nbf * d.Nbf);
      mat_to_f32_launch(P, ldp, d.P32.p, d.Nbf, s);
    }
  }
  if (d.tiled) {
    const int64_t n_tiles = (int64_t)d.Nel * d.Nel * d.n_src, n_wg = (n_tiles + NT / 64 - 1) / (NT / 64);
    if (n_wg > 0x7fffffff) throw Error(-1, "density tile grid too large");
    TimedLaunch tl(timer, fp32 ? "diatomic_ptile_f32" : "diatomic_ptile", s, 0.0);
    if (fp32) {
      d.ptile32.alloc((size_t)n_tiles * TILE2);
      hipLaunchKernelGGL((k_dia_ptile<float>), dim3((unsigned)n_wg), dim3(NT), 0, s, P, ldp, d.Nel, d.first.p,
                         d.ni.p, d.skip.p, d.poff.p, d.Nang, d.src_blk.p, d.n_src, d.ptile32.p);
    } else {
      d.ptile.alloc((size_t)n_tiles * TILE2);
      hipLaunchKernelGGL((k_dia_ptile<double>), dim3((unsigned)n_wg), dim3(NT), 0, s, P, ldp, d.Nel, d.first.p,
                         d.ni.p, d.skip.p, d.poff.p, d.Nang, d.src_blk.p, d.n_src, d.ptile.p);
    }
    hip_check(hipGetLastError(), "diatomic_ptile");
  }
  // two launches: element pairs e != f (disjoint P/Q factors) and the
  // in-element tiles (Cholesky factor); boundary rows/cols shared between
  // neighbouring tiles are accumulated atomically in both
  for (int part = 0; part < 2; ++part) {
    const int n_ef = part == 0 ? d.Nel * (d.Nel - 1) / (d.sym ? 2 : 1) : d.Nel;
    if (n_ef == 0) continue;
    const char *name = part == 0 ? (fp32 ? "diatomic_k_off_f32" : "diatomic_k_off")
                                 : (fp32 ? "diatomic_k_in_f32" : "diatomic_k_in");
    const double flops = part == 0 ? d.flops_off : d.flops_in;
    if (part == 1 && d.dense_in && !fp32) {
      DKInArgs g{P, ldp, d.Nel, d.Nang, d.first.p, d.ni.p, d.skip.p, d.poff.p, d.Top.p, d.wg_in.p,
                 d.ilm_rstart.p, d.ilm_runs.p, d.lrun_tstart.p, d.term_il.p, d.term_f.p, d.Ypart.p};
      DKRedArgs r{K, ldk, d.Nel, d.Nang, d.first.p, d.ni.p, d.skip.p, d.poff.p, d.act_jk.p, d.act_lstart.p,
                  d.Ypart.p};
      TimedLaunch tl(timer, name, s, flops, "k_dia_kin_gemm");
      hipLaunchKernelGGL(k_dia_kin_gemm, dim3(d.n_wg_in), dim3(NT), 0, s, g);
      hip_check(hipGetLastError(), "diatomic_kin_gemm");
      hipLaunchKernelGGL(k_dia_kin_reduce, dim3(d.n_act * d.Nel), dim3(NT), 0, s, r);
      hip_check(hipGetLastError(), "diatomic_kin_reduce");
      continue;
    }
    if (part == 1 && d.fold_in && d.n_wg_kf > 0) {
      TimedLaunch tl(timer, name, s, d.flops_in_kf, "k_dia_kin_fold");
      if (fp32)
        launch_fold<float>(d, d.Tfold32.p, d.kf_u32.p, d.kf_v32.p, d.ptile32.p, K, ldk, s);
      else
        launch_fold<double>(d, d.Tfold.p, d.kf_u.p, d.kf_v.p, d.ptile.p, K, ldk, s);
      continue;
    }
    if (part == 1 && d.op_in && d.tiled && !fp32 && d.n_wg_op > 0) {
      // timed against the Cholesky-form flop count of the same results (the
      // reference's algorithm), so the rate compares with the other form
      TimedLaunch tl(timer, name, s, flops, "k_dia_kin_op");
      DOpArgs a{K, ldk, d.Nel, d.Nang, d.first.p, d.ni.p, d.skip.p, d.poff.p, d.Top2.p, d.act_jk.p,
                d.lrun_tstart.p, d.term_f.p, d.wg_op.p, d.kl_runs.p, d.run_act.p, d.ptile.p, d.term_tile.p,
                d.n_src, (int)d.sym};
      hipLaunchKernelGGL(k_dia_kin_op, dim3(d.n_wg_op), dim3(NT), 0, s, a);
      hip_check(hipGetLastError(), "diatomic_kin_op");
      continue;
    }
    if (part == 1 && d.n_wg_kl > 0) {
      TimedLaunch tl(timer, name, s, flops, "k_dia_kin_lds");
      if (fp32) {
        DKLArgs<float> a{d.P32.p, d.Nbf, K, ldk, d.Nel, d.Nang, d.first.p, d.ni.p, d.skip.p, d.poff.p,
                         d.chol32.p, d.sigma32.p, d.chol_off.p, d.chol_rank.p, d.act_jk.p, d.lrun_tstart.p,
                         d.term_pos.p, d.term_f32.p, d.wg_kl.p, d.kl_runs.p, d.run_act.p,
                         d.tiled ? d.ptile32.p : nullptr, d.term_tile.p, d.n_src, (int)d.sym};
        if (d.tiled)
          hipLaunchKernelGGL((k_dia_kin_lds<float, true>), dim3(d.n_wg_kl), dim3(KL_THREADS), 0, s, a);
        else
          hipLaunchKernelGGL((k_dia_kin_lds<float, false>), dim3(d.n_wg_kl), dim3(KL_THREADS), 0, s, a);
      } else {
        DKLArgs<double> a{P, ldp, K, ldk, d.Nel, d.Nang, d.first.p, d.ni.p, d.skip.p, d.poff.p, d.chol.p,
                          d.sigma.p, d.chol_off.p, d.chol_rank.p, d.act_jk.p, d.lrun_tstart.p, d.term_pos.p,
                          d.term_f.p, d.wg_kl.p, d.kl_runs.p, d.run_act.p,
                          d.tiled ? d.ptile.p : nullptr, d.term_tile.p, d.n_src, (int)d.sym};
        if (d.tiled)
          hipLaunchKernelGGL((k_dia_kin_lds<double, true>), dim3(d.n_wg_kl), dim3(KL_THREADS), 0, s, a);
        else
          hipLaunchKernelGGL((k_dia_kin_lds<double, false>), dim3(d.n_wg_kl), dim3(KL_THREADS), 0, s, a);
      }
      hip_check(hipGetLastError(), "diatomic_kin_lds");
      continue;
    }
    if (part == 0 && d.k2) {
      TimedLaunch tl(timer, name, s, d.flops_off_k2, "k_dia_k2_off");
      if (fp32) {
        DK2Args<float> a{d.ptile32.p, d.n_src, K, ldk, d.Nel, d.Nang, d.first.p, d.ni.p, d.skip.p, d.poff.p,
                         d.pqo32.p, d.lsig.p, d.k2_wg.p, d.k2_kshell.p, d.k2_rows.p, d.k2_kg.p, d.k2_gilm.p,
                         d.k2_gslot.p, d.k2_sl.p, d.k2_lt.p, d.k2_jo.p, d.k2_js.p, d.k2_ltv32.p, d.k2_jtc32.p,
                         (int)d.sym};
        hipLaunchKernelGGL((k_dia_k2_off<float>), dim3(d.n_wg_k2), dim3(K2_THREADS), 0, s, a);
      } else {
        DK2Args<double> a{d.ptile.p, d.n_src, K, ldk, d.Nel, d.Nang, d.first.p, d.ni.p, d.skip.p, d.poff.p, d.pqo.p,
                          nullptr, d.k2_wg.p, d.k2_kshell.p, d.k2_rows.p, d.k2_kg.p, d.k2_gilm.p, d.k2_gslot.p,
                          d.k2_sl.p, d.k2_lt.p, d.k2_jo.p, d.k2_js.p, d.k2_ltv.p, d.k2_jtc.p, (int)d.sym};
        hipLaunchKernelGGL((k_dia_k2_off<double>), dim3(d.n_wg_k2), dim3(K2_THREADS), 0, s, a);
      }
      hip_check(hipGetLastError(), "diatomic_k2_off");
      continue;
    }
    const int n_ef_pad = ((n_ef + 7) / 8) * 8;
    const int64_t grid = (int64_t)n_ef_pad * d.n_act;
    if (grid > 0x7fffffff) throw Error(-1, "exchange grid too large");
    const int *efl = part == 0 ? (d.sym ? d.ef_low.p : d.ef_off.p) : d.ef_in.p;
    TimedLaunch tl(timer, name, s, flops, part == 0 ? "k_dia_k_off" : "k_dia_k_in");
    if (fp32) {
      DKArgs<float> a{d.P32.p, d.Nbf, K, ldk, d.Nel, d.Nang, d.n_act, d.first.p, d.ni.p, d.skip.p, d.poff.p,
                      d.pq32.p, d.chol32.p, d.sigma32.p, d.chol_off.p, d.chol_rank.p, d.act_jk.p, d.act_lstart.p,
                      d.lrun_ilm.p, d.lrun_tstart.p, d.term_pos.p, d.term_f32.p, efl, n_ef, d.lsig.p,
                      d.tiled ? d.ptile32.p : nullptr, d.term_tile.p, d.n_src, (int)d.sym};
      launch_dia_k<float>(part, d.tiled, grid, s, a);
    } else {
      DKArgs<double> a{P, ldp, K, ldk, d.Nel, d.Nang, d.n_act, d.first.p, d.ni.p, d.skip.p, d.poff.p, d.pq.p,
                       d.chol.p, d.sigma.p, d.chol_off.p, d.chol_rank.p, d.act_jk.p, d.act_lstart.p, d.lrun_ilm.p,
                       d.lrun_tstart.p, d.term_pos.p, d.term_f.p, efl, n_ef, nullptr,
                       d.tiled ? d.ptile.p : nullptr, d.term_tile.p, d.n_src, (int)d.sym};
      launch_dia_k<double>(part, d.tiled, grid, s, a);
    }
    hip_check(hipGetLastError(), "diatomic_k");
  }
  if (d.n_mirror > 0) {
    hipLaunchKernelGGL(k_dia_mirror, dim3(d.n_mirror), dim3(NT), 0, s, K, ldk, d.Nrad, d.poff.p, d.mirror.p,
                       d.Nang);
    hip_check(hipGetLastError(), "diatomic_mirror");
  }
}

}  // namespace hfg
