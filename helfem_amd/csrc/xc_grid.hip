// LDA exchange-correlation on the atomic and pure-m diatomic DFT grids
// (FP64), gfx950.
//
// Atomic grid (src/atomic/dftgrid.cpp:470-576): per element, nrad Chebyshev
// radial points x lang cos(theta) Chebyshev nodes x mang even phi points.
// Pure-m diatomic grid (src/diatomic/dftgrid_purem.cpp:87-199): per element,
// the mu points x lang nu points, the phi integral analytic.  In both the
// basis values factorise, chi_(a,r) = R_r(i) Theta_a(t) e^(i m_a phi_k), so
// instead of the reference's dense (functions x points) products the kernels
// contract one index at a time:
//   k_xc_rad_in   D_i(p)   = sum_rs R_r(i) P_(a,r),(b,s) R_s(i),  p = (a,b)
//   k_xc_point    rho(i,t,k) = sum_d C_d(i,t) cos(d phi_k),
//                 C_d(i,t) = sum_{p: m_a - m_b = d} Theta_a(t) Theta_b(t) D_i(p);
//                 LDA exc and v pointwise; V_d(i,t) = sum_k w v cos(d phi_k);
//                 W_i(p) = sum_t Theta_a(t) Theta_b(t) V_{m_a-m_b}(i,t)
//   k_xc_rad_out  H_(a,r),(b,s) = sum_i R_r(i) R_s(i) W_i(p), element bands
// which is the reference's rho = sum_uv P_uv Re(chi_u chi_v*) and
// H += (a .* w v) a' + (b .* w v) b' (dftgrid.cpp:51-128, 304-359;
// dftgrid_purem.cpp:212-260, 468-500) with the sums reordered.
//
// GGA (atomic: dftgrid.cpp:75-86, 166-180, 320-334, 382-405; pure-m
// diatomic: dftgrid_purem.cpp:248-260, 382-395, 468-500; 3D diatomic:
// src/diatomic/dftgrid.cpp:75-100, 292-305; dftgrid_common.h:188-216).  The
// gradient in the grid's orthogonal components, g = 2 Re sum P (d chi) chi* /
// (h_1, h_2, h_3), factorises the same way, with c_k = 1/h_k per point
// (atomic (1, 1/r, 1/(r sin theta)); diatomic 1/h_mu = 1/h_nu =
// 1/(Rh sqrt(sinh^2 mu + sin^2 nu)), 1/h_phi = 1/(Rh sinh mu sin nu)):
//   g_1 = 2 c_1 sum_d G_d cos(d phi),  G_d(t) = sum_{x in d} Theta_a Theta_b E(x),
//         E(x) = sum_rs R'_r P_(a,r),(b,s) R_s (k_xc_rad_in alongside D)
//   g_2 = c_2 sum_d T_d cos(d phi),  T_d(t) = sum_{x in d} (Theta_a Theta_b)' D(x)
//   g_3 = -c_3 sum_d d C_d sin(d phi)      (zero on the pure-m grid: d = 0)
// (the last two use D(a,b) = D(b,a), P symmetric, as the reference's factor
// 2 does).  With U = 2 w vsigma grad rho (restricted) the potential term
// H += X + X', X = sum U . Re(grad chi_u) chi_v*, becomes per pair x = (a,b)
//   H_(a,r),(b,s) += sum_i R_r R_s W2(x) + R'_r R_s Y(x) + R_r R'_s Y(x')
//   W2(x) = sum_t Theta_a Theta_b [V_d - d Vphi_d] + (Theta_a Theta_b)' Vtheta_d
//   Y(x)  = sum_t Theta_a Theta_b Vr_d,   x' = (b, a)
// with V_d, Vr_d, Vtheta_d = sum_k (w vrho, c_1 U_1, c_2 U_2) cos(d phi_k) and
// Vphi_d = sum_k c_3 U_3 sin(d phi_k).
//
// Meta-GGA (tau; dftgrid.cpp:89-107, 336-349; dftgrid_purem.cpp:287-318,
// 482-494): tau = 1/2 sum_c c_c^2 Re sum P d_c chi d_c chi*, per pair
//   radial  F(x) = sum_rs R'_r P R'_s  with Theta_a Theta_b,
//   theta   D(x) with Theta'_a Theta'_b,   phi  D(x) with m_a m_b Theta_a Theta_b,
// and H += sum_c (w vtau/2) c_c^2 Re d_c chi_u d_c chi_v*: with
// S_d = sum_k (w vtau / 2) cos(d phi_k), per pair
//   H += sum_i R'_r R'_s Z(x) + R_r R_s sum_t (c_2^2 Theta'_a Theta'_b + c_3^2 m_a m_b Theta_a Theta_b) S_d,
//   Z(x) = sum_t c_1^2 Theta_a Theta_b S_d.
//
// Everything above is symmetric in the two shells of a pair and even in phi
// (g_3 and U_3 are odd, and enter with the odd sin), so a pair {a, b} is taken
// once, with D and F of both orders added, E of both orders with the derivative
// on the row, one W and Y for H_ab and H_ba = H_ab', classes d >= 0, and the phi
// points k <= mang / 2 with weight 2 for k and mang - k.  That and one radial
// workgroup per run of pairs instead of per shell or pair: J + XC builds of Xe
// (lmax 6, 25 elements, LDA) 2.57 -> 1.56 ms, O (lmax 3, 12 elements, polarized
// PBE) 0.75 -> 0.42 ms, N2 (16 shells per |m| <= 2, 7 elements, pure-m LDA)
// 1.59 -> 0.98 ms.
#include "hfgpu_internal.hpp"
#include "device_common.hpp"
#include "xc_func.hpp"
#include <algorithm>

namespace hfg {
namespace {

using namespace dev;

// lda_x (id 1) and lda_c_vwn (id 7, VWN5), spin-unpolarised, as the libxc
// formulas: Slater e_x = -(3/4)(3/pi)^(1/3) rho^(1/3), v_x = 4/3 e_x; VWN5
// paramagnetic interpolation in x = sqrt(rs), v_c = e_c - (x/6) de_c/dx.
// Densities below thr give zero (libxc's density threshold).
__device__ inline void lda_point(int xf, int cf, double rho, double thr, double &exc, double &v) {
  exc = 0.0;
  v = 0.0;
  if (!(rho >= thr)) return;
  const double pi = 3.14159265358979323846;
  if (xf == 1) {
    const double ex = -0.75 * cbrt(3.0 / pi) * cbrt(rho);
    exc += ex;
    v += (4.0 / 3.0) * ex;
  }
  if (cf == 7) {
    const double A = 0.0310907, b = 3.72744, c = 12.9352, x0 = -0.10498;
    const double rs = cbrt(3.0 / (4.0 * pi * rho));
    const double x = sqrt(rs);
    const double Q = sqrt(4.0 * c - b * b);
    const double X = x * x + b * x + c, Xp = 2.0 * x + b, X0 = x0 * x0 + b * x0 + c;
    const double f1 = 2.0 * b / Q, f2 = b * x0 / X0, f3 = 2.0 * (2.0 * x0 + b) / Q;
    const double at = atan(Q / (2.0 * x + b));
    const double F = A * (log(x * x / X) + (f1 - f2 * f3) * at - f2 * log((x - x0) * (x - x0) / X));
    const double dF = A * (2.0 / x - Xp / X + (f1 - f2 * f3) * (-Q / (2.0 * X)) - f2 * (2.0 / (x - x0) - Xp / X));
    exc += F;
    v += F - x / 6.0 * dF;
  }
}

// Spin-polarized form: Slater exchange by spin scaling, VWN5 correlation
// e_c = e_P + alpha_c f(z)(1 - z^4)/f''(0) + (e_F - e_P) f(z) z^4 with
// v_cs = e_c - (rs/3) de/drs - (z - s) de/dz (libxc lda_c_vwn).
__device__ inline void vwn_aux(double A, double b, double c, double x0, double x, double &F, double &dF) {
  const double Q = sqrt(4.0 * c - b * b);
  const double X = x * x + b * x + c, Xp = 2.0 * x + b, X0 = x0 * x0 + b * x0 + c;
  const double f1 = 2.0 * b / Q, f2 = b * x0 / X0, f3 = 2.0 * (2.0 * x0 + b) / Q;
  const double at = atan(Q / (2.0 * x + b));
  F = A * (log(x * x / X) + (f1 - f2 * f3) * at - f2 * log((x - x0) * (x - x0) / X));
  dF = A * (2.0 / x - Xp / X + (f1 - f2 * f3) * (-Q / (2.0 * X)) - f2 * (2.0 / (x - x0) - Xp / X));
}

__device__ inline void lda_point_pol(int xf, int cf, double ra, double rb, double thr, double &exc, double &va,
                                     double &vb) {
  exc = 0.0;
  va = 0.0;
  vb = 0.0;
  const double rho = ra + rb;
  if (!(rho >= thr)) return;
  const double pi = 3.14159265358979323846;
  if (xf == 1) {
    const double c6 = cbrt(6.0 / pi);
    const double a3 = ra > 0.0 ? cbrt(ra) : 0.0, b3 = rb > 0.0 ? cbrt(rb) : 0.0;
    exc += -0.75 * c6 * (ra * a3 + rb * b3) / rho;
    va += -c6 * a3;
    vb += -c6 * b3;
  }
  if (cf == 7) {
    const double rs = cbrt(3.0 / (4.0 * pi * rho)), x = sqrt(rs);
    const double z = fmax(-1.0, fmin(1.0, (ra - rb) / rho));
    double eP, dP, eF, dF, eA, dA;
    vwn_aux(0.0310907, 3.72744, 12.9352, -0.10498, x, eP, dP);
    vwn_aux(0.01554535, 7.06042, 18.0578, -0.32500, x, eF, dF);
    vwn_aux(-1.0 / (6.0 * pi * pi), 1.13107, 13.0045, -0.0047584, x, eA, dA);
    const double c43 = cbrt(2.0) * 2.0 - 2.0;
    const double opz = 1.0 + z, omz = 1.0 - z, opz13 = cbrt(opz), omz13 = cbrt(omz);
    const double fz = (opz * opz13 + omz * omz13 - 2.0) / c43;
    const double dfz = 4.0 / 3.0 * (opz13 - omz13) / c43;
    const double fpp = 4.0 / (9.0 * (cbrt(2.0) - 1.0));
    const double z3 = z * z * z, z4 = z3 * z;
    const double e = eP + eA * fz * (1.0 - z4) / fpp + (eF - eP) * fz * z4;
    const double dedx = dP + dA * fz * (1.0 - z4) / fpp + (dF - dP) * fz * z4;
    const double dedz = eA * (dfz * (1.0 - z4) - 4.0 * z3 * fz) / fpp + (eF - eP) * (dfz * z4 + 4.0 * z3 * fz);
    const double base = e - x / 6.0 * dedx;
    exc += e;
    va += base - (z - 1.0) * dedz;
    vb += base - (z + 1.0) * dedz;
  }
}

__device__ inline long long grid_row(const int *skip, const long long *poff, int shell, int r) {
  const int s = skip[shell];
  return r >= s ? poff[shell] + (r - s) : -1;
}

struct XCArgs {
  const double *P;
  int64_t ldp;
  double *H;
  int64_t ldh;
  int Nel, Nang, nrad, lang, nk, nd, npiece, xf, cf, npair;
  double thr;
  const int *first, *ni, *skip;
  const long long *poff;
  const int2 *pab;
  const int *xd, *pstart;
  const int4 *piece;
  const double *R, *wpt, *thx, *thxt, *cs, *pw;
  double *D, *W, *part;
  double *Db, *Wb;  // second spin (polarized evaluation), else null
  // gradient terms (k_xc_rad_in<1>, k_xc_point_gga, k_xc_rad_out<1>);
  // gsc [Nel][nrad][lang][3] = 1/(h_1, h_2, h_3) per point
  const double *dR, *gsc, *sn, *thd, *thdt;
  double *E, *Y, *Eb, *Yb;
  // kinetic energy density terms (meta-GGA)
  const double *thdd, *thddt, *thmm, *thmmt;
  double *F, *Z, *Fb, *Zb;
};

// Both radial kernels take a run of consecutive pairs {a, b} of one element per
// workgroup and the radial points in runs of XR_PTS, so that the arrays
// [point][pair] are read and written in runs of pairs.
constexpr int XR_PAIRS = 16, XR_PTS = 80, XR_RS = TILE + 1, XR_WS = XR_PAIRS + 1;
// k_xc_rad_in: XI_J pairs contracted at a time by 40 threads each, two points
// per thread; XI_PAIRS pairs per workgroup, XI_J where that leaves CUs idle
constexpr int XI_J = 6, XI_PAIRS = 12, XI_WS = XI_PAIRS + 1, XI_PT = XR_PTS / 2;
static_assert(XI_J * XI_PT <= NT && XI_PAIRS % XI_J == 0, "pairs of a batch");

// D(x) = sum_rs R_r (P_ab + P_ba') R_s of every pair and radial point (P_aa for
// a = b), folded over r <= s: 136 terms; with GGA also E = sum_rs R'_r (P_ab +
// P_ba) R_s (the derivative on the row), with tau F = sum_rs R'_r (P_ab + P_ba')
// R'_s.  A thread takes two points of a pair with R in registers, so that each
// broadcast tile read serves two; the R rows sit in LDS at an odd stride.  R and
// the tiles are zero outside the element.  blockIdx.y: spin.  Bound by the LDS
// tile reads and the chain shell offsets -> P -> LDS of each batch.  Xe LDA 260
// (a workgroup per shell, ordered pairs) -> 240 (one point per thread, folded)
// -> 169 us; O polarized PBE 2 x 75 -> 41 us, there with XI_J pairs per workgroup
// (XI_PAIRS: half as many workgroups, fewer than 512 leave CUs idle).
// MODE 0: D only (LDA); 1: also E (GGA); 2: also F (meta-GGA)
template <int MODE>
__global__ void __launch_bounds__(NT) k_xc_rad_in(XCArgs A, XCArgs B, int per) {
  if (blockIdx.y) A = B;
  const int groups = (A.npair + per - 1) / per;
  const int e = blockIdx.x / groups, x0 = (blockIdx.x - e * groups) * per;
  const int t = threadIdx.x;
  const int ni = A.ni[e], f0 = A.first[e];
  const int np = min(per, A.npair - x0);
  extern __shared__ double sm[];
  double *sR = sm;                                   // [XR_PTS][XR_RS]
  double *sdR = sR + XR_PTS * XR_RS;                 // with GGA
  double *sS = sR + (MODE ? 2 : 1) * XR_PTS * XR_RS;  // [XI_J][TILE2], folded to r <= s
  double *sG = sS + XI_J * TILE2;                    // with GGA: not folded
  double *sO = sS + (MODE ? 2 : 1) * XI_J * TILE2;   // [MODE + 1][XR_PTS][XI_WS]
  const int r = t & 15, s = t >> 4;
  const int j = t / XI_PT, i = t - j * XI_PT;
  for (int i0 = 0; i0 < A.nrad; i0 += XR_PTS) {
    const int nq = min(XR_PTS, A.nrad - i0);
    for (int q = t; q < XR_PTS * TILE; q += NT) {
      const bool in = (q >> 4) < nq;
      sR[(q >> 4) * XR_RS + (q & 15)] = in ? A.R[((size_t)e * A.nrad + i0) * TILE + q] : 0.0;
      if (MODE) sdR[(q >> 4) * XR_RS + (q & 15)] = in ? A.dR[((size_t)e * A.nrad + i0) * TILE + q] : 0.0;
    }
    for (int xb = 0; xb < np; xb += XI_J) {
      __syncthreads();
#pragma unroll
      for (int jj = 0; jj < XI_J; ++jj) {
        double gv = 0.0;
        if (xb + jj < np && r < ni && s < ni) {
          const int2 ab = A.pab[x0 + xb + jj];
          const long long ra = grid_row(A.skip, A.poff, ab.x, f0 + r), cb = grid_row(A.skip, A.poff, ab.y, f0 + s);
          if (ra >= 0 && cb >= 0) gv = A.P[ra + cb * A.ldp];
          if (ab.x != ab.y) {
            const long long rb = grid_row(A.skip, A.poff, ab.y, f0 + r), ca = grid_row(A.skip, A.poff, ab.x, f0 + s);
            if (rb >= 0 && ca >= 0) gv += A.P[rb + ca * A.ldp];
          }
        }
        sS[jj * TILE2 + t] = gv;
        if (MODE) sG[jj * TILE2 + t] = gv;
      }
      __syncthreads();
      if (r < s)  // only r > s is read
#pragma unroll
        for (int jj = 0; jj < XI_J; ++jj) sS[jj * TILE2 + t] += sS[jj * TILE2 + s + TILE * r];
      __syncthreads();
      if (j < XI_J && xb + j < np) {
        const double *St = sS + j * TILE2, *Gt = sG + j * TILE2;
        const double *dR0 = sdR + i * XR_RS, *dR1 = dR0 + XI_PT * XR_RS;
        double r0[TILE], r1[TILE];
#pragma unroll
        for (int c = 0; c < TILE; ++c) {
          r0[c] = sR[i * XR_RS + c];
          r1[c] = sR[(i + XI_PT) * XR_RS + c];
        }
        double d0 = 0.0, d1 = 0.0;
#pragma unroll
        for (int c = 0; c < TILE; ++c) {
          double t0 = 0.0, t1 = 0.0;
#pragma unroll
          for (int k = 0; k <= c; ++k) {
            const double v = St[k + TILE * c];
            t0 += v * r0[k];
            t1 += v * r1[k];
          }
          d0 += r0[c] * t0;
          d1 += r1[c] * t1;
        }
        double *o = sO + i * XI_WS + xb + j;
        o[0] = d0;
        o[XI_PT * XI_WS] = d1;
        if (MODE) {
          double e0 = 0.0, e1 = 0.0;
          for (int k = 0; k < TILE; ++k) {
            double t0 = 0.0, t1 = 0.0;
#pragma unroll
            for (int c = 0; c < TILE; ++c) {
              const double v = Gt[k + TILE * c];
              t0 += v * r0[c];
              t1 += v * r1[c];
            }
            e0 += dR0[k] * t0;
            e1 += dR1[k] * t1;
          }
          o[XR_PTS * XI_WS] = e0;
          o[(XR_PTS + XI_PT) * XI_WS] = e1;
        }
        if (MODE == 2) {
#pragma unroll
          for (int c = 0; c < TILE; ++c) {
            r0[c] = dR0[c];
            r1[c] = dR1[c];
          }
          double f0k = 0.0, f1k = 0.0;
#pragma unroll
          for (int c = 0; c < TILE; ++c) {
            double t0 = 0.0, t1 = 0.0;
#pragma unroll
            for (int k = 0; k <= c; ++k) {
              const double v = St[k + TILE * c];
              t0 += v * r0[k];
              t1 += v * r1[k];
            }
            f0k += r0[c] * t0;
            f1k += r1[c] * t1;
          }
          o[2 * XR_PTS * XI_WS] = f0k;
          o[(2 * XR_PTS + XI_PT) * XI_WS] = f1k;
        }
      }
    }
    __syncthreads();
    for (int q = t; q < nq * per; q += NT) {
      const int p = q / per, x = q - p * per;
      if (x >= np) continue;
      const size_t o = ((size_t)e * A.nrad + i0 + p) * A.npair + x0 + x;
      A.D[o] = sO[p * XI_WS + x];
      if (MODE) A.E[o] = sO[(XR_PTS + p) * XI_WS + x];
      if (MODE == 2) A.F[o] = sO[(2 * XR_PTS + p) * XI_WS + x];
    }
    __syncthreads();
  }
}

// Class sums out[c][d][t] = sum_{x in d} table_c[x][t] src_c[x] of one radial
// point: threads (piece, t) form partial sums over at most 32 pairs (lanes read
// consecutive t), then (d, t) add the class' pieces in order.
template <typename Table, typename Source>
__device__ inline void class_sums(const XCArgs &A, int ncs, Table table, Source src, double *partial, double *out) {
  const int lang = A.lang, npc = A.npiece * lang;
  const bool one = A.npiece == 1 && A.nd == 1;  // the piece is the sum
  if (one) partial = out;
  for (int q = threadIdx.x; q < ncs * npc; q += blockDim.x) {
    const int c = q / npc, r = q - c * npc, p = r / lang, tt = r - p * lang;
    const int4 pc = A.piece[p];
    const double *tab = table(c) + tt, *s = src(c);
    double v = 0.0;
#pragma unroll 4
    for (int x = pc.y; x < pc.z; ++x) v += tab[(size_t)x * lang] * s[x];
    partial[q] = v;
  }
  __syncthreads();
  if (one) return;
  for (int q = threadIdx.x; q < ncs * A.nd * lang; q += blockDim.x) {
    const int c = q / (A.nd * lang), r = q - c * A.nd * lang, d = r / lang, tt = r - d * lang;
    double v = 0.0;
    for (int p = A.pstart[d]; p < A.pstart[d + 1]; ++p) v += partial[c * npc + p * lang + tt];
    out[q] = v;
  }
  __syncthreads();
}

// One workgroup per (element, radial point); with A.Db set the density of the
// second spin is contracted alongside and the polarized functional used.  The
// pairs x are numbered by class d = m_a - m_b, so the class sums read contiguous
// runs of D and of the Theta_a Theta_b table, and thread x forms W(x) from the
// [t][x] table (lanes read consecutive x).  Bound by the two Theta tables read
// from L2 for every radial point (Xe: 2 x 0.35 MB) and the latency of the chain of
// phases: Xe LDA 811 (ordered pairs, all phi points) -> 156 us, N2 pure-m
// 629 -> 70 us (512 threads: 182 and 74).
constexpr int LP_MAX = 256;

__global__ void __launch_bounds__(LP_MAX) k_xc_point(XCArgs A) {
  const int e = blockIdx.x / A.nrad, i = blockIdx.x - e * A.nrad;
  const int t = threadIdx.x, nt = blockDim.x;
  const int np = A.npair, nd = A.nd, lang = A.lang, nk = A.nk, nang = lang * nk;
  const bool pol = A.Db != nullptr;
  const int ns = pol ? 2 : 1;
  extern __shared__ double sm[];
  double *sD = sm;                    // [ns][np]
  double *sC = sD + ns * np;          // [ns][nd][lang]
  double *sV = sC + ns * nd * lang;   // [ns][lang][nk]; first the partial class sums
  __shared__ double red[2 * LP_MAX / 64];
  const size_t row = ((size_t)e * A.nrad + i) * np;
  for (int x = t; x < np; x += nt) {
    sD[x] = A.D[row + x];
    if (pol) sD[np + x] = A.Db[row + x];
  }
  __syncthreads();
  class_sums(A, ns, [&](int) { return A.thxt; }, [&](int c) { return sD + c * np; }, sV, sC);
  const double *wp = A.wpt + ((size_t)e * A.nrad + i) * lang;
  double ex = 0.0, ne = 0.0;
  for (int q = t; q < nang; q += nt) {
    const int tt = q / nk, k = q - tt * nk;
    double ra = 0.0, rb = 0.0;
    for (int d = 0; d < nd; ++d) ra += sC[d * lang + tt] * A.cs[(size_t)d * nk + k];
    if (pol)
      for (int d = 0; d < nd; ++d) rb += sC[nd * lang + d * lang + tt] * A.cs[(size_t)d * nk + k];
    const double w = wp[tt] * A.pw[k];
    double exc, va, vb = 0.0;
    if (pol)
      lda_point_pol(A.xf, A.cf, ra, rb, A.thr, exc, va, vb);
    else
      lda_point(A.xf, A.cf, ra, A.thr, exc, va);
    ex += w * exc * (ra + rb);
    ne += w * (ra + rb);
    sV[q] = w * va;
    if (pol) sV[nang + q] = w * vb;
  }
  ex = wave_sum(ex);
  ne = wave_sum(ne);
  if ((t & 63) == 0) {
    red[t >> 6] = ex;
    red[LP_MAX / 64 + (t >> 6)] = ne;
  }
  __syncthreads();
  if (t == 0) {
    double sx = 0.0, sn = 0.0;
    for (int w = 0; w < nt / 64; ++w) {
      sx += red[w];
      sn += red[LP_MAX / 64 + w];
    }
    A.part[3 * ((size_t)e * A.nrad + i)] = sx;
    A.part[3 * ((size_t)e * A.nrad + i) + 1] = sn;
    A.part[3 * ((size_t)e * A.nrad + i) + 2] = 0.0;
  }
  for (int q = t; q < ns * nd * lang; q += nt) {
    const int sp = q / (nd * lang), qq = q - sp * nd * lang;
    const int d = qq / lang, tt = qq - d * lang;
    const double *V = sV + sp * nang + tt * nk;
    double s = 0.0;
    for (int k = 0; k < nk; ++k) s += V[k] * A.cs[(size_t)d * nk + k];
    sC[q] = s;
  }
  __syncthreads();
  for (int sp = 0; sp < ns; ++sp) {
    double *Wout = sp == 0 ? A.W : A.Wb;
    const double *C = sC + sp * nd * lang;
    for (int x = t; x < np; x += nt) {
      const double *Cd = C + A.xd[x] * lang;
      double w = 0.0;
#pragma unroll 4
      for (int tt = 0; tt < lang; ++tt) w += A.thx[(size_t)tt * np + x] * Cd[tt];
      Wout[row + x] = w;
    }
  }
}

// General point kernel: one workgroup per (element, radial point), both spins
// when polarized.  LDS: region A holds each spin's radial contractions (D, E
// and with tau F), then its point values (w vrho, c_1 U_1, c_2 U_2, c_3 U_3
// and with tau w vtau/2); region B holds the class sums (C, G, T and with tau
// the three tau sums), then the class transforms (V_d - d Vphi_d, Vr_d,
// Vtheta_d and with tau S_d); region C the pieces of the class sums.  Any
// supported functional pair runs here (vsigma = 0 without a GGA part, vtau = 0
// without a meta-GGA part).
template <int MODE> struct GgaShape {
  static constexpr int nin = MODE == 2 ? 3 : 2;  // radial contractions per spin
  static constexpr int ncs = MODE == 2 ? 6 : 3;  // class sums per spin
  static constexpr int npv = MODE == 2 ? 5 : 4;  // point arrays per spin
};

// Threads: one per angular point, at least 256, at most 512.  Bound by the
// functional's FP64 arithmetic and its register spills at 256 registers: O polarized
// PBE 459 (ordered pairs, all phi points, 1024 threads) -> 236 (folded) -> 181 us
// (all derivatives in one pass over the functional instead of one pass each).  256
// threads: 169 us there, but TPSS and CAM-B3LYP of Xe 4 to 5% slower.
constexpr int XP_MAX = 512;

template <int MODE>
__global__ void __launch_bounds__(XP_MAX) k_xc_point_gga(XCArgs A) {
  typedef GgaShape<MODE> G;
  const int e = blockIdx.x / A.nrad, i = blockIdx.x - e * A.nrad;
  const int t = threadIdx.x, nt = blockDim.x;
  const int np = A.npair, nd = A.nd, lang = A.lang, nk = A.nk, nang = lang * nk;
  const bool pol = A.Db != nullptr;
  const int ns = pol ? 2 : 1;
  constexpr bool tau = MODE == 2;
  const int na = max(G::nin * np, G::npv * nang), ncl = nd * lang;
  extern __shared__ double sm[];
  double *sA = sm;                         // [ns][na]
  double *sB = sm + ns * na;               // [ncs][ns][nd][lang]
  double *sP = sB + ns * G::ncs * ncl;     // [ns][pieces][lang]
  __shared__ double red[3 * XP_MAX / 64];
  const size_t row = ((size_t)e * A.nrad + i) * np;
  for (int x = t; x < np; x += nt) {
    sA[x] = A.D[row + x];
    sA[np + x] = A.E[row + x];
    if (tau) sA[2 * np + x] = A.F[row + x];
    if (pol) {
      sA[na + x] = A.Db[row + x];
      sA[na + np + x] = A.Eb[row + x];
      if (tau) sA[na + 2 * np + x] = A.Fb[row + x];
    }
  }
  __syncthreads();
  // class sums: 0 C (Theta Theta D), 1 G (Theta Theta E), 2 T ((Theta Theta)' D),
  // with tau 3 (Theta Theta F), 4 (Theta' Theta' D), 5 (m m Theta Theta D)
  for (int c = 0; c < G::ncs; ++c) {
    const double *tab = c == 2 ? A.thdt : c == 4 ? A.thddt : c == 5 ? A.thmmt : A.thxt;
    const int off = c == 1 ? np : c == 3 ? 2 * np : 0;
    class_sums(A, ns, [&](int) { return tab; }, [&](int sp) { return sA + sp * na + off; }, sP, sB + c * ns * ncl);
  }
  const double *wp = A.wpt + ((size_t)e * A.nrad + i) * lang;
  const double *gs = A.gsc + ((size_t)e * A.nrad + i) * lang * 3;
  double ex = 0.0, ne = 0.0, ek = 0.0;
  for (int q = t; q < nang; q += nt) {
    const int tt = q / nk, k = q - tt * nk;
    const double c1 = gs[3 * tt], c2 = gs[3 * tt + 1], c3 = gs[3 * tt + 2];
    double rho[2] = {0.0, 0.0}, g[2][3] = {{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}}, tk[2] = {0.0, 0.0};
    for (int sp = 0; sp < ns; ++sp) {
      const double *C = sB + sp * ncl;
      const int cst = ns * ncl;
      double r0 = 0.0, gr = 0.0, gt = 0.0, gp = 0.0, kf = 0.0, kt = 0.0, km = 0.0;
      for (int d = 0; d < nd; ++d) {
        const double cc = A.cs[(size_t)d * nk + k], cd = C[d * lang + tt];
        r0 += cd * cc;
        gr += C[cst + d * lang + tt] * cc;
        gt += C[2 * cst + d * lang + tt] * cc;
        gp += (double)d * cd * A.sn[(size_t)d * nk + k];
        if (tau) {
          kf += C[3 * cst + d * lang + tt] * cc;
          kt += C[4 * cst + d * lang + tt] * cc;
          km += C[5 * cst + d * lang + tt] * cc;
        }
      }
      rho[sp] = r0;
      g[sp][0] = 2.0 * c1 * gr;
      g[sp][1] = c2 * gt;
      g[sp][2] = -c3 * gp;
      if (tau) tk[sp] = 0.5 * (c1 * c1 * kf + c2 * c2 * kt + c3 * c3 * km);
    }
    const double w = wp[tt] * A.pw[k];
    double f, va, vb = 0.0, vta = 0.0, vtb = 0.0, u[2][3];
    if (pol) {
      const double x7[7] = {rho[0], rho[1], g[0][0] * g[0][0] + g[0][1] * g[0][1] + g[0][2] * g[0][2],
                            g[0][0] * g[1][0] + g[0][1] * g[1][1] + g[0][2] * g[1][2],
                            g[1][0] * g[1][0] + g[1][1] * g[1][1] + g[1][2] * g[1][2], tk[0], tk[1]};
      double v[7];
      xcf::eval_pol<tau>(A.xf, A.cf, x7, A.thr, f, v);
      va = v[0];
      vb = v[1];
      vta = v[5];
      vtb = v[6];
      for (int c = 0; c < 3; ++c) {
        u[0][c] = w * (2.0 * v[2] * g[0][c] + v[3] * g[1][c]);
        u[1][c] = w * (2.0 * v[4] * g[1][c] + v[3] * g[0][c]);
      }
    } else {
      const double x3[3] = {rho[0], g[0][0] * g[0][0] + g[0][1] * g[0][1] + g[0][2] * g[0][2], tk[0]};
      double v[3];
      xcf::eval_unpol<tau>(A.xf, A.cf, x3, A.thr, f, v);
      va = v[0];
      vta = v[2];
      for (int c = 0; c < 3; ++c) u[0][c] = 2.0 * w * v[1] * g[0][c];
    }
    ex += w * f;
    ne += w * (rho[0] + rho[1]);
    ek += w * (tk[0] + tk[1]);
    sA[q] = w * va;
    sA[nang + q] = c1 * u[0][0];
    sA[2 * nang + q] = c2 * u[0][1];
    sA[3 * nang + q] = c3 * u[0][2];
    if (tau) sA[4 * nang + q] = 0.5 * w * vta;
    if (pol) {
      sA[na + q] = w * vb;
      sA[na + nang + q] = c1 * u[1][0];
      sA[na + 2 * nang + q] = c2 * u[1][1];
      sA[na + 3 * nang + q] = c3 * u[1][2];
      if (tau) sA[na + 4 * nang + q] = 0.5 * w * vtb;
    }
  }
  ex = wave_sum(ex);
  ne = wave_sum(ne);
  ek = wave_sum(ek);
  if ((t & 63) == 0) {
    red[t >> 6] = ex;
    red[XP_MAX / 64 + (t >> 6)] = ne;
    red[2 * XP_MAX / 64 + (t >> 6)] = ek;
  }
  __syncthreads();
  if (t == 0) {
    double sx = 0.0, sn = 0.0, sk = 0.0;
    for (int w = 0; w < nt / 64; ++w) {
      sx += red[w];
      sn += red[XP_MAX / 64 + w];
      sk += red[2 * XP_MAX / 64 + w];
    }
    A.part[3 * ((size_t)e * A.nrad + i)] = sx;
    A.part[3 * ((size_t)e * A.nrad + i) + 1] = sn;
    A.part[3 * ((size_t)e * A.nrad + i) + 2] = sk;
  }
  // class transforms: 0 Q = V_d - d Vphi_d, 1 Vr_d, 2 Vtheta_d, with tau 3 S_d
  const int ntr = tau ? 4 : 3;
  for (int q = t; q < ns * ntr * ncl; q += nt) {
    const int sp = q / (ntr * ncl), r1 = q - sp * ntr * ncl, c = r1 / ncl, r2 = r1 - c * ncl;
    const int d = r2 / lang, tt = r2 - d * lang;
    const double *V = sA + sp * na + tt * nk;
    const double *cs = A.cs + (size_t)d * nk, *snd = A.sn + (size_t)d * nk;
    double acc = 0.0;
    if (c == 0) {
      const double *Vp = V + 3 * nang;
      for (int k = 0; k < nk; ++k) acc += V[k] * cs[k] - (double)d * Vp[k] * snd[k];
    } else {
      const double *Vc = V + (c == 1 ? 1 : c == 2 ? 2 : 4) * nang;
      for (int k = 0; k < nk; ++k) acc += Vc[k] * cs[k];
    }
    sB[sp * G::ncs * ncl + c * ncl + d * lang + tt] = acc;
  }
  __syncthreads();
  for (int sp = 0; sp < ns; ++sp) {
    double *Wout = sp == 0 ? A.W : A.Wb, *Yout = sp == 0 ? A.Y : A.Yb, *Zout = sp == 0 ? A.Z : A.Zb;
    const double *Q = sB + sp * G::ncs * ncl, *Vr = Q + ncl, *Vt = Vr + ncl, *S = Vt + ncl;
    for (int x = t; x < np; x += nt) {
      const int d = A.xd[x];
      const double *Qd = Q + d * lang, *Vrd = Vr + d * lang, *Vtd = Vt + d * lang, *Sd = S + d * lang;
      double w2 = 0.0, y = 0.0, z = 0.0;
#pragma unroll 4
      for (int tt = 0; tt < lang; ++tt) {
        const double th = A.thx[(size_t)tt * np + x];
        w2 += th * Qd[tt] + A.thd[(size_t)tt * np + x] * Vtd[tt];
        y += th * Vrd[tt];
        if (tau) {
          const double c1 = gs[3 * tt], c2 = gs[3 * tt + 1], c3 = gs[3 * tt + 2];
          w2 += (c2 * c2 * A.thdd[(size_t)tt * np + x] + c3 * c3 * A.thmm[(size_t)tt * np + x]) * Sd[tt];
          z += c1 * c1 * th * Sd[tt];
        }
      }
      Wout[row + x] = w2;
      Yout[row + x] = y;
      if (tau) Zout[row + x] = z;
    }
  }
}

// H_ab = H_ba = sum_i R' diag(W) R of every pair (with GGA M + M', M = sum_i
// (R W / 2 + dR Y)' R; with tau also dR' diag(Z) dR) on the FP64 matrix cores:
// one wave per pair, 16 pairs per workgroup.  The corner entry shared with
// element e+1 is written by e with both contributions (the wave sums e+1's over
// its points); e > 0 skips its own (0,0).  blockIdx.y: spin.
// Bound by the band writes and the W reads: Xe LDA 393 (FP64 vector sums, a
// workgroup per ordered pair) -> 100 us, N2 68 -> 34, O polarized PBE 2 x 124 -> 30.
template <int MODE>
__global__ void __launch_bounds__(NT) k_xc_rad_out(XCArgs A, XCArgs B) {
  if (blockIdx.y) A = B;
  const int groups = (A.npair + XR_PAIRS - 1) / XR_PAIRS;
  const int e = blockIdx.x / groups, x0 = (blockIdx.x - e * groups) * XR_PAIRS;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6, g = lane >> 4, c = lane & 15;
  const int ni = A.ni[e], f0 = A.first[e];
  const int np = min(XR_PAIRS, A.npair - x0);
  const bool has_next = e + 1 < A.Nel;
  constexpr int PW = XR_PAIRS / (NT / 64);
  extern __shared__ double sm[];
  double *sR = sm;                                    // [XR_PTS][XR_RS]
  double *sdR = sR + XR_PTS * XR_RS;                  // with GGA
  double *sW = sR + (MODE ? 2 : 1) * XR_PTS * XR_RS;  // [MODE + 1][XR_PTS][XR_WS]
  v4d acc[PW];
  double crn[PW];  // e+1's share of the corner entry, per lane
#pragma unroll
  for (int p = 0; p < PW; ++p) {
    acc[p] = v4d{0.0, 0.0, 0.0, 0.0};
    crn[p] = 0.0;
  }
  for (int i0 = 0; i0 < A.nrad; i0 += XR_PTS) {
    const int nq = min(XR_PTS, A.nrad - i0), nq4 = (nq + 3) & ~3;
    __syncthreads();
    for (int q = t; q < nq4 * TILE; q += NT) {  // zeros up to a whole k-step
      const bool in = (q >> 4) < nq;
      sR[(q >> 4) * XR_RS + (q & 15)] = in ? A.R[((size_t)e * A.nrad + i0) * TILE + q] : 0.0;
      if (MODE) sdR[(q >> 4) * XR_RS + (q & 15)] = in ? A.dR[((size_t)e * A.nrad + i0) * TILE + q] : 0.0;
    }
    for (int q = t; q < nq4 * XR_PAIRS; q += NT) {
      const int i = q >> 4, x = q & 15;
      const bool in = i < nq && x < np;
      const size_t o = ((size_t)e * A.nrad + i0 + i) * A.npair + x0 + x;
      sW[i * XR_WS + x] = in ? A.W[o] : 0.0;
      if (MODE) sW[(XR_PTS + i) * XR_WS + x] = in ? A.Y[o] : 0.0;
      if (MODE == 2) sW[(2 * XR_PTS + i) * XR_WS + x] = in ? A.Z[o] : 0.0;
    }
    __syncthreads();
    for (int ks = 0; ks < nq4; ks += 4) {
      const double r = sR[(ks + g) * XR_RS + c], dr = MODE ? sdR[(ks + g) * XR_RS + c] : 0.0;
#pragma unroll
      for (int p = 0; p < PW; ++p) {
        const int x = wv * PW + p;
        const double w = sW[(ks + g) * XR_WS + x];
        if (MODE == 0) {
          acc[p] = __builtin_amdgcn_mfma_f64_16x16x4f64(w * r, r, acc[p], 0, 0, 0);
        } else {
          const double y = sW[(XR_PTS + ks + g) * XR_WS + x];
          acc[p] = __builtin_amdgcn_mfma_f64_16x16x4f64(0.5 * w * r + y * dr, r, acc[p], 0, 0, 0);
          if (MODE == 2) {
            // symmetric: half of it survives the M + M' below
            const double z = sW[(2 * XR_PTS + ks + g) * XR_WS + x];
            acc[p] = __builtin_amdgcn_mfma_f64_16x16x4f64(0.5 * z * dr, dr, acc[p], 0, 0, 0);
          }
        }
      }
    }
    if (has_next)
#pragma unroll
      for (int p = 0; p < PW; ++p) {
        const int x = wv * PW + p;
        if (x >= np) continue;
        for (int i = lane; i < nq; i += 64) {
          const size_t n = (size_t)(e + 1) * A.nrad + i0 + i, o = n * A.npair + x0 + x;
          const double r = A.R[n * TILE];
          double v = r * r * A.W[o];
          if (MODE) {
            const double dr = A.dR[n * TILE];
            v += 2.0 * r * dr * A.Y[o];
            if (MODE == 2) v += dr * dr * A.Z[o];
          }
          crn[p] += v;
        }
      }
  }
  double *sT = sW;  // transposes, one 16 x 17 tile per wave
  if (MODE) __syncthreads();
#pragma unroll
  for (int p = 0; p < PW; ++p) {
    const int x = wv * PW + p;
    if (x >= np) continue;
    v4d v = acc[p];  // lane (g,c): entry (g + 4 s, c)
    if (MODE) {
      double *T = sT + wv * TILE * XR_RS;
#pragma unroll
      for (int s = 0; s < 4; ++s) T[(g + 4 * s) * XR_RS + c] = v[s];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int s = 0; s < 4; ++s) v[s] += T[c * XR_RS + g + 4 * s];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    double corner = 0.0;
    if (has_next) {
      corner = wave_sum(crn[p]);
      corner = __shfl(corner, 0, 64);
    }
    const int2 ab = A.pab[x0 + x];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      // the tile is symmetric: entry (c, col), so that lanes of one column
      // write consecutive rows
      const int cl = g + 4 * s;
      if (c >= ni || cl >= ni || (e > 0 && c == 0 && cl == 0)) continue;
      double h = v[s];
      if (has_next && c == ni - 1 && cl == ni - 1) h += corner;
      const long long ra = grid_row(A.skip, A.poff, ab.x, f0 + c), cb = grid_row(A.skip, A.poff, ab.y, f0 + cl);
      if (ra >= 0 && cb >= 0) A.H[ra + cb * A.ldh] = h;
      if (ab.x != ab.y) {
        const long long rb = grid_row(A.skip, A.poff, ab.y, f0 + c), ca = grid_row(A.skip, A.poff, ab.x, f0 + cl);
        if (rb >= 0 && ca >= 0) A.H[rb + ca * A.ldh] = h;
      }
    }
  }
}

}  // namespace

bool xc_generic(int xf, int cf) { return !((xf == 0 || xf == 1) && (cf == 0 || cf == 7)); }
bool xc_tau(int xf, int cf) { return xcf::is_mgga(xf) || xcf::is_mgga(cf); }

size_t xc_gga_limit_lds(const XCGridDevice &g, int ns, bool tau) {
  const int nin = tau ? 3 : 2, ncs = tau ? 6 : 3, npv = tau ? 5 : 4;
  const size_t na = (size_t)std::max(nin * g.npair_all, npv * g.lang * g.mang);
  return sizeof(double) * ns * (na + (size_t)ncs * (2 * g.dmax + 1) * g.lang);
}

size_t xc_gga_point_lds(const XCGridDevice &g, int ns, bool tau) {
  const int nin = tau ? 3 : 2, ncs = tau ? 6 : 3, npv = tau ? 5 : 4;
  const size_t na = (size_t)std::max(nin * g.npair, npv * g.lang * g.nk);
  const size_t pieces = g.npiece == 1 && g.dmax == 0 ? 0 : (size_t)g.npiece * g.lang;
  return sizeof(double) * ns * (na + (size_t)ncs * (g.dmax + 1) * g.lang + pieces);
}

size_t xc_limit_lds(const XCGridDevice &g, int xf, int cf, bool pol) {
  const int ns = pol ? 2 : 1, nd = 2 * g.dmax + 1;
  if (xc_generic(xf, cf)) return xc_gga_limit_lds(g, ns, xc_tau(xf, cf));
  return sizeof(double) * ns * ((size_t)g.npair_all + (size_t)g.lang * nd + (size_t)g.lang * g.mang);
}

namespace {
template <typename F>
void allow_lds(F f, size_t bytes, const char *what) {
  if (bytes > 64 * 1024)
    hip_check(hipFuncSetAttribute(reinterpret_cast<const void *>(f), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)bytes),
              what);
}

template <int MODE>
void launch_general(const XCGridDevice &g, const XCArgs &a, const XCArgs &b, bool pol, hipStream_t s,
                    KernelTimer *timer) {
  const int ns = pol ? 2 : 1, nd = g.dmax + 1;
  const unsigned groups = (unsigned)((g.npair + XR_PAIRS - 1) / XR_PAIRS) * g.Nel;
  const size_t radial = sizeof(double) * (MODE ? 2 : 1) * XR_PTS * XR_RS;
  const size_t vals = sizeof(double) * (MODE + 1) * XR_PTS * XR_WS;
  {
    TimedLaunch tl(timer, "xc_rad_in", s);
    const size_t lds =
        radial + sizeof(double) * ((MODE ? 2 : 1) * XI_J * TILE2 + (MODE + 1) * XR_PTS * XI_WS);
    const int per = (size_t)g.npair * g.Nel * ns >= 512 * XI_PAIRS ? XI_PAIRS : XI_J;
    allow_lds(&k_xc_rad_in<MODE>, lds, "xc_rad_in LDS size");
    hipLaunchKernelGGL(k_xc_rad_in<MODE>, dim3((unsigned)((g.npair + per - 1) / per) * g.Nel, ns), dim3(NT), lds, s, a,
                       b, per);
    hip_check(hipGetLastError(), "xc_rad_in");
  }
  {
    TimedLaunch tl(timer, "xc_point", s);
    const unsigned points = (unsigned)(g.Nel * g.nrad);
    if constexpr (MODE == 0) {
      const size_t lds = sizeof(double) * ns *
                         ((size_t)g.npair + (size_t)g.lang * nd + (size_t)g.lang * std::max(g.nk, g.npiece));
      allow_lds(&k_xc_point, lds, "xc_point LDS size");
      hipLaunchKernelGGL(k_xc_point, dim3(points), dim3(LP_MAX), lds, s, a);
    } else {
      const size_t lds = xc_gga_point_lds(g, ns, MODE == 2);
      const int threads = std::min(XP_MAX, std::max(256, (g.lang * g.nk + 63) / 64 * 64));
      allow_lds(&k_xc_point_gga<MODE>, lds, "xc_point_gga LDS size");
      hipLaunchKernelGGL(k_xc_point_gga<MODE>, dim3(points), dim3(threads), lds, s, a);
    }
    hip_check(hipGetLastError(), "xc_point");
  }
  {
    TimedLaunch tl(timer, "xc_rad_out", s);
    const size_t lds = radial + std::max(vals, sizeof(double) * (NT / 64) * TILE * XR_RS);
    allow_lds(&k_xc_rad_out<MODE>, lds, "xc_rad_out LDS size");
    hipLaunchKernelGGL(k_xc_rad_out<MODE>, dim3(groups, ns), dim3(NT), lds, s, a, b);
    hip_check(hipGetLastError(), "xc_rad_out");
  }
}
}  // namespace

void xc_grid_launch(XCGridDevice &g, int xf, int cf, double thr, const double *Pa, int64_t ldpa, const double *Pb,
                    int64_t ldpb, double *Ha, int64_t ldha, double *Hb, int64_t ldhb, hipStream_t s,
                    KernelTimer *timer) {
  const bool pol = Pb != nullptr;
  const int mode = xc_tau(xf, cf) ? 2 : xc_generic(xf, cf) ? 1 : 0;
  fill_zero_launch(Ha, g.Nbf, g.Nbf, ldha, s);
  if (pol) fill_zero_launch(Hb, g.Nbf, g.Nbf, ldhb, s);
  XCArgs a{Pa, ldpa, Ha, ldha, g.Nel, g.Nang, g.nrad, g.lang, g.nk, g.dmax + 1, g.npiece, xf, cf, g.npair, thr,
           g.first.p, g.ni.p, g.skip.p, g.poff.p, g.pab.p, g.xd.p, g.pstart.p, g.piece.p,
           g.R.p, g.wpt.p, g.thx.p, g.thxt.p, g.cs.p, g.pw.p, g.D.p, g.W.p, g.part.p, pol ? g.Db.p : nullptr,
           pol ? g.Wb.p : nullptr, g.dR.p, g.gsc.p, g.sn.p, g.thd.p, g.thdt.p,
           g.E.p, g.Y.p, pol ? g.Eb.p : nullptr, pol ? g.Yb.p : nullptr,
           g.thdd.p, g.thddt.p, g.thmm.p, g.thmmt.p, g.F.p, g.Z.p, pol ? g.Fb.p : nullptr, pol ? g.Zb.p : nullptr};
  XCArgs b = a;  // second spin: its density in, its matrix out
  if (pol) {
    b.P = Pb;
    b.ldp = ldpb;
    b.H = Hb;
    b.ldh = ldhb;
    b.D = g.Db.p;
    b.W = g.Wb.p;
    b.E = g.Eb.p;
    b.Y = g.Yb.p;
    b.F = g.Fb.p;
    b.Z = g.Zb.p;
  }
  if (mode == 2)
    launch_general<2>(g, a, b, pol, s, timer);
  else if (mode == 1)
    launch_general<1>(g, a, b, pol, s, timer);
  else
    launch_general<0>(g, a, b, pol, s, timer);
}

}  // namespace hfg
