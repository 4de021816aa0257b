// C-ABI for the diatomic basis (include/hfgpu.h): handle, device tables and
// the coupling lists of the Coulomb and exchange kernels (diatomic_jk.hip).
#include "capi_common.hpp"
#include <array>
#include <tuple>
#include <cstring>
#include <cstdlib>
#include <cmath>
#include <memory>
#ifdef _OPENMP
#include <omp.h>
#endif

using namespace hfg;

namespace hfg {

// In-element exchange operator per ((L,|M|), element), from the sign-aware
// Cholesky factor: W~(i, j) = sum_p sigma_p B(i, p) B(j, p) over the two
// channel blocks (basis.cpp:1992-2033 contracts the same factor as
// sum_p sigma_p [M0' R00 M0' - M0' R02 M2' - M2' R20 M0' + M2' R22 M2']).
// Built only when the environment variable HFGPU_EXCHANGE_OPERATOR_GIB grants
// a budget (in GiB) that holds the tables; otherwise (dense_in = false) the
// Cholesky-form in-element kernel runs, which on gfx950 is the faster of the
// two (64 vs 216 ms for N2 at lmax 16), so the operator path is opt-in.
void diatomic_build_operator(const DiatomicSetup &S, DiatomicDevice &d, hipStream_t s) {
  const int Nel = S.Nel(), nlm = (int)S.lm_map.size();
  const size_t per = (size_t)4 * KC * TILE2;
  const double bytes = 8.0 * per * nlm * Nel;
  double budget = 0.0;
  if (const char *env = std::getenv("HFGPU_EXCHANGE_OPERATOR_GIB")) budget = std::atof(env) * (1ull << 30);
  d.dense_in = false;
  d.Top.release();
  if (nlm == 0 || bytes > budget) return;
  std::vector<double> T(per * nlm * Nel, 0.0);
#pragma omp parallel for schedule(dynamic)
  for (int x = 0; x < nlm * Nel; ++x) {
    const int e = x % Nel;
    const int n = S.rad.ni[e], nn = n * n, N = 2 * nn;
    const Blk &B = S.cdB[x];
    const std::vector<double> &sg = S.cdS[x];
    std::vector<double> W((size_t)N * N, 0.0);
    for (int p = 0; p < B.c; ++p) {
      const double *bp = &B.v[(size_t)p * N];
      for (int j = 0; j < N; ++j) {
        const double f = sg[p] * bp[j];
        double *wj = &W[(size_t)j * N];
        for (int i = 0; i < N; ++i) wj[i] += f * bp[i];
      }
    }
    double *Tx = &T[per * x];
    const int xo[4] = {0, 0, nn, nn}, yo[4] = {0, nn, 0, nn};
    const double sgn[4] = {1.0, -1.0, -1.0, 1.0};
    for (int ch = 0; ch < 4; ++ch)
      for (int dd = 0; dd < n; ++dd)
        for (int cc = 0; cc < n; ++cc) {
          double *row = Tx + ((size_t)ch * KC + cc + 15 * dd) * TILE2;
          for (int b = 0; b < n; ++b)
            for (int a = 0; a < n; ++a)
              row[a + TILE * b] = sgn[ch] * W[(size_t)(xo[ch] + cc + a * n) + (size_t)(yo[ch] + b + dd * n) * N];
        }
  }
  d.Top.upload(T, s);
  hip_check(hipStreamSynchronize(s), "exchange operator upload");
  d.dense_in = true;
}

}  // namespace hfg

namespace {

// Per (j, i, L) Gaunt couplings with M = mj - mi: g0 = mod_coeff (cosh^0
// channel), g2 = coeff (cosh^2 channel), basis.cpp:1650-1665, 1908-1916.
void gaunt_tables(const DiatomicSetup &S, DiatomicDevice &d) {
  const int Na = S.Nang();
  int lmax = 0;
  for (int l : S.lval) lmax = std::max(lmax, l);
  d.gL = 2 * lmax + 3;
  d.h_g0.assign((size_t)Na * Na * d.gL, 0.0);
  d.h_g2.assign((size_t)Na * Na * d.gL, 0.0);
#pragma omp parallel for schedule(dynamic)
  for (int j = 0; j < Na; ++j)
    for (int i = 0; i < Na; ++i) {
      const int lj = S.lval[j], mj = S.mval[j], li = S.lval[i], mi = S.mval[i], M = mj - mi;
      for (int L = std::max(std::abs(lj - li) - 2, std::abs(M)); L <= lj + li + 2; ++L) {
        const size_t x = ((size_t)j * Na + i) * d.gL + L;
        d.h_g0[x] = gaunt_mod(lj, mj, L, M, li, mi);
        d.h_g2[x] = gaunt3(lj, mj, L, M, li);
      }
    }
}

void diatomic_upload(hf_diatomic *h) {
  const DiatomicSetup &S = h->host;
  DiatomicDevice &d = h->dev;
  hipStream_t s = h->ctx->cur;
  const int Nel = S.Nel(), Na = S.Nang(), nlm = (int)S.lm_map.size(), nLM = (int)S.LM_map.size();
  d.Nel = Nel;
  d.Nrad = S.Nrad();
  d.Nang = Na;
  d.n_lm = nlm;
  d.n_LM = nLM;
  d.Nbf = S.Nbf();
  for (int e = 0; e < Nel; ++e)
    if (S.rad.ni[e] > TILE) throw Error(HF_EINVAL, "elements with more than 16 functions are not supported");
  d.first.upload(S.rad.first, s);
  d.ni.upload(S.rad.ni, s);
  std::vector<int> skip(Na);
  for (int a = 0; a < Na; ++a) skip[a] = S.skip(a);
  d.skip.upload(skip, s);
  std::vector<long long> poff(S.poff.begin(), S.poff.end());
  d.poff.upload(poff, s);

  // P/Q tiles and Cholesky channel tiles
  std::vector<double> pq((size_t)std::max(nlm, 1) * Nel * 4 * TILE2, 0.0), ch, sg;
  std::vector<int> choff((size_t)std::max(nlm, 1) * Nel, 0), chrank((size_t)std::max(nlm, 1) * Nel, 0);
  int maxr = 0;
  for (int q = 0; q < nlm; ++q)
    for (int e = 0; e < Nel; ++e) {
      const size_t x = (size_t)q * Nel + e;
      const int n = S.rad.ni[e];
      const Blk *src[4] = {&S.P0[x], &S.P2[x], &S.Q0[x], &S.Q2[x]};
      for (int kind = 0; kind < 4; ++kind) {
        need(src[kind]->r == n && src[kind]->c == n, "P/Q cache has the wrong shape");
        for (int b = 0; b < n; ++b)
          for (int a = 0; a < n; ++a) pq[(x * 4 + kind) * TILE2 + a + TILE * b] = (*src[kind])(a, b);
      }
      const Blk &B = S.cdB[x];
      const int nn = n * n;
      need(B.r == 2 * nn, "Cholesky cache has the wrong number of rows");
      need((int)S.cdS[x].size() == B.c, "Cholesky signs have the wrong length");
      need(B.c <= 2 * TILE2, "Cholesky rank above 512 is not supported");
      choff[x] = (int)sg.size();
      chrank[x] = B.c;
      maxr = std::max(maxr, B.c);
      const size_t base = ch.size();
      ch.resize(base + (size_t)B.c * 2 * TILE2, 0.0);
      for (int p = 0; p < B.c; ++p) {
        double *m0 = &ch[base + (size_t)p * 2 * TILE2], *m2 = m0 + TILE2;
        for (int b = 0; b < n; ++b)
          for (int a = 0; a < n; ++a) {
            m0[a + TILE * b] = B(a + b * n, p);
            m2[a + TILE * b] = B(nn + a + b * n, p);
          }
        sg.push_back(S.cdS[x][p]);
      }
    }
  d.max_rank = maxr;
  if (ch.empty()) ch.push_back(0.0);
  if (sg.empty()) sg.push_back(0.0);
  d.pq.upload(pq, s);
  // log scale per (L,|M|, element) that brings the P and Q tiles to the same
  // magnitude, sqrt(max|P| max|Q|): P_L(cosh mu) reaches 1e75 and Q_L 1e-56
  // at L = 34, outside FP32, while their products across elements are O(1).
  // Pairs take P of the lower and Q of the upper element: the first element's Q
  // (~ mu^-|M|, 1e60 at its first points) and the last one's P have no part in it;
  // the tile that is used there is scaled to sqrt((L+|M|)!/(L-|M|)!), the usual
  // magnitude.
  {
    std::vector<double> lsig((size_t)std::max(nlm, 1) * Nel, 0.0);
    for (size_t x = 0; x < (size_t)nlm * Nel; ++x) {
      double mp = 0.0, mq = 0.0;
      for (int kind = 0; kind < 4; ++kind)
        for (int u = 0; u < TILE2; ++u) {
          const double v = std::fabs(pq[(x * 4 + kind) * TILE2 + u]);
          if (kind < 2)
            mp = std::max(mp, v);
          else
            mq = std::max(mq, v);
        }
      const int e = (int)(x % Nel);
      const double usual = -0.5 * std::log(std::fabs(S.LMfac(S.lm_map[x / Nel].first, S.lm_map[x / Nel].second)));
      if (e == 0 && mp > 0.0)
        lsig[x] = std::log(mp) - usual;
      else if (e == Nel - 1 && mq > 0.0)
        lsig[x] = usual - std::log(mq);
      else if (mp > 0.0 && mq > 0.0)
        lsig[x] = 0.5 * (std::log(mp) - std::log(mq));
    }
    d.lsig.upload(lsig, s);
  }
  d.chol.upload(ch, s);
  d.sigma.upload(sg, s);
  d.chol_off.upload(choff, s);
  d.chol_rank.upload(chrank, s);

  // Coulomb tables (basis.cpp:1633-1660, 1790-1810)
  gaunt_tables(S, d);
  const auto &lv = S.lval;
  const auto &mv = S.mval;
  std::vector<int> LMilm(std::max(nLM, 1), 0);
  std::vector<double> LMfac(std::max(nLM, 1), 0.0);
  for (int q = 0; q < nLM; ++q) {
    LMilm[q] = S.lmind(S.LM_map[q].first, S.LM_map[q].second);
    LMfac[q] = S.LMfac(S.LM_map[q].first, S.LM_map[q].second);
  }
  std::vector<std::vector<std::pair<int, std::pair<double, double>>>> pairs(nLM);
  for (int k = 0; k < Na; ++k)
    for (int l = 0; l < Na; ++l) {
      const int M = mv[k] - mv[l];
      for (int L = std::max(std::abs(lv[k] - lv[l]) - 2, std::abs(M)); L <= lv[k] + lv[l] + 2; ++L) {
        const size_t x = ((size_t)k * Na + l) * d.gL + L;
        const double c0 = d.h_g0[x], c2 = d.h_g2[x];
        if (c0 == 0.0 && c2 == 0.0) continue;
        pairs[S.LMind(L, M)].push_back({k * Na + l, {c0, c2}});
      }
    }
  std::vector<int> pstart(nLM + 1, 0), pkl;
  std::vector<double> pc;
  for (int q = 0; q < nLM; ++q) {
    for (auto &pr : pairs[q]) {
      pkl.push_back(pr.first);
      pc.push_back(pr.second.first);
      pc.push_back(pr.second.second);
    }
    pstart[q + 1] = (int)pkl.size();
  }
  std::vector<int> ostart((size_t)Na * Na + 1, 0), oq;
  std::vector<double> oc;
  for (int i = 0; i < Na; ++i)
    for (int j = 0; j < Na; ++j) {
      const int M = mv[j] - mv[i];
      for (int L = std::max(std::abs(lv[j] - lv[i]) - 2, std::abs(M)); L <= lv[j] + lv[i] + 2; ++L) {
        const size_t x = ((size_t)j * Na + i) * d.gL + L;
        const double c0 = d.h_g0[x], c2 = d.h_g2[x];
        if (c0 == 0.0 && c2 == 0.0) continue;
        oq.push_back(S.LMind(L, M));
        oc.push_back(c0);
        oc.push_back(c2);
      }
      ostart[(size_t)i * Na + j + 1] = (int)oq.size();
    }
  d.n_pairs = (int64_t)pkl.size();
  if (pkl.empty()) {
    pkl.push_back(0);
    pc.assign(2, 0.0);
  }
  if (oq.empty()) {
    oq.push_back(0);
    oc.assign(2, 0.0);
  }
  // power of two that brings the coupling factor of each (L,|M|) to [1, 4)
  d.h_fexp.assign(std::max(nlm, 1), 0);
  for (int q = 0; q < nLM; ++q)
    d.h_fexp[LMilm[q]] = LMfac[q] != 0.0 ? -2 * (int)std::floor(0.5 * std::ilogb(LMfac[q])) : 0;
  d.fexp.upload(d.h_fexp, s);
  d.LM_ilm.upload(LMilm, s);
  d.LM_fac.upload(LMfac, s);
  d.pstart.upload(pstart, s);
  d.pair_kl.upload(pkl, s);
  d.pair_c.upload(pc, s);
  d.out_start.upload(ostart, s);
  d.out_q.upload(oq, s);
  d.out_c.upload(oc, s);

  // radial RI-K flops per coupled (output block, (L,|M|)): 12 r n^3 inside
  // each element, 2 (4 ni nj^2 + 2 ni^2 nj) per element pair
  d.h_rad_in.assign(std::max(nlm, 1), 0.0);
  d.h_rad_off.assign(std::max(nlm, 1), 0.0);
  d.h_rad_low.assign(std::max(nlm, 1), 0.0);
  for (int q = 0; q < nlm; ++q) {
    double fi = 0.0, fo = 0.0, fl = 0.0;
    for (int e = 0; e < Nel; ++e) {
      const double n = S.rad.ni[e];
      fi += 12.0 * S.cdB[(size_t)q * Nel + e].c * n * n * n;
      for (int g = 0; g < Nel; ++g)
        if (g != e) {
          const double m = S.rad.ni[g], x = 2.0 * (4.0 * n * m * m + 2.0 * n * n * m);
          fo += x;
          if (e > g) fl += x;
        }
    }
    d.h_rad_in[q] = fi;
    d.h_rad_off[q] = fo;
    d.h_rad_low[q] = fl;
  }
  std::vector<int> efi, efo, efl;
  for (int e = 0; e < Nel; ++e)
    for (int f = 0; f < Nel; ++f) {
      (e == f ? efi : efo).push_back(e * Nel + f);
      if (e > f) efl.push_back(e * Nel + f);
    }
  if (efo.empty()) efo.push_back(0);
  if (efl.empty()) efl.push_back(0);
  d.ef_in.upload(efi, s);
  d.ef_off.upload(efo, s);
  d.ef_low.upload(efl, s);
  // absm mirror pairs: K(j,k) = K(jm,km) for mj, mk < 0 (basis.cpp:2067-2086)
  std::vector<int> mir;
  if (h->absm) {
    std::vector<int> partner(Na, -1);
    for (int a = 0; a < Na; ++a)
      for (int b = 0; b < Na; ++b)
        if (lv[b] == lv[a] && mv[b] == -mv[a]) {
          partner[a] = b;
          break;
        }
    for (int j = 0; j < Na; ++j) {
      if (mv[j] >= 0 || partner[j] < 0) continue;
      for (int k = 0; k < Na; ++k) {
        if (mv[k] >= 0 || partner[k] < 0) continue;
        mir.push_back(j * Na + k);
        mir.push_back(partner[j] * Na + partner[k]);
      }
    }
  }
  d.absm = h->absm;
  d.n_mirror = (int)mir.size() / 2;
  if (mir.empty()) mir.assign(2, 0);
  d.mirror.upload(mir, s);
  d.screen_mask.clear();
  d.n_act = 0;
  d.h_bnorm.alloc((size_t)Na * Na);

  d.h_stats.alloc((size_t)Na * Na * 4 * block_stats_chunks(d.Nrad));
  d.stats.alloc((size_t)Na * Na * 4 * block_stats_chunks(d.Nrad));
  d.Jin.alloc((size_t)std::max(nLM, 1) * Nel * 2 * TILE2);
  d.ds.alloc((size_t)std::max(nLM, 1) * Nel);
  d.db.alloc((size_t)std::max(nLM, 1) * Nel);
  hip_check(hipStreamSynchronize(s), "upload sync");
  diatomic_build_operator(S, d, s);
  d.op_ready = d.f32_tables = false;
  h->uploaded = true;
}

// Factorised exchange couplings of one column shell k and (L,|M|): the terms
// of output block (j,k) and (L,M) factor as fac(L,M) u(j,i) v(k,l) with u =
// (mod Gaunt, plain Gaunt) of (j,i) and v the same of (k,l)
// (basis.cpp:1905-1960), so R(j,k) = fac sum_i u(j,i) (x) V(i) with V_b(i) =
// sum_l v_b(k,l) P(i,l), and the V tiles serve every row j.  A slot is one
// (M, i); its lt entries are the (tile of (i,l), v0, v1) that pass the screen;
// a row's jt entries are (slot, fac u0, fac u1), fac times its power of two
// (h_fexp).  l_j + L + l_i is even for every coupling, so the slots of one parity
// of l_i have rows of their own.
struct CoupleGroup {
  typedef std::pair<int, std::pair<double, double>> Entry;
  int ilm, par;
  std::vector<std::pair<int, int>> slots;  // (M, i)
  std::vector<std::vector<Entry>> lt, jt;  // per slot: (tile, v); per row: (slot, c)
};

// The groups of every column shell k (ascending ilm, then parity) over its
// rows[k] (ascending shell).
std::vector<std::vector<CoupleGroup>> couple_groups(hf_diatomic *h, const std::vector<std::vector<int>> &rows,
                                                    const std::vector<int> &tile_of,
                                                    const std::vector<unsigned char> &mask,
                                                    const std::vector<int> &ilm_of,
                                                    const std::vector<double> &fac_of, int Mext, int dmoff) {
  const DiatomicSetup &S = h->host;
  const DiatomicDevice &d = h->dev;
  const int Na = S.Nang(), nlm = d.n_lm, gL = d.gL;
  const auto &lv = S.lval;
  const auto &mv = S.mval;
  std::vector<std::vector<int>> sector(2 * dmoff + 1);  // shells by m + dmoff
  for (int a = 0; a < Na; ++a) sector[mv[a] + dmoff].push_back(a);
  std::vector<std::vector<CoupleGroup>> groups(Na);
#pragma omp parallel for schedule(dynamic)
  for (int k = 0; k < Na; ++k) {
    const int mk = mv[k];
    const std::vector<int> &js = rows[k];
    if (js.empty()) continue;
    std::vector<CoupleGroup> &G = groups[k];
    std::vector<int> gidx((size_t)2 * nlm, -1);
    std::vector<int> Lk;
    for (int L = 0; L < gL; ++L)
      for (int M = -std::min(L, dmoff); M <= std::min(L, dmoff); ++M) {
        const int ml = mk - M;
        if (std::abs(ml) > dmoff / 2) continue;
        Lk.clear();
        for (int l : sector[ml + dmoff]) {
          const size_t x = ((size_t)k * Na + l) * gL + L;
          if (d.h_g0[x] != 0.0 || d.h_g2[x] != 0.0) Lk.push_back(l);
        }
        if (Lk.empty()) continue;
        const size_t lm = (size_t)L * Mext + M + dmoff;
        const int ilm = ilm_of[lm];
        const double fac = std::ldexp(fac_of[lm], d.h_fexp[ilm]);
        for (size_t q = 0; q < js.size(); ++q) {
          const int j = js[q], mi = mv[j] - M;
          if (std::abs(mi) > dmoff / 2) continue;
          for (int i : sector[mi + dmoff]) {
            const size_t xu = ((size_t)j * Na + i) * gL + L;
            const double u0 = d.h_g0[xu], u1 = d.h_g2[xu];
            if (u0 == 0.0 && u1 == 0.0) continue;
            const int par = lv[i] & 1;
            int &g = gidx[(size_t)2 * ilm + par];
            int sl = -1;
            if (g >= 0)
              for (size_t z = 0; z < G[g].slots.size(); ++z)
                if (G[g].slots[z].first == M && G[g].slots[z].second == i) {
                  sl = (int)z;
                  break;
                }
            if (sl < 0) {
              // the slot's density blocks (i,l) that pass the screen; a group
              // is opened only with its first non-empty slot
              std::vector<CoupleGroup::Entry> ltv;
              for (int l : Lk) {
                const int tl = mask[(size_t)i * Na + l] ? tile_of[(size_t)i * Na + l] : -1;
                if (tl < 0) continue;
                const size_t x = ((size_t)k * Na + l) * gL + L;
                ltv.push_back({tl, {d.h_g0[x], d.h_g2[x]}});
              }
              if (ltv.empty()) continue;
              if (g < 0) {
                g = (int)G.size();
                G.push_back(CoupleGroup{ilm, par, {}, {}, std::vector<std::vector<CoupleGroup::Entry>>(js.size())});
              }
              sl = (int)G[g].slots.size();
              G[g].slots.push_back({M, i});
              G[g].lt.push_back(std::move(ltv));
            }
            G[g].jt[q].push_back({sl, {fac * u0, fac * u1}});
          }
        }
      }
    std::sort(G.begin(), G.end(), [](const CoupleGroup &a, const CoupleGroup &b) {
      return a.ilm < b.ilm || (a.ilm == b.ilm && a.par < b.par);
    });
  }
  return groups;
}

// Lists of the two-step cross-element exchange (k_dia_k2_off) from the
// groups of every column shell.  The rows of a column with one m and parity
// of l share their slots, so they are dealt to waves in such sets (a wave
// reads each slot tile once for its rows), the waves of a workgroup divided
// over its sets so that the largest number of rows in a wave is least; a
// column with more rows than a workgroup holds gets several.  The two
// parities of an (L,|M|) share one group when their slots fit the K2_SLOTS
// tiles of LDS (half the barriers, and the rows of both parities keep all
// waves busy), else each has its own, cut again when it still does not fit
// (the sums over slots are linear).
void build_twostep(hf_diatomic *h, const std::vector<std::vector<int>> &rows,
                   const std::vector<std::vector<CoupleGroup>> &groups, hipStream_t s) {
  const DiatomicSetup &S = h->host;
  DiatomicDevice &d = h->dev;
  const int Na = S.Nang(), Nel = S.Nel();
  d.k2 = false;
  d.n_wg_k2 = 0;
  if (!d.tiled || Nel < 2 || !d.finite) return;
  if (std::getenv("HFGPU_EXCHANGE_TWOSTEP") && std::atoi(std::getenv("HFGPU_EXCHANGE_TWOSTEP")) == 0) return;
  std::vector<int> kshell, wrows, kg(1, 0), gilm, gslot(1, 0), sl(1, 0), lt, jo(1, 0), js;
  std::vector<double> ltv, jtc, kcost;
  double n_lt = 0.0, n_jt = 0.0, frad = 0.0;
  // radial products per slot (H) and per row: two 16x16x16 each
  double f_slot = 0.0, f_row = 0.0, sum_off = 0.0;
  for (int e = 0; e < Nel; ++e)
    for (int f = 0; f < Nel; ++f)
      if (d.sym ? e > f : e != f) {
        const double a = S.rad.ni[e], b = S.rad.ni[f];
        f_slot += 4.0 * a * b * b;
        f_row += 4.0 * a * a * b;
        sum_off += a * b;
      }
  typedef std::vector<std::pair<const CoupleGroup *, int>> SlotList;
  for (int k = 0; k < Na; ++k) {
    // sets of rows (positions in rows[k]) by (m, parity of l)
    std::map<std::pair<int, int>, std::vector<int>> sets;
    for (size_t q = 0; q < rows[k].size(); ++q)
      sets[{S.mval[rows[k][q]], S.lval[rows[k][q]] & 1}].push_back((int)q);
    // workgroups of whole sets, or of as much of a set as fits
    std::vector<std::vector<std::vector<int>>> wgs(1);
    int waves = 0;
    for (auto &kv : sets)
      for (size_t q0 = 0; q0 < kv.second.size();) {
        if (waves == K2_WAVES) {
          wgs.emplace_back();
          waves = 0;
        }
        const size_t q1 = std::min(kv.second.size(), q0 + (size_t)(K2_WAVES - waves) * K2_ROWS);
        wgs.back().emplace_back(kv.second.begin() + q0, kv.second.begin() + q1);
        waves += (int)((q1 - q0 + K2_ROWS - 1) / K2_ROWS);
        q0 = q1;
      }
    for (const auto &set_list : wgs) {
      if (set_list.empty()) continue;
      std::vector<int> nw;
      int used_w = 0;
      for (const auto &st : set_list) {
        nw.push_back(((int)st.size() + K2_ROWS - 1) / K2_ROWS);
        used_w += nw.back();
      }
      auto most = [&](size_t x) { return ((int)set_list[x].size() + nw[x] - 1) / nw[x]; };
      for (; used_w < K2_WAVES; ++used_w) {
        size_t best = 0;
        for (size_t x = 1; x < nw.size(); ++x)
          if (most(x) > most(best)) best = x;
        if (most(best) <= 1) break;
        ++nw[best];
      }
      std::vector<std::vector<int>> wr;  // rows of every wave
      std::vector<int> part;
      for (size_t x = 0; x < set_list.size(); ++x)
        for (int u = 0; u < nw[x]; ++u) {
          const size_t n = set_list[x].size(), a = n * u / nw[x], b = n * (u + 1) / nw[x];
          wr.emplace_back(set_list[x].begin() + a, set_list[x].begin() + b);
          part.insert(part.end(), wr.back().begin(), wr.back().end());
        }
      wr.resize(K2_WAVES);
      double cost = 0.0;
      kshell.push_back(k);
      for (const auto &w : wr)
        for (int r = 0; r < K2_ROWS; ++r) wrows.push_back(r < (int)w.size() ? rows[k][w[r]] : -1);
      auto emit = [&](int ilm, const SlotList &ss) {
        gilm.push_back(ilm);
        std::map<std::pair<const CoupleGroup *, int>, int> at;
        for (const auto &x : ss) {
          const int z = (int)at.size();
          at[x] = z;
          for (const auto &e : x.first->lt[x.second]) {
            lt.push_back(e.first);
            ltv.push_back(e.second.first);
            ltv.push_back(e.second.second);
          }
          // in fours: the padding repeats a tile of the slot with zero weights
          while (lt.size() % 4) {
            lt.push_back(lt.back());
            ltv.insert(ltv.end(), 2, 0.0);
          }
          sl.push_back((int)lt.size());
          n_lt += (double)x.first->lt[x.second].size();
          frad += f_slot;
          cost += (double)x.first->lt[x.second].size() + 8.0;
        }
        gslot.push_back((int)sl.size() - 1);
        std::vector<const CoupleGroup *> gs(1, ss.front().first);
        if (ss.back().first != ss.front().first) gs.push_back(ss.back().first);
        for (const auto &w : wr) {
          std::map<int, std::array<double, 2 * K2_ROWS>> cf;  // slot -> coefficients of the wave's rows
          for (size_t r = 0; r < w.size(); ++r) {
            bool any = false;
            for (const CoupleGroup *g : gs)
              for (const auto &e : g->jt[w[r]]) {
                const auto it = at.find({g, e.first});
                if (it == at.end()) continue;
                auto &c = cf.emplace(it->second, std::array<double, 2 * K2_ROWS>{}).first->second;
                c[2 * r] = e.second.first;
                c[2 * r + 1] = -e.second.second;
                n_jt += 1.0;
                any = true;
              }
            if (any) {
              frad += f_row;
              cost += 8.0;
            }
          }
          for (const auto &x : cf) {
            js.push_back(x.first);
            jtc.insert(jtc.end(), x.second.begin(), x.second.end());
          }
          if (js.size() % 2) {  // in twos
            js.push_back(js.back());
            jtc.insert(jtc.end(), 2 * K2_ROWS, 0.0);
          }
          cost += (double)(cf.size() * w.size());
          jo.push_back((int)js.size());
        }
      };
      const std::vector<CoupleGroup> &G = groups[k];
      for (size_t a = 0; a < G.size();) {
        size_t b = a;
        std::vector<SlotList> parts;
        size_t total = 0;
        for (; b < G.size() && G[b].ilm == G[a].ilm; ++b) {
          SlotList ss;
          std::vector<unsigned char> used(G[b].slots.size(), 0);
          for (int q : part)
            for (const auto &e : G[b].jt[q]) used[e.first] = 1;
          for (size_t z = 0; z < used.size(); ++z)
            if (used[z]) ss.push_back({&G[b], (int)z});
          total += ss.size();
          if (!ss.empty()) parts.push_back(std::move(ss));
        }
        if (parts.size() == 2 && total <= (size_t)K2_SLOTS) {
          parts[0].insert(parts[0].end(), parts[1].begin(), parts[1].end());
          parts.pop_back();
        }
        for (const SlotList &ss : parts)
          for (size_t z = 0; z < ss.size(); z += K2_SLOTS)
            emit(G[a].ilm, SlotList(ss.begin() + z, ss.begin() + std::min(ss.size(), z + K2_SLOTS)));
        a = b;
      }
      kg.push_back((int)gilm.size());
      kcost.push_back(cost);
    }
  }
  if (gilm.empty()) return;
  // workgroups: the element pairs one after another, columns in decreasing
  // cost within each, are cut into eight runs of equal cost, one per XCD (few
  // pairs' slices of the density tiles per L2); an XCD takes its run column by
  // column, so neighbouring CUs, which share a scalar cache, read the same
  // lists (N2: 5.1 ms against 5.7 pair by pair)
  std::vector<int> efs;
  for (int e = 0; e < Nel; ++e)
    for (int f = 0; f < Nel; ++f)
      if (d.sym ? e > f : e != f) efs.push_back(e * Nel + f);
  std::vector<int> korder(kshell.size());
  double ktot = 0.0;
  for (size_t q = 0; q < korder.size(); ++q) {
    korder[q] = (int)q;
    ktot += kcost[q];
  }
  std::sort(korder.begin(), korder.end(), [&](int a, int b) { return kcost[a] > kcost[b]; });
  std::vector<std::vector<std::pair<int, int>>> per_xcd(8);  // (position in korder, element pair)
  double done = 0.0;
  const double all = ktot * (double)efs.size();
  for (int ef : efs)
    for (size_t q = 0; q < korder.size(); ++q) {
      const double c = kcost[korder[q]];
      per_xcd[std::min(7, (int)(8.0 * (done + 0.5 * c) / all))].push_back({(int)q, ef});
      done += c;
    }
  size_t mx = 0;
  for (auto &v : per_xcd) mx = std::max(mx, v.size());
  std::vector<int> wg(mx * 8 * 2, -1);
  for (int x = 0; x < 8; ++x) {
    std::stable_sort(per_xcd[x].begin(), per_xcd[x].end());
    for (size_t q = 0; q < per_xcd[x].size(); ++q) {
      wg[(q * 8 + x) * 2] = korder[per_xcd[x][q].first];
      wg[(q * 8 + x) * 2 + 1] = per_xcd[x][q].second;
    }
  }
  d.k2_wg.upload(wg, s);
  d.k2_kshell.upload(kshell, s);
  d.k2_rows.upload(wrows, s);
  d.k2_kg.upload(kg, s);
  d.k2_gilm.upload(gilm, s);
  d.k2_gslot.upload(gslot, s);
  d.k2_sl.upload(sl, s);
  d.k2_lt.upload(lt, s);
  d.k2_ltv.upload(ltv, s);
  d.k2_jo.upload(jo, s);
  d.k2_js.upload(js, s);
  d.k2_jtc.upload(jtc, s);
  hip_check(hipStreamSynchronize(s), "two-step list upload");  // before the host lists go
  d.n_wg_k2 = (int)(mx * 8);
  // per element pair and tile entry 4 flops per lt entry (two channels) and
  // 4 per jt entry (two row sums), plus the radial products
  d.flops_off_k2 = frad + 4.0 * (n_lt + n_jt) * sum_off;
  d.k2 = true;
}

// Lists of the folded-operator in-element exchange (k_dia_kin_fold) from the
// groups of every column shell: the rows of a group go in units of two, which
// share the group's slots, the units of one (L,|M|) in workgroups of
// KF_WAVES per element.  In the symmetric mode only the rows j <= k.
void build_fold(hf_diatomic *h, const std::vector<std::vector<int>> &rows,
                const std::vector<std::vector<CoupleGroup>> &groups, hipStream_t s) {
  const DiatomicSetup &S = h->host;
  DiatomicDevice &d = h->dev;
  const int Na = S.Nang(), Nel = S.Nel(), nlm = d.n_lm;
  d.n_wg_kf = 0;
  if (!d.list_fold || !d.tiled || !d.finite || d.dense_in) return;
  struct Unit {
    int jk[KF_ROWS];
    std::vector<int4> rec;
    std::vector<std::array<double, 2 * KF_ROWS>> u;
  };
  std::vector<std::vector<Unit>> units(nlm);
  std::vector<int4> more;
  std::vector<double> v;
  double f_gather = 0.0;
  std::vector<double> f_op(Nel);
  for (int e = 0; e < Nel; ++e) {
    const double n = S.rad.ni[e], ns = n * (n + 1) / 2, na = n * (n - 1) / 2;
    f_op[e] = 2.0 * (ns * (2 * ns + n * n) + na * (2 * na + n * n));
  }
  double n_rows = 0.0;
  for (int k = 0; k < Na; ++k) {
    std::map<std::vector<double>, int> runs;  // weight runs of this column
    for (const CoupleGroup &G : groups[k]) {
      std::vector<int> rr;
      for (size_t q = 0; q < rows[k].size(); ++q)
        if (!G.jt[q].empty() && (!d.sym || rows[k][q] <= k)) rr.push_back((int)q);
      std::vector<int4> rec(G.slots.size(), make_int4(-1, 0, 0, -1));
      auto record = [&](int z) {
        if (rec[z].x >= 0) return rec[z];
        // runs of consecutive tiles, the later ones chained
        std::vector<int4> parts;
        const auto &lt = G.lt[z];
        for (size_t a = 0; a < lt.size();) {
          size_t b = a + 1;
          while (b < lt.size() && lt[b].first == lt[b - 1].first + 1) ++b;
          std::vector<double> w;
          for (size_t x = a; x < b; ++x) {
            w.push_back(lt[x].second.first);
            w.push_back(lt[x].second.second);
          }
          const auto ins = runs.emplace(w, (int)v.size() / 2);
          if (ins.second) {
            v.insert(v.end(), w.begin(), w.end());
            while (v.size() % 8) v.push_back(0.0);
          }
          parts.push_back(make_int4(lt[a].first, (int)(b - a), ins.first->second, -1));
          a = b;
        }
        for (size_t x = parts.size() - 1; x > 0; --x) {
          parts[x - 1].w = (int)more.size();
          more.push_back(parts[x]);
        }
        return rec[z] = parts[0];
      };
      for (size_t a = 0; a < rr.size(); a += KF_ROWS) {
        Unit U;
        std::map<int, std::array<double, 2 * KF_ROWS>> co;
        for (int r = 0; r < KF_ROWS; ++r) {
          const bool have = a + r < rr.size();
          U.jk[r] = have ? rows[k][rr[a + r]] * Na + k : -1;
          if (!have) continue;
          n_rows += 1.0;
          for (const auto &e : G.jt[rr[a + r]]) {
            auto &q = co.emplace(e.first, std::array<double, 2 * KF_ROWS>{}).first->second;
            q[2 * r] = e.second.first;
            q[2 * r + 1] = e.second.second;
            f_gather += 8.0;
          }
        }
        for (const auto &x : co) {
          U.rec.push_back(record(x.first));
          U.u.push_back(x.second);
          f_gather += 4.0 * (double)G.lt[x.first].size();
        }
        units[G.ilm].push_back(std::move(U));
      }
    }
  }
  std::vector<int> jk, ent(1, 0);
  std::vector<int4> rec;
  std::vector<double> u;
  // workgroups: element e's on XCD e % 8, (L,|M|) by (L,|M|), so the
  // workgroups of one operator run together and share it in that XCD's L2
  std::vector<std::vector<int4>> per_xcd(8);
  for (int q = 0; q < nlm; ++q) {
    const int u0 = (int)jk.size() / KF_ROWS, nu = (int)units[q].size();
    for (const Unit &U : units[q]) {
      jk.insert(jk.end(), U.jk, U.jk + KF_ROWS);
      rec.insert(rec.end(), U.rec.begin(), U.rec.end());
      for (const auto &c : U.u) u.insert(u.end(), c.begin(), c.end());
      ent.push_back((int)rec.size());
    }
    for (int e = 0; e < Nel; ++e)
      for (int b = 0; b < nu; b += KF_WAVES)
        per_xcd[e % 8].push_back(make_int4(q, e, u0 + b, std::min(KF_WAVES, nu - b)));
  }
  if (rec.empty()) return;
  size_t mx = 0;
  for (auto &x : per_xcd) mx = std::max(mx, x.size());
  std::vector<int4> wg(mx * 8, make_int4(-1, 0, 0, 0));
  for (int x = 0; x < 8; ++x)
    for (size_t q = 0; q < per_xcd[x].size(); ++q) wg[q * 8 + x] = per_xcd[x][q];
  if (more.empty()) more.push_back(make_int4(0, 0, 0, -1));
  d.wg_kf.upload(wg, s);
  d.kf_jk.upload(jk, s);
  d.kf_ent.upload(ent, s);
  d.kf_rec.upload(rec, s);
  d.kf_more.upload(more, s);
  d.kf_u.upload(u, s);
  d.kf_v.upload(v, s);
  hip_check(hipStreamSynchronize(s), "folded exchange list upload");  // before the host lists go
  d.flops_in_kf = 0.0;
  for (int e = 0; e < Nel; ++e) d.flops_in_kf += n_rows * f_op[e] + f_gather * S.rad.ni[e] * S.rad.ni[e];
  d.n_wg_kf = (int)wg.size();
}

// Exchange coupling lists for the density blocks that pass the norm screen
// (|P_il|_F >= 10 eps, basis.cpp:1858-1875).  For each output block (j,k):
// runs of terms per (L,|M|), each term a density block (i,l) with
// mi - ml = mj - mk and the four channel weights LMfac * {mji mkl, -mji gkl,
// -gji mkl, gji gkl} (basis.cpp:1905-1960).  Rebuilt only when the screening
// pattern changes.
void build_exchange_lists(hf_diatomic *h, hipStream_t s) {
  const DiatomicSetup &S = h->host;
  DiatomicDevice &d = h->dev;
  const int Na = S.Nang(), nlm = d.n_lm;
  const auto &lv = S.lval;
  const auto &mv = S.mval;
  std::vector<unsigned char> mask((size_t)Na * Na);
  const double thr = 10.0 * 2.220446049250313e-16;
  for (size_t q = 0; q < mask.size(); ++q) mask[q] = d.h_bnorm.p[q] >= thr ? 1 : 0;
  // the symmetric exchange needs the mirror of every coupled block coupled
  if (d.sym)
    for (int i = 0; i < Na; ++i)
      for (int l = 0; l < i; ++l) {
        const unsigned char m = mask[(size_t)i * Na + l] | mask[(size_t)l * Na + i];
        mask[(size_t)i * Na + l] = mask[(size_t)l * Na + i] = m;
      }
  // a density with infinities or NaNs (or beyond FP32's range) takes the
  // one-step kernels, whose sums hold exactly the coupled terms (no padding,
  // no shared rows)
  bool finite = true;
  for (size_t q = 0; q < mask.size(); ++q) finite = finite && d.h_bnorm.p[q] < 1e30;
  if (!d.screen_mask.empty() && mask == d.screen_mask && d.sym == d.list_sym && finite == d.finite &&
      (d.fold_in ? d.list_fold : d.list_terms))
    return;
  d.finite = finite;
  // the lists serve both precisions where one has the folded operators and the
  // other does not
  d.list_fold = d.fold_state[0] == 1 || d.fold_state[1] == 1;
  const bool want_terms = d.fold_state[0] == -1 || d.fold_state[1] == -1;
  d.screen_mask.clear();  // no lists until all of them are there
  auto done = [&] {
    d.screen_mask = mask;
    d.list_sym = d.sym;
    ++d.list_gen;
  };
  int mabs = 0;
  for (int m : mv) mabs = std::max(mabs, std::abs(m));
  const int dmoff = 2 * mabs;
  std::vector<std::vector<int>> bydm(4 * mabs + 1);
  for (int i = 0; i < Na; ++i)
    for (int l = 0; l < Na; ++l)
      if (mask[(size_t)i * Na + l]) bydm[mv[i] - mv[l] + dmoff].push_back(i * Na + l);
  // (L, M) -> ilm and LMfac lookups
  const int Lext = d.gL, Mext = 2 * dmoff + 1;
  std::vector<int> ilm_of((size_t)Lext * Mext, -1);
  std::vector<double> fac_of((size_t)Lext * Mext, 0.0);
  for (auto &e : S.LM_map)
    if (e.first < Lext && std::abs(e.second) <= dmoff) {
      ilm_of[(size_t)e.first * Mext + e.second + dmoff] = S.lmind(e.first, e.second);
      fac_of[(size_t)e.first * Mext + e.second + dmoff] = S.LMfac(e.first, e.second);
    }
  // density tiles of the coupled blocks: by row shell, then m, parity and l of
  // the column shell, so the sources of one slot are consecutive tiles
  std::vector<int> id((size_t)Na * Na, -1), src;
  for (const auto &v : bydm) src.insert(src.end(), v.begin(), v.end());
  std::sort(src.begin(), src.end(), [&](int x, int y) {
    const int i = x / Na, j = y / Na, a = x % Na, b = y % Na;
    return std::make_tuple(i, mv[a], lv[a] & 1, lv[a], a) < std::make_tuple(j, mv[b], lv[b] & 1, lv[b], b);
  });
  for (size_t q = 0; q < src.size(); ++q) id[src[q]] = (int)q;
  const double bytes = (double)src.size() * S.Nel() * S.Nel() * TILE2 * sizeof(double);
  d.tiled = bytes <= exchange_tile_budget(d.ptile.n * sizeof(double) + d.ptile32.n * sizeof(float));
  d.n_src = (int)src.size();
  if (src.empty()) src.push_back(0);
  d.src_blk.upload(src, s);
  hip_check(hipStreamSynchronize(s), "exchange source upload");
  // factorised couplings of every output block that m allows; those with any
  // are the active ones
  const int njk = Na * Na;
  std::vector<int> act;
  {
    std::vector<std::vector<int>> rows(Na);  // of every column shell k
    for (int k = 0; k < Na; ++k)
      for (int j = 0; j < Na; ++j) {
        if (h->absm && (mv[j] < 0 || mv[k] < 0)) continue;
        const int dm = mv[j] - mv[k];
        if (std::abs(dm) <= 2 * mabs && !bydm[dm + dmoff].empty()) rows[k].push_back(j);
      }
    const auto groups = couple_groups(h, rows, id, mask, ilm_of, fac_of, Mext, dmoff);
    // work: radial flops per (block, (L,|M|)) run, 4 channels x 2 flops per term
    // and tile entry for the Gaunt-weighted density sums
    double frad_in = 0.0, frad_off = 0.0;
    int64_t nterm = 0, nterm_in = 0, nrun = 0;
    std::vector<unsigned char> active(njk, 0);
    for (int k = 0; k < Na; ++k) {
      std::vector<int> last(rows[k].size(), -1);
      for (const CoupleGroup &G : groups[k])
        for (size_t q = 0; q < rows[k].size(); ++q) {
          if (G.jt[q].empty()) continue;
          const bool in_done = !d.sym || rows[k][q] <= k;
          int64_t n = 0;
          for (const auto &e : G.jt[q]) n += (int64_t)G.lt[e.first].size();
          nterm += n;
          if (in_done) nterm_in += n;
          if (last[q] != G.ilm) {
            last[q] = G.ilm;
            ++nrun;
            if (in_done) frad_in += d.h_rad_in[G.ilm];
            frad_off += d.sym ? d.h_rad_low[G.ilm] : d.h_rad_off[G.ilm];
          }
          active[rows[k][q] * Na + k] = 1;
        }
    }
    for (int jk = 0; jk < njk; ++jk)
      if (active[jk]) act.push_back(jk);
    d.n_act = (int)act.size();
    d.n_runs = nrun;
    d.n_terms = nterm;
    double sum_in = 0.0, sum_off = 0.0;
    for (int e = 0; e < S.Nel(); ++e) {
      sum_in += (double)S.rad.ni[e] * S.rad.ni[e];
      for (int f = 0; f < S.Nel(); ++f)
        if (d.sym ? e > f : e != f) sum_off += (double)S.rad.ni[e] * S.rad.ni[f];
    }
    d.flops_in = frad_in + 8.0 * (double)nterm_in * sum_in;
    d.flops_off = frad_off + 8.0 * (double)nterm * sum_off;
    d.flops_k_angular = 8.0 * ((double)nterm_in * sum_in + (double)nterm * sum_off);
    d.flops_k_radial = frad_in + frad_off;
    build_twostep(h, rows, groups, s);
    build_fold(h, rows, groups, s);
  }
  // the lists of every single term only for the kernels that read them (N2:
  // 3.8 M terms, 0.2 GB): the one-step, Cholesky-form and dense ones
  d.n_wg_kl = 0;
  d.n_wg_op = 0;
  d.list_terms = act.empty() || want_terms || !((S.Nel() < 2 || d.k2) && d.n_wg_kf > 0);
  if (act.empty() || !d.list_terms) {
    done();
    return;
  }
  struct Term {
    int ilm, il;
    double f[4];
  };
  std::vector<std::vector<Term>> per(njk);
#pragma omp parallel for schedule(dynamic, 4)
  for (int jk = 0; jk < njk; ++jk) {
    const int j = jk / Na, k = jk - j * Na;
    const int lj = lv[j], mj = mv[j], lk = lv[k], mk = mv[k];
    if (h->absm && (mj < 0 || mk < 0)) continue;
    const int dm = mj - mk;
    if (std::abs(dm) > 2 * mabs) continue;
    std::vector<Term> &out = per[jk];
    for (int il : bydm[dm + dmoff]) {
      const int i = il / Na, l = il - i * Na;
      const int li = lv[i], mi = mv[i], ll = lv[l], ml = mv[l], M = mj - mi;
      const int Lmin = std::max(std::max(std::abs(li - lj), std::abs(lk - ll)) - 2, std::abs(M));
      const int Lmax = std::min(li + lj, lk + ll) + 2;
      const size_t gji = ((size_t)j * Na + i) * Lext, gkl = ((size_t)k * Na + l) * Lext;
      for (int L = Lmin; L <= Lmax; ++L) {
        const double mji = d.h_g0[gji + L], g_ji = d.h_g2[gji + L];
        const double mkl = d.h_g0[gkl + L], g_kl = d.h_g2[gkl + L];
        const double c00 = mji * mkl, c02 = -mji * g_kl, c20 = -g_ji * mkl, c22 = g_ji * g_kl;
        if (c00 == 0.0 && c02 == 0.0 && c20 == 0.0 && c22 == 0.0) continue;
        const size_t lm = (size_t)L * Mext + M + dmoff;
        const double fac = fac_of[lm];
        out.push_back({ilm_of[lm], il, {fac * c00, fac * c02, fac * c20, fac * c22}});
      }
    }
    std::stable_sort(out.begin(), out.end(), [](const Term &a, const Term &b) { return a.ilm < b.ilm; });
  }
  std::vector<int> lstart(1, 0), rilm, rstart(1, 0), til;
  std::vector<double> tf;
  act.clear();
  for (int jk = 0; jk < njk; ++jk) {
    const std::vector<Term> &v = per[jk];
    if (v.empty()) continue;
    act.push_back(jk);
    for (size_t a = 0; a < v.size();) {
      size_t b = a;
      while (b < v.size() && v[b].ilm == v[a].ilm) {
        til.push_back(v[b].il);
        tf.insert(tf.end(), v[b].f, v[b].f + 4);
        ++b;
      }
      rilm.push_back(v[a].ilm);
      rstart.push_back((int)til.size());
      a = b;
    }
    lstart.push_back((int)rilm.size());
  }
  d.n_act = (int)act.size();
  d.n_runs = (int64_t)rilm.size();
  // dense in-element path: runs grouped by (L,|M|); one workgroup per
  // (ilm, element, 32 runs), groups dealt round-robin to the 8 XCDs so the
  // workgroups sharing one operator table run on the same L2
  if (d.dense_in && d.n_runs > 0) {
    const int Nel = S.Nel();
    std::vector<int> rs(nlm + 1, 0), runs(rilm.size());
    for (int r : rilm) ++rs[r + 1];
    for (int q = 0; q < nlm; ++q) rs[q + 1] += rs[q];
    std::vector<int> fill(rs.begin(), rs.end() - 1);
    for (size_t r = 0; r < rilm.size(); ++r) runs[fill[rilm[r]]++] = (int)r;
    std::vector<std::vector<int>> per_xcd(8);
    int grp = 0;
    for (int q = 0; q < nlm; ++q) {
      const int nr = rs[q + 1] - rs[q];
      if (!nr) continue;
      for (int e = 0; e < Nel; ++e, ++grp)
        for (int c0 = 0; c0 < nr; c0 += 32) {
          auto &v = per_xcd[grp % 8];
          v.push_back(q);
          v.push_back(e);
          v.push_back(c0);
        }
    }
    size_t mx = 0;
    for (auto &v : per_xcd) mx = std::max(mx, v.size() / 3);
    std::vector<int> wg(mx * 8 * 3, -1);
    for (int x = 0; x < 8; ++x)
      for (size_t j = 0; j < per_xcd[x].size() / 3; ++j)
        for (int u = 0; u < 3; ++u) wg[(j * 8 + x) * 3 + u] = per_xcd[x][3 * j + u];
    d.n_wg_in = (int)(mx * 8);
    d.ilm_rstart.upload(rs, s);
    d.ilm_runs.upload(runs, s);
    d.wg_in.upload(wg, s);
    d.Ypart.alloc((size_t)d.n_runs * Nel * TILE2);
    // the dense operator replaces 12 r n^3 by 8 n^4 per (run, element)
    double fr = 0.0;
    for (int e = 0; e < Nel; ++e) fr += 8.0 * std::pow((double)S.rad.ni[e], 4);
    double sum_in = 0.0;
    for (int e = 0; e < Nel; ++e) sum_in += (double)S.rad.ni[e] * S.rad.ni[e];
    d.flops_in = (double)d.n_runs * fr + 8.0 * (double)d.n_terms * sum_in;
  }
  // in-element workgroups of the LDS-resident kernel: runs grouped by ilm,
  // batches of KL_BATCH per (ilm, element), element e's batches on XCD e % 8
  if (!d.dense_in && d.max_rank <= KL_RANK_MAX && !rilm.empty()) {
    const int Nel = S.Nel(), nr = (int)rilm.size();
    std::vector<int> run_act(nr), cnt(nlm + 1, 0), runs;
    std::vector<unsigned char> keep(nr, 1);
    for (size_t a = 0; a < act.size(); ++a)
      for (int r = lstart[a]; r < lstart[a + 1]; ++r) {
        run_act[r] = (int)a;
        if (d.sym && act[a] / Na > act[a] % Na) keep[r] = 0;  // the mirror of block (k, j) covers it
      }
    for (int r = 0; r < nr; ++r)
      if (keep[r]) ++cnt[rilm[r] + 1];
    for (int q = 0; q < nlm; ++q) cnt[q + 1] += cnt[q];
    runs.resize(cnt[nlm]);
    std::vector<int> fill(cnt.begin(), cnt.end() - 1);
    for (int r = 0; r < nr; ++r)
      if (keep[r]) runs[fill[rilm[r]]++] = r;
    if (runs.empty()) runs.push_back(0);
    std::vector<std::vector<int>> per_xcd(8);
    for (int q = 0; q < nlm; ++q)
      for (int e = 0; e < Nel; ++e)
        for (int b = cnt[q]; b < cnt[q + 1]; b += KL_BATCH) {
          auto &v = per_xcd[e % 8];
          v.insert(v.end(), {q, e, b, std::min(KL_BATCH, cnt[q + 1] - b)});
        }
    size_t mx = 0;
    for (auto &v : per_xcd) mx = std::max(mx, v.size() / 4);
    std::vector<int> wg(mx * 8 * 4, -1);
    for (int x = 0; x < 8; ++x)
      for (size_t j = 0; j < per_xcd[x].size() / 4; ++j)
        for (int u = 0; u < 4; ++u) wg[(j * 8 + x) * 4 + u] = per_xcd[x][4 * j + u];
    d.wg_kl.upload(wg, s);
    d.kl_runs.upload(runs, s);
    d.run_act.upload(run_act, s);
    d.n_wg_kl = (int)(mx * 8);
    // the matrix-core operator form: OP_RUNS runs per workgroup, the groups
    // of one (ilm, element) dealt to one XCD so they share its operator in L2
    if (d.op_in) {
      std::vector<std::vector<int>> px(8);
      int grp = 0;
      for (int q = 0; q < nlm; ++q)
        for (int e = 0; e < Nel; ++e) {
          if (cnt[q + 1] == cnt[q]) continue;
          auto &v = px[grp++ % 8];
          for (int b = cnt[q]; b < cnt[q + 1]; b += OP_RUNS)
            v.insert(v.end(), {q, e, b, std::min(OP_RUNS, cnt[q + 1] - b)});
        }
      size_t mo = 0;
      for (auto &v : px) mo = std::max(mo, v.size() / 4);
      std::vector<int> wo(mo * 8 * 4, -1);
      for (int xc = 0; xc < 8; ++xc)
        for (size_t j = 0; j < px[xc].size() / 4; ++j)
          for (int u = 0; u < 4; ++u) wo[(j * 8 + xc) * 4 + u] = px[xc][4 * j + u];
      d.wg_op.upload(wo, s);
      d.n_wg_op = (int)(mo * 8);
    }
  }
  if (act.empty()) act.push_back(0);
  if (rilm.empty()) rilm.push_back(0);
  if (til.empty()) {
    til.push_back(0);
    tf.assign(4, 0.0);
  }
  d.act_jk.upload(act, s);
  d.act_lstart.upload(lstart, s);
  d.lrun_ilm.upload(rilm, s);
  d.lrun_tstart.upload(rstart, s);
  d.term_il.upload(til, s);
  std::vector<int4> tpos(til.size());
  std::vector<int> tt(til.size());  // each term's tile
  for (size_t q = 0; q < til.size(); ++q) {
    const int i = til[q] / Na, l = til[q] % Na;
    tpos[q] = make_int4((int)S.poff[i], (int)(S.poff[l] - S.skip(l)), S.skip(i), S.skip(l));
    tt[q] = id[til[q]];
  }
  d.term_pos.upload(tpos, s);
  d.term_tile.upload(tt, s);
  d.term_f.upload(tf, s);
  hip_check(hipStreamSynchronize(s), "exchange list upload");
  done();
}

void ensure_ready(hf_diatomic *h) {
  if (!h->ctx) throw Error(HF_ESTATE, "handle was created without a device context");
  if (!h->host.have_tei) throw Error(HF_ESTATE, "Primitive teis have not been computed!");
  if (!h->uploaded) diatomic_upload(h);
}

// whether the folded operators keep FP32's accuracy on this basis
bool fold_fp32(const DiatomicSetup &S) {
  for (int e = 0; e < S.Nel(); ++e)
    if (S.rad.ni[e] < KF_MIN_N32 || S.rad.bval[e + 1] - S.rad.bval[e] > KF_MAX_MU32) return false;
  return true;
}

void exchange_launch(hf_diatomic *h, const double *P, int64_t ldp, double *K, int64_t ldk, bool fp32 = false) {
  DiatomicDevice &d = h->dev;
  hipStream_t s = h->ctx->cur;
  if (!d.op_ready) {
    // before the first exchange of these tables (density-functional builds
    // without exact exchange never need it)
    diatomic_op_build(d, h->host.rad.ni, s);
    d.op_ready = true;
  }
  d.fold_in = diatomic_fold_ready(d, fp32, !d.dense_in && (!fp32 || fold_fp32(h->host)), s);
  block_stats_launch(P, ldp, d.Nrad, d.Nang, d.skip.p, d.poff.p, d.stats.p, d.h_stats.p, s);
  hip_check(hipStreamSynchronize(s), "block statistics sync");
  const bool symmetric = block_stats_reduce(d.h_stats.p, d.Nrad, d.Nang, d.h_bnorm.p);
  d.sym = !d.dense_in && symmetric_exchange_allowed() && symmetric;
  build_exchange_lists(h, s);
  diatomic_exchange_kernels(d, P, ldp, K, ldk, s, &h->ctx->timer, fp32);
}

hf_diatomic *checked(hf_diatomic *h) {
  need(h != nullptr, "NULL handle");
  need(h->ctx != nullptr, "handle was created without a device context");
  return h;
}

}  // namespace

extern "C" {

int hf_diatomic_create(hf_ctx *ctx, int Z1, int Z2, double Rhalf, int nnodes, int nquad, const double *bval,
                       int nbval, const int *lval, const int *mval, int nang, hf_diatomic **out) {
  return guarded([&] {
    need(bval && lval && mval && out, "NULL argument");
    need(nbval >= 2, "need at least one element (nbval >= 2)");
    need(nang >= 1, "need at least one angular shell");
    need(nnodes >= 2 && nnodes <= TILE, "nnodes must be in [2, 16]");
    need(Z1 >= 0 && Z2 >= 0, "nuclear charges must be non-negative");
    need(Rhalf > 0.0, "Rhalf must be positive");
    for (int i = 0; i + 1 < nbval; ++i) need(bval[i + 1] > bval[i], "element boundaries must increase");
    need(bval[0] == 0.0, "the first element boundary must be mu=0");
    std::unique_ptr<hf_diatomic> h(new hf_diatomic);
    h->ctx = ctx;
    h->host.build(Z1, Z2, Rhalf, nnodes, nquad > 0 ? nquad : 5 * nnodes, std::vector<double>(bval, bval + nbval),
                  std::vector<int>(lval, lval + nang), std::vector<int>(mval, mval + nang));
    *out = h.release();
  });
}

int hf_diatomic_destroy(hf_diatomic *h) {
  return guarded([&] {
    if (!h) return;
    if (h->ctx) {
      DeviceGuard g(h->ctx->device);
      (void)hipStreamSynchronize(h->ctx->cur);
    }
    delete h;
  });
}

int hf_diatomic_sizes(const hf_diatomic *h, int64_t out[7]) {
  return guarded([&] {
    need(h && out, "NULL argument");
    out[0] = h->host.Nbf();
    out[1] = h->host.Ndummy();
    out[2] = h->host.Nrad();
    out[3] = h->host.Nang();
    out[4] = h->host.Nel();
    out[5] = (int64_t)h->host.lm_map.size();
    out[6] = (int64_t)h->host.LM_map.size();
  });
}

int hf_diatomic_pure_index(const hf_diatomic *h, int64_t *idx) {
  return guarded([&] {
    need(h && idx, "NULL argument");
    const DiatomicSetup &S = h->host;
    int64_t q = 0;
    for (int a = 0; a < S.Nang(); ++a)
      for (int r = S.skip(a); r < S.Nrad(); ++r) idx[q++] = (int64_t)a * S.Nrad() + r;
  });
}

int hf_diatomic_maps(const hf_diatomic *h, int *lm, int *LM) {
  return guarded([&] {
    need(h != nullptr, "NULL handle");
    const DiatomicSetup &S = h->host;
    if (lm)
      for (size_t i = 0; i < S.lm_map.size(); ++i) {
        lm[2 * i] = S.lm_map[i].first;
        lm[2 * i + 1] = S.lm_map[i].second;
      }
    if (LM)
      for (size_t i = 0; i < S.LM_map.size(); ++i) {
        LM[2 * i] = S.LM_map[i].first;
        LM[2 * i + 1] = S.LM_map[i].second;
      }
  });
}

int hf_diatomic_set_absm_symmetric(hf_diatomic *h, int sym) {
  return guarded([&] {
    need(h != nullptr, "NULL handle");
    if (h->absm != (sym != 0)) {
      h->absm = sym != 0;
      h->uploaded = false;
    }
  });
}

int hf_diatomic_compute_tei(hf_diatomic *h, int exchange) {
  (void)exchange;
  return guarded([&] {
    need(h != nullptr, "NULL handle");
    h->host.compute_tei();
    h->uploaded = false;
  });
}

int hf_diatomic_compute_tei_device(hf_diatomic *h, double *seconds) {
  return guarded([&] {
    need(h != nullptr, "NULL handle");
    need(h->ctx != nullptr, "handle was created without a device context");
    DeviceGuard g(h->ctx->device);
    diatomic_tei_device(h->host, h->ctx->cur, seconds);
    h->uploaded = false;
  });
}

int hf_diatomic_get_cache(const hf_diatomic *h, int kind, int ilm, int iel, int dims[2], double *data) {
  return guarded([&] {
    need(h && dims, "NULL argument");
    const DiatomicSetup &S = h->host;
    need(kind >= 0 && kind <= 5, "kind must be in 0..5");
    need(ilm >= 0 && ilm < (int)S.lm_map.size() && iel >= 0 && iel < S.Nel(), "(ilm, iel) out of range");
    if (!S.have_tei) throw Error(HF_ESTATE, "Primitive teis have not been computed!");
    const size_t x = (size_t)ilm * S.Nel() + iel;
    if (kind == 5) {
      dims[0] = (int)S.cdS[x].size();
      dims[1] = 1;
      if (data && dims[0]) std::memcpy(data, S.cdS[x].data(), sizeof(double) * S.cdS[x].size());
      return;
    }
    const Blk &b = kind == 0 ? S.P0[x] : kind == 1 ? S.P2[x] : kind == 2 ? S.Q0[x] : kind == 3 ? S.Q2[x] : S.cdB[x];
    dims[0] = b.r;
    dims[1] = b.c;
    if (data && !b.v.empty()) std::memcpy(data, b.v.data(), sizeof(double) * b.v.size());
  });
}

int hf_diatomic_one_electron(const hf_diatomic *h, int which, double *out, int64_t ld) {
  return guarded([&] {
    need(h != nullptr, "NULL handle");
    check_matrix(out, ld, h->host.Nbf(), "out");
    if (which == 0)
      h->host.overlap(out, ld);
    else if (which == 1)
      h->host.kinetic(out, ld);
    else if (which == 2)
      h->host.nuclear(out, ld);
    else
      throw Error(HF_EINVAL, "which must be 0 (overlap), 1 (kinetic) or 2 (nuclear)");
  });
}

int hf_diatomic_work(hf_diatomic *h, double out[4]) {
  return guarded([&] {
    checked(h);
    out[0] = h->dev.flops_k_angular;
    out[1] = h->dev.flops_k_radial;
    out[2] = (double)h->dev.n_terms;
    out[3] = (double)h->dev.n_act;
  });
}

int hf_diatomic_one_electron_dev(const hf_diatomic *h, int which, double *dOut, int64_t ld) {
  return guarded([&] {
    need(h != nullptr, "NULL handle");
    need(h->ctx != nullptr, "handle was created without a device context");
    need(which >= 0 && which <= 2, "which must be 0 (overlap), 1 (kinetic) or 2 (nuclear)");
    DeviceGuard g(h->ctx->device);
    check_matrix(dOut, ld, h->host.Nbf(), "out");
    BlockList b;
    h->host.one_electron_blocks(which, b);
    scatter_blocks_launch(dOut, ld, h->host.Nbf(), b.meta, b.vals, h->ctx->cur);
  });
}

int hf_diatomic_coulomb_dev(hf_diatomic *h, const double *dP, int64_t ldp, double *dJ, int64_t ldj) {
  return guarded([&] {
    checked(h);
    DeviceGuard g(h->ctx->device);
    ensure_ready(h);
    check_matrix(dP, ldp, h->host.Nbf(), "P");
    check_matrix(dJ, ldj, h->host.Nbf(), "J");
    diatomic_coulomb_launch(h->dev, dP, ldp, dJ, ldj, h->ctx->cur, &h->ctx->timer);
  });
}

int hf_diatomic_exchange_dev(hf_diatomic *h, const double *dP, int64_t ldp, double *dK, int64_t ldk) {
  return guarded([&] {
    checked(h);
    DeviceGuard g(h->ctx->device);
    ensure_ready(h);
    check_matrix(dP, ldp, h->host.Nbf(), "P");
    check_matrix(dK, ldk, h->host.Nbf(), "K");
    exchange_launch(h, dP, ldp, dK, ldk);
  });
}

int hf_diatomic_coulomb(hf_diatomic *h, const double *P, int64_t ldp, double *J, int64_t ldj) {
  return guarded([&] {
    checked(h);
    DeviceGuard g(h->ctx->device);
    ensure_ready(h);
    host_roundtrip(h->ctx->cur, h->host.Nbf(), h->dev.hostP, h->dev.hostOut, P, ldp, J, ldj,
                   [&](const double *dp, int64_t lp, double *dout, int64_t lo) {
                     diatomic_coulomb_launch(h->dev, dp, lp, dout, lo, h->ctx->cur, &h->ctx->timer);
                   });
  });
}

int hf_diatomic_exchange_fp32_dev(hf_diatomic *h, const double *dP, int64_t ldp, double *dK, int64_t ldk) {
  return guarded([&] {
    checked(h);
    DeviceGuard g(h->ctx->device);
    ensure_ready(h);
    check_matrix(dP, ldp, h->host.Nbf(), "P");
    check_matrix(dK, ldk, h->host.Nbf(), "K");
    exchange_launch(h, dP, ldp, dK, ldk, true);
  });
}

int hf_diatomic_exchange(hf_diatomic *h, const double *P, int64_t ldp, double *K, int64_t ldk) {
  return guarded([&] {
    checked(h);
    DeviceGuard g(h->ctx->device);
    ensure_ready(h);
    host_roundtrip(h->ctx->cur, h->host.Nbf(), h->dev.hostP, h->dev.hostOut, P, ldp, K, ldk,
                   [&](const double *dp, int64_t lp, double *dout, int64_t lo) { exchange_launch(h, dp, lp, dout, lo); });
  });
}

}  // extern "C"
