"""The work a user of this framework has it do, as measurable cases.

Every case is one Fock build on a density that is resident on the GPU, the
step an SCF iteration repeats: the Coulomb matrix J(P) with the exchange
K(P/2) (Hartree-Fock), with the exchange-correlation matrix (Kohn-Sham), or J
and K of many atoms at once (batched solves).  The basis with its two-electron
tables, the DFT grid and the output matrices are what an SCF program keeps
from iteration to iteration; the density is new for every seed.

    listed()   the cases by name, smallest to largest per family
    draw(rng)  one more case of the same ranges
    prepare / run / work / tolerance / exact   as their docstrings say
"""
import math

import numpy as np
import torch

import helfem_amd as H
from helfem_amd.dftgrid import DFTGrid

THR = 1e-12  # density threshold of the DFT grids (the default of eval_Fxc)
XC = {"lda": (1, 7), "pbe": (101, 130)}
DEV = "cuda"


def listed():
    return [
        # Ne with s functions only: the smallest build there is, all launches and latency
        _atom("ne-hf", 10, 0, 0, 10, 15),
        # Ar, 10-node elements (4x4 to 10x10 tiles of a 16x16 kernel), few shells: an ordinary light atom
        _atom("ar-hf-order10", 18, 2, 2, 7, 10),
        # Kr with mmax < lmax in the reduced precision of early SCF iterations
        _atom("kr-hf-fp32", 36, 4, 3, 17, 15, precision="fp32"),
        # Xe, lmax = mmax = 6, 25 elements (Nbf 17101): the largest atom of the configurations
        _atom("xe-hf", 54, 6, 6, 25, 15),
        # H2 at its equilibrium distance, the small diatomic of the reference's own tests
        _dia("h2-hf", 1, 1, 1.4, [4, 4], 3, 15),
        # CO with a ragged angular basis (fewer l for higher |m|), an odd element count
        _dia("co-hf-ragged", 6, 8, 2.132, [13, 11, 7], 5, 15),
        # N2, lmax 16 for m = 0..3, 8 elements (Nbf 11894): the headline benchmark
        _dia("n2-hf", 7, 7, 2.074, [16, 16, 16, 16], 8, 15),
        # N2 in the reduced precision of early SCF iterations, served-request size
        _dia("n2-hf-fp32", 7, 7, 2.074, [12, 12, 12], 6, 15, precision="fp32"),
        # Xe Kohn-Sham LDA on the 36 x 36 angular rule: the largest DFT build
        _atom("xe-lda", 54, 6, 6, 25, 15, xc="lda"),
        # O, spin-polarised PBE (open-shell GGA)
        _atom("o-pbe-pol", 8, 3, 3, 12, 15, xc="pbe", pol=True),
        # N2 LDA on the pure-m diatomic grid (half of the served requests are LDA)
        _dia("n2-lda", 7, 7, 2.074, [16, 16, 16], 7, 15, xc="lda"),
        # two dozen atoms of the 512-atom distribution in one batched build
        {"name": "atoms-batch", "kind": "batch", "n": 24, "spec": 1004},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    family = rng.choice(["atom", "atom", "dia", "dia", "atom-xc", "dia-xc", "batch"])
    if family == "batch":
        return _plain({"kind": "batch", "n": log_int(2, 24), "spec": rng.randrange(1, 1 << 30)})
    precision = rng.choice(["fp64", "fp64", "fp32"])
    nnodes = rng.choice([8, 10, 11, 13, 15, 15])
    if family.startswith("atom"):
        lmax = rng.randint(0, 6)
        pol = family == "atom-xc" and lmax <= 4 and rng.random() < 0.5
        c = _atom(None, rng.randint(1, 86), lmax, rng.randint(min(1, lmax), lmax), log_int(4, 25), nnodes)
        if family == "atom":
            c["precision"] = precision
        else:
            c.update(xc=rng.choice(["lda", "pbe"]) if lmax <= 4 else "lda", pol=pol)
        return _plain(c)
    mmax = rng.randint(0, 3)
    lmmax = [log_int(4, 16)]
    for _ in range(mmax):
        lmmax.append(max(len(lmmax), lmmax[-1] - rng.choice([0, 0, 1, 2])))
    c = _dia(None, rng.randint(1, 18), rng.randint(1, 18), round(rng.uniform(1.0, 6.0), 3), lmmax, log_int(3, 8), nnodes)
    if family == "dia":
        c["precision"] = precision
    else:
        c.update(xc=rng.choice(["lda", "pbe"]), pol=rng.random() < 0.5)
    return _plain(c)


def _atom(name, Z, lmax, mmax, nelem, nnodes, precision="fp64", xc="", pol=False):
    return _plain({"name": name, "kind": "atom", "Z": Z, "lmax": lmax, "mmax": mmax, "nelem": nelem, "nnodes": nnodes,
                   "precision": precision, "xc": xc, "pol": pol})


def _dia(name, Z1, Z2, R, lmmax, nelem, nnodes, precision="fp64", xc="", pol=False):
    return _plain({"name": name, "kind": "dia", "Z1": Z1, "Z2": Z2, "R": R,
                   "lmmax": ",".join(str(v) for v in lmmax), "nelem": nelem, "nnodes": nnodes,
                   "precision": precision, "xc": xc, "pol": pol})


def _plain(c):
    return {k: v for k, v in c.items() if not (k == "name" and v is None)}


# --- inputs ------------------------------------------------------------------


def _batch_specs(case):
    """(Z, elements, order, lmax) of each atom, drawn like the 512-atom configuration."""
    rng = np.random.default_rng(case["spec"])
    out = []
    for _ in range(case["n"]):
        Z, nel = int(rng.integers(1, 87)), int(rng.integers(4, 25))
        out.append((Z, nel, int(rng.choice((10, 15))), int(rng.integers(0, 5))))
    return out


def _shells(case):
    if case["kind"] == "atom":
        return H.angular_basis(case["lmax"], case["mmax"])
    return H.diatomic_shells([int(v) for v in case["lmmax"].split(",")])


def _madelung(norb_pairs, lmax):
    """Occupied subshells per l for 2 norb_pairs electrons (n + l, then n), l <= lmax."""
    shells = sorted(((n, l) for n in range(1, 61) for l in range(0, min(n, lmax + 1))), key=lambda s: (s[0] + s[1], s[0]))
    per_l, left = {}, norb_pairs
    for _, l in shells:
        if left <= 0:
            break
        per_l[l] = per_l.get(l, 0) + 1
        left -= 2 * l + 1
    return per_l


def _occupied(case, spin=0):
    """{m: doubly (or per spin singly) occupied orbitals} of the neutral system; the
    beta spin (1) of a polarised case holds one orbital less in m = 0."""
    if case["kind"] == "atom":
        per_l = _madelung((case["Z"] + 1) // 2, case["lmax"])
        occ = {m: sum(n for l, n in per_l.items() if l >= abs(m)) for m in range(-case["mmax"], case["mmax"] + 1)}
    else:
        norb = (case["Z1"] + case["Z2"] + 1) // 2
        mmax = len(case["lmmax"].split(",")) - 1
        npi = norb // 7 if mmax >= 1 else 0
        occ = {0: norb - 2 * npi, 1: npi, -1: npi}
    if spin:
        occ[0] = max(occ[0] - 1, 0)
    return {m: n for m, n in occ.items() if n > 0}


def _lobatto(n):
    """Gauss-Lobatto nodes on [-1, 1]."""
    x = np.concatenate([[-1.0], np.sort(np.polynomial.legendre.Legendre.basis(n - 1).deriv().roots().real), [1.0]])
    return 0.5 * (x - x[::-1])


def _nodes(basis, nnodes, atomic):
    """Grid coordinate of every radial function's node (Lagrange functions: their own node)."""
    x, b = _lobatto(nnodes), np.asarray(basis.bval)
    g = np.concatenate([0.5 * (b[e] + b[e + 1]) + 0.5 * (b[e + 1] - b[e]) * x[:-1] for e in range(len(b) - 1)])
    return g[1:] if atomic else g


def _density(basis, case, seed, spin=0, nnodes=None):
    """Density sum_k f C_k C_k' (f = 2, or 1 per spin when polarised) of S-orthonormal
    smooth orbitals per m: products r^(l+1) exp(-zeta r) (atom; exp(-zeta R/2 (cosh mu - 1))
    in mu for a diatomic) with random shell weights, decaying as SCF orbitals do."""
    atomic = case["kind"] == "atom"
    gen = torch.Generator().manual_seed(int(seed) * 2 + spin + 1)
    g = torch.as_tensor(_nodes(basis, nnodes or case["nnodes"], atomic))
    Zc = float(case["Z"] if atomic else max(case["Z1"], case["Z2"]))
    S = basis.one_electron_dev(0)
    nrad = basis.Nrad
    if atomic:
        offs, skip = [a * nrad for a in range(basis.Nang)], [0] * basis.Nang
    else:
        skip = [0 if m == 0 else 1 for m in basis.mval.tolist()]
        offs = np.concatenate([[0], np.cumsum([nrad - s for s in skip])[:-1]]).tolist()
    P = torch.zeros(basis.Nbf, basis.Nbf, dtype=torch.float64, device=DEV)
    f = 1.0 if case["pol"] else 2.0
    for m, nocc in sorted(_occupied(case, spin).items()):
        sh = [a for a in range(basis.Nang) if basis.mval[a] == m]
        idx = torch.cat([torch.arange(offs[a], offs[a] + nrad - skip[a]) for a in sh])
        cols = []
        for k in range(nocc):
            zeta = Zc ** (1.0 - k / nocc) * (0.7 + 0.6 * torch.rand(len(sh), generator=gen, dtype=torch.float64)) + 0.3
            w = torch.randn(len(sh), generator=gen, dtype=torch.float64)
            col = []
            for q, a in enumerate(sh):
                l = int(basis.lval[a])
                if atomic:
                    t = zeta[q] * g
                    v = t ** (l + 1) * torch.exp(-t) / math.gamma(l + 2)
                else:
                    t = zeta[q] * 0.5 * basis.Rbond * (torch.cosh(g) - 1.0)
                    v = torch.sinh(g) ** abs(m) * torch.exp(-t) / (1.0 + l) ** 2
                col.append(w[q] * v[skip[a]:])
            cols.append(torch.cat(col))
        X = torch.stack(cols, 1).to(DEV)
        idx = idx.to(DEV)
        G = X.T @ S[idx][:, idx] @ X
        d = torch.rsqrt(torch.diagonal(G))
        e, v = torch.linalg.eigh(d[:, None] * G * d[None, :])
        C = (X * d) @ ((v / torch.sqrt(torch.clamp(e, min=1e-13))) @ v.T)
        Pm = f * (C @ C.T)
        P[idx[:, None], idx[None, :]] = 0.5 * (Pm + Pm.T)
    return P


def _basis(case, ctx):
    if case["kind"] == "atom":
        b = H.AtomicBasis(case["Z"], case["lmax"], case["mmax"], case["nelem"], nnodes=case["nnodes"], ctx=ctx)
    else:
        b = H.DiatomicBasis(case["Z1"], case["Z2"], case["R"], [int(v) for v in case["lmmax"].split(",")], case["nelem"],
                            nnodes=case["nnodes"], ctx=ctx)
    b.compute_tei(device=True)
    return b


def prepare(case, seed):
    """The basis with its tables, the grid, the density of this seed and the output matrices."""
    ctx = H.Context(0)
    if case["kind"] == "batch":
        bases, Ps = [], []
        for i, (Z, nel, nnodes, lmax) in enumerate(_batch_specs(case)):
            c = _atom(None, Z, lmax, lmax, nel, nnodes)
            b = _basis(c, ctx)
            bases.append(b)
            Ps.append(_density(b, c, seed * 1009 + i))
        st = {"ctx": ctx, "bases": bases, "batch": H.AtomicBatch(bases, ctx), "P": Ps, "Pa": [0.5 * P for P in Ps]}
        st["J"] = [torch.empty_like(P) for P in Ps]
        st["K"] = [torch.empty_like(P) for P in Ps]
        return st
    b = _basis(case, ctx)
    st = {"ctx": ctx, "basis": b, "case": case}
    if case["pol"]:
        st["Pa"], st["Pb"] = _density(b, case, seed, 0), _density(b, case, seed, 1)
        st["P"] = st["Pa"] + st["Pb"]
    else:
        st["P"] = _density(b, case, seed)
        if not case["xc"]:
            st["Pa"] = 0.5 * st["P"]
    st["J"] = torch.empty_like(st["P"])
    st["K"] = torch.empty_like(st["P"])
    if case["xc"]:
        st["grid"] = DFTGrid(b)  # the driver's default rule, 4 lmax + 12 (x 4 mmax + 12); pure-m for a diatomic
    return st


def run(st):
    """One Fock build: J, and K or the exchange-correlation matrix with its energy and electron count."""
    if "batch" in st:
        st["batch"].coulomb(st["P"], st["J"])
        st["batch"].exchange(st["Pa"], st["K"])
        return {"J": st["J"], "K": st["K"]}
    b, c = st["basis"], st["case"]
    J = b.coulomb(st["P"], out=st["J"])
    if not c["xc"]:
        return {"J": J, "K": b.exchange(st["Pa"], out=st["K"], precision=c["precision"])}
    x, cf = XC[c["xc"]]
    if c["pol"]:
        Ha, Hb, exc, nel, _ = st["grid"].eval_Fxc_pol(x, cf, st["Pa"], st["Pb"], thr=THR)
        return {"J": J, "Ha": Ha, "Hb": Hb, "exc": exc, "nel": nel}
    V, exc, nel, _ = st["grid"].eval_Fxc(x, cf, st["P"], thr=THR, out=st["K"])
    return {"J": J, "V": V, "exc": exc, "nel": nel}


# --- work and tolerance ------------------------------------------------------


def _sizes(case):
    """(radial functions, functions per element) of the finite-element grid."""
    n, nel = case["nnodes"], case["nelem"]
    atomic = case["kind"] == "atom"
    ni = [n - (1 if atomic and e == 0 else 0) - (1 if e == nel - 1 else 0) for e in range(nel)]
    return nel * (n - 1) - (1 if atomic else 0), ni


def work(case):
    """Bytes: every input and output matrix once, 8 bytes an entry (J takes only the element
    bands of its input).  Flops, least known for the contractions: J, 4 per band entry and
    coupled multipole; K, per coupled (output block, multipole) 4 n^3 a channel for each pair
    e > f of elements (a symmetric density gives the mirror) and 2 n^4 / 4 a channel inside an
    element (a dense operator that keeps the integrals' two transposition symmetries); Vxc,
    the radial and angular sums of the distinct shell pairs both ways."""
    if case["kind"] == "batch":
        tot = {"bytes": 0.0, "flops": 0.0}
        for Z, nel, nnodes, lmax in _batch_specs(case):
            w = work(_atom(None, Z, lmax, lmax, nel, nnodes))
            tot = {k: tot[k] + w[k] for k in tot}
        return tot
    lv, mv = (v.tolist() for v in _shells(case))
    nrad, ni = _sizes(case)
    ch = 1 if case["kind"] == "atom" else 4  # density channels of the two-electron kernel
    ext = 0 if ch == 1 else 2
    nbf = sum(nrad - (1 if ch == 4 and m else 0) for m in mv)
    lmax, occ = max(lv), set(_occupied(case))
    band = sum(n * n for n in ni)
    pairs = [(j, k) for j in range(len(lv)) for k in range(len(lv)) if mv[j] == mv[k]]
    nJ = sum(lv[j] + lv[k] + ext + 1 - abs(lv[j] - lv[k]) for j, k in pairs)
    flops = 4.0 * band * nJ * (1 if ch == 1 else 2)
    nbytes = 8.0 * (band * len(pairs) + nbf * nbf)
    if case["xc"]:
        ns = 2 if case["pol"] else 1
        nq, lang = 5 * case["nnodes"], 4 * lmax + 12
        mang = 4 * max(mv) + 12 if ch == 1 else 1
        dist = [1 for a in range(len(lv)) for b in range(a, len(lv)) if ch == 1 or mv[a] == mv[b]]
        nd = 2 * max(mv) + 1 if ch == 1 else 1
        gga = 2 if case["xc"] == "pbe" else 1
        per_point = 2.0 * len(dist) * 2 * lang + 4.0 * lang * (mang // 2 + 1) * nd
        flops += ns * gga * nq * (len(dist) * 4.0 * band + len(ni) * per_point)
        nbytes += ns * 8.0 * (nbf * nbf + band * len(pairs))
        return {"bytes": nbytes, "flops": flops}
    runs = runs_in = 0
    for j, k in pairs:
        c = 0
        for M in sorted({abs(mv[j] - m) for m in occ}):
            c += max(0, min(lv[j], lv[k]) + lmax + ext + 1 - M)
        if ch == 1:  # one radial contraction per L, whatever the M
            c = min(c, min(lv[j], lv[k]) + lmax + 1)
        runs += c
        runs_in += c if j <= k else 0
    off = sum(2.0 * (a * b * b + a * a * b) for e, a in enumerate(ni) for b in ni[:e])
    flops += runs * off * (1 if ch == 1 else 3) + runs_in * ch * sum(0.5 * n ** 4 for n in ni)
    return {"bytes": nbytes + 16.0 * nbf * nbf, "flops": flops}


def tolerance(case):
    """About four times the largest distance from exact() over the listed and two dozen drawn cases:
    5e-7 for the 32-bit exchange (density, weights and radial factors rounded to 24 bits), 1.2e-12
    for PBE (the thin outer density) and 1.6e-13 for the 64-bit J and K (orders of summation)."""
    if case.get("precision") == "fp32":
        return {"rel": 2e-6}
    return {"rel": 5e-12 if case.get("xc") == "pbe" else 6e-13}


# --- the same results in plain torch ------------------------------------------


def exact(case, seed):
    """What run() returns, by dense torch contractions in 64 bits.  The radial tables (element
    matrices and Cholesky factors, which a caller may also supply with set_cache) are taken from
    the basis; Gaunt coefficients, couplings, grids and functionals are formed here."""
    if case["kind"] == "batch":
        ctx = H.Context(0)
        Js, Ks = [], []
        for i, (Z, nel, nnodes, lmax) in enumerate(_batch_specs(case)):
            c = _atom(None, Z, lmax, lmax, nel, nnodes)
            b = _basis(c, ctx)
            P = _density(b, c, seed * 1009 + i)
            J, K = _exact_jk(b, c, P, 0.5 * P)
            Js.append(J)
            Ks.append(K)
        return {"J": Js, "K": Ks}
    ctx = H.Context(0)
    b = _basis(case, ctx)
    if not case["xc"]:
        P = _density(b, case, seed)
        J, K = _exact_jk(b, case, P, 0.5 * P)
        return {"J": J, "K": K}
    if case["pol"]:
        Ps = [_density(b, case, seed, 0), _density(b, case, seed, 1)]
    else:
        Ps = [_density(b, case, seed)]
    J, _ = _exact_jk(b, case, sum(Ps), None)
    Hs, exc, nel = _exact_xc(b, case, Ps)
    if case["pol"]:
        return {"J": J, "Ha": Hs[0], "Hb": Hs[1], "exc": exc, "nel": nel}
    return {"J": J, "V": Hs[0], "exc": exc, "nel": nel}


def _theta(lmax, x):
    """Normalised associated Legendre functions Y_l^m(arccos x, 0), m >= 0, by upward recurrence."""
    s = np.sqrt(1.0 - x * x)
    T = {}
    for m in range(lmax + 1):
        T[m, m] = np.full_like(x, math.sqrt(1.0 / (4.0 * math.pi))) if m == 0 else -math.sqrt((2 * m + 1) / (2.0 * m)) * s * T[m - 1, m - 1]
        for l in range(m + 1, lmax + 1):
            a = math.sqrt((4.0 * l * l - 1.0) / (l * l - m * m))
            b = math.sqrt(((l - 1.0) ** 2 - m * m) / (4.0 * (l - 1.0) ** 2 - 1.0)) if l > m + 1 else 0.0
            T[l, m] = a * (x * T[l - 1, m] - (b * T[l - 2, m] if l > m + 1 else 0.0))
    return lambda l, m: T[l, abs(m)] * (-1.0 if m < 0 and m % 2 else 1.0)


def _gaunts(lv, mv, Lmax, weight):
    """{(L, M): G[j, i]} with G = integral of Y_j* Y_LM Y_i weight(cos theta), M = mj - mi."""
    x, w = np.polynomial.legendre.leggauss(2 * (max(lv) + Lmax) + 6)
    th = _theta(max(max(lv), Lmax), x)
    ang = np.stack([th(l, m) for l, m in zip(lv, mv)])
    out = {}
    for M in sorted({a - b for a in mv for b in mv}):
        sel = np.equal.outer(np.array(mv), np.array(mv) + M)
        for L in range(abs(M), Lmax + 1):
            G = 2.0 * math.pi * (ang * (w * weight(x) * th(L, M))) @ ang.T
            G = np.where(sel & (np.abs(G) > 1e-13), G, 0.0)
            if np.any(G):
                out[L, M] = torch.as_tensor(G, device=DEV)
    return out


def _couple(Gl, Gr, P4):
    """sum_il Gl[j, i] P[i, :, l, :] Gr[k, l], over the rows and columns that take part."""
    j, i = torch.nonzero(Gl.abs().sum(1))[:, 0], torch.nonzero(Gl.abs().sum(0))[:, 0]
    k, l = torch.nonzero(Gr.abs().sum(1))[:, 0], torch.nonzero(Gr.abs().sum(0))[:, 0]
    n = P4.shape[1]
    X = P4[i][:, :, l]
    X = (Gl[j][:, i] @ X.reshape(len(i), -1)).reshape(len(j) * n, len(l), n)
    X = torch.einsum("kl,xlb->xkb", Gr[k][:, l], X)
    return j, k, X.reshape(len(j), n, len(k), n)


def _tiles(b, case):
    """First radial index and size of every element."""
    _, ni = _sizes(case)
    n = case["nnodes"]
    return [max(e * (n - 1) - (1 if case["kind"] == "atom" else 0), 0) for e in range(len(ni))], ni


def _cuda(a):
    return torch.as_tensor(np.ascontiguousarray(a), device=DEV)


def _exact_jk(b, case, P, Pk):
    """(J(P), -K(Pk)); Pk None: J alone."""
    atomic = case["kind"] == "atom"
    lv, mv = b.lval.tolist(), b.mval.tolist()
    na, n = b.Nang, b.Nrad
    first, ni = _tiles(b, case)
    nel = len(ni)
    full = torch.arange(na * n, device=DEV) if atomic else torch.as_tensor(b.pure_idx, device=DEV)

    def expand(M):
        X = torch.zeros(na * n, na * n, dtype=torch.float64, device=DEV)
        X[full[:, None], full[None, :]] = M
        return X.reshape(na, n, na, n)

    def shrink(X):
        return X.reshape(na * n, na * n)[full][:, full].contiguous()

    Lmax = 2 * max(lv) + (0 if atomic else 2)
    if atomic:
        chans = [_gaunts(lv, mv, Lmax, lambda x: np.ones_like(x))]
    else:
        chans = [_gaunts(lv, mv, Lmax, lambda x: x * x), _gaunts(lv, mv, Lmax, lambda x: np.ones_like(x))]
    lm = {} if atomic else {tuple(v): q for q, v in enumerate(b.maps()[0].tolist())}
    tabs = {}

    def tables(L, M):
        """Per element: low[c], high[c] (the factors of r<, r> or P, Q per channel) and the
        in-element tensor W[c][c2][a, c', b, d]."""
        key = L if atomic else lm[L, abs(M)]
        if key not in tabs:
            tabs.clear()
            low, high, W = [], [], []
            for e in range(nel):
                m = ni[e]
                if atomic:
                    low.append([_cuda(b.get_cache(0, L, e))])
                    high.append([_cuda(b.get_cache(1, L, e)) if e else torch.zeros_like(low[-1][0])])
                    B = _cuda(b.get_cache(2, L, e).reshape(m, m, -1, order="F"))
                    W.append([[torch.einsum("acp,bdp->acbd", B, B)]])
                else:
                    low.append([_cuda(b.get_cache(0, key, e)), _cuda(b.get_cache(1, key, e))])
                    high.append([_cuda(b.get_cache(2, key, e)), _cuda(b.get_cache(3, key, e))])
                    B = _cuda(b.get_cache(4, key, e))
                    sg = _cuda(b.get_cache(5, key, e)[:, 0])
                    C = [B[x * m * m:(x + 1) * m * m].reshape(m, m, -1).transpose(0, 1) for x in (0, 1)]
                    W.append([[torch.einsum("acp,bdp,p->acbd", C[x], C[y], sg) for y in (0, 1)] for x in (0, 1)])
            tabs[key] = (low, high, W)
        return tabs[key]

    def factor(L, M):
        if atomic:
            return 4.0 * math.pi / (2 * L + 1)
        f = 1.0
        for p in range(L - abs(M) + 1, L + abs(M) + 1):
            f *= p
        return (-1.0 if M % 2 else 1.0) * 4.0 * math.pi * b.Rhalf ** 5 / f

    nch = len(chans)
    keys = sorted({k for g in chans for k in g}, key=lambda k: (k[0], abs(k[1]), k[1]))
    zero = torch.zeros(na, na, dtype=torch.float64, device=DEV)
    sgn = [1.0, -1.0]  # the second channel of the pair enters with a minus sign

    P4 = expand(P)
    J = torch.zeros_like(P4)
    for L, M in keys:
        low, high, W = tables(L, M)
        G = [g.get((L, M), zero) for g in chans]
        sub = [[torch.einsum("kl,kalb->ab", g, P4[:, f:f + m][:, :, :, f:f + m]) for g in G] for f, m in zip(first, ni)]
        if not any(bool(s.any()) for ss in sub for s in ss):
            continue
        tl = [sum(sgn[x] * torch.sum(low[e][x] * sub[e][x].T) for x in range(nch)) for e in range(nel)]
        th = [sum(sgn[x] * torch.sum(high[e][x] * sub[e][x].T) for x in range(nch)) for e in range(nel)]
        for e in range(nel):
            f, m = first[e], ni[e]
            for x in range(nch):
                jx = sum(torch.einsum("acbd,bd->ac", W[e][x][y], sub[e][y]) for y in range(nch))
                if e + 1 < nel:
                    jx = jx + sgn[x] * sum(th[e + 1:]) * low[e][x]
                if e:
                    jx = jx + sgn[x] * sum(tl[:e]) * high[e][x]
                # J[i, j] couples with M = mj - mi
                J[:, f:f + m, :, f:f + m] += torch.einsum("ji,ab->iajb", factor(L, M) * G[x], jx)
    J = shrink(J)
    if Pk is None:
        return J, None
    del P4
    P4 = expand(Pk)
    K = torch.zeros_like(P4)
    # the multipoles of one set of tables together: per L (atom) or (L, |M|)
    groups = {}
    for L, M in keys:
        groups.setdefault(L if atomic else (L, abs(M)), []).append((L, M))
    for ms in groups.values():
        low, high, W = tables(*ms[0])
        R = [[torch.zeros_like(P4) for _ in range(nch)] for _ in range(nch)]
        for L, M in ms:
            for x in range(nch):
                for y in range(nch):
                    gx, gy = chans[x].get((L, M)), chans[y].get((L, M))
                    if gx is None or gy is None:
                        continue
                    j, k, X = _couple(gx, gy, P4)
                    R[x][y][j[:, None], :, k[None, :], :] += factor(L, M) * X.permute(0, 2, 1, 3)
        for e in range(nel):
            f, m = first[e], ni[e]
            rows = [[R[x][y][:, f:f + m].reshape(na * m * na, n) for y in range(nch)] for x in range(nch)]
            for x in range(nch):
                for side, own, other, fs in ((0, high, low, range(e)), (1, low, high, range(e + 1, nel))):
                    acc = torch.zeros_like(rows[0][0])
                    for y in range(nch):
                        E = torch.zeros(n, n, dtype=torch.float64, device=DEV)
                        for q in fs:
                            E[first[q]:first[q] + ni[q], first[q]:first[q] + ni[q]] += sgn[y] * other[q][y]
                        acc += rows[x][y] @ E.T
                    K[:, f:f + m] -= sgn[x] * torch.einsum("ac,jckb->jakb", own[e][x], acc.reshape(na, m, na, n))
                for y in range(nch):
                    T = W[e][x][y].permute(0, 2, 1, 3).reshape(m * m, m * m)  # (a, b), (c, d)
                    Y = R[x][y][:, f:f + m][:, :, :, f:f + m].permute(0, 2, 1, 3).reshape(na * na, m * m) @ T.T
                    K[:, f:f + m, :, f:f + m] -= Y.reshape(na, na, m, m).permute(0, 2, 1, 3)
    return J, shrink(K)


def _lagrange(nodes, x):
    """Lagrange polynomials on `nodes` and their derivatives at x: (points, functions) each."""
    n = len(nodes)
    L, D = np.ones((len(x), n)), np.zeros((len(x), n))
    for j in range(n):
        for k in range(n):
            if k != j:
                L[:, j] *= (x - nodes[k]) / (nodes[j] - nodes[k])
        for m in range(n):
            if m == j:
                continue
            t = np.full(len(x), 1.0 / (nodes[j] - nodes[m]))
            for k in range(n):
                if k not in (j, m):
                    t *= (x - nodes[k]) / (nodes[j] - nodes[k])
            D[:, j] += t
    return L, D


def _chebyshev(n):
    """The grid's Chebyshev rule on [-1, 1] (second kind, mapped so that its weight is one)."""
    t = np.arange(n, 0, -1) * math.pi / (n + 1)
    s, c = np.sin(t), np.cos(t)
    x = 1.0 - 2.0 * np.arange(n, 0, -1) / (n + 1) + (2.0 / math.pi) * (1.0 + 2.0 / 3.0 * s * s) * c * s
    return x, 16.0 / 3.0 / (n + 1) * s ** 4


def _exact_xc(b, case, Ps):
    """Per spin (or total) the exchange-correlation matrix, as the symmetrised derivative of the
    grid's energy with respect to the density matrix; Exc and the electron count."""
    atomic = case["kind"] == "atom"
    lv, mv = b.lval.tolist(), b.mval.tolist()
    na, n = b.Nang, b.Nrad
    first, ni = _tiles(b, case)
    gga = case["xc"] == "pbe"
    lang = 4 * max(lv) + 12
    mang = 4 * max(mv) + 12 if atomic else 1
    xt, wt = _chebyshev(lang)
    xq, wq = _chebyshev(5 * case["nnodes"])
    sth = np.sqrt((1.0 - xt) * (1.0 + xt))
    th = _theta(max(lv) + 1, xt)
    ang = np.stack([th(l, m) for l, m in zip(lv, mv)])
    dang = np.stack([m * xt / sth * th(l, m) + (math.sqrt((l - m) * (l + m + 1.0)) * th(l, m + 1) if m < l else 0.0)
                     for l, m in zip(lv, mv)])
    classes = {}
    for i in range(na):
        for j in range(na):
            if atomic or mv[i] == mv[j]:
                classes.setdefault(mv[i] - mv[j], []).append((i, j))
    phi = 2.0 * math.pi / mang * np.arange(mang)
    lob = _lobatto(case["nnodes"])
    L, D = _lagrange(lob, xq)
    ps = [P.clone().requires_grad_(True) for P in Ps]
    full = torch.arange(na * n, device=DEV) if atomic else torch.as_tensor(b.pure_idx, device=DEV)
    pos = torch.full((na * n,), -1, dtype=torch.long, device=DEV)
    pos[full] = torch.arange(b.Nbf, device=DEV)
    grads = [torch.zeros_like(P) for P in Ps]
    exc = nel = 0.0
    pt = {d: (_cuda([p[0] for p in v]), _cuda([p[1] for p in v])) for d, v in classes.items()}
    tt = {d: _cuda(np.stack([ang[i] * ang[j] for i, j in v])) for d, v in classes.items()}
    td = {d: _cuda(np.stack([dang[i] * ang[j] + ang[i] * dang[j] for i, j in v])) for d, v in classes.items()}
    for e in range(len(ni)):
        lo, hi = float(b.bval[e]), float(b.bval[e + 1])
        r = 0.5 * (lo + hi) + 0.5 * (hi - lo) * xq
        s0 = 1 if atomic and e == 0 else 0
        B, dB = L[:, s0:s0 + ni[e]], D[:, s0:s0 + ni[e]] * (2.0 / (hi - lo))
        if atomic:
            B, dB = B / r[:, None], dB / r[:, None] - B / (r * r)[:, None]
            w = np.outer(0.5 * (hi - lo) * wq * r * r, wt * 2.0 * math.pi / mang)
            c = [np.ones((len(r), lang)), np.outer(1.0 / r, np.ones(lang)), 1.0 / np.outer(r, sth)]
        else:
            sh = np.sinh(r)[:, None]
            q = sh * sh + sth[None, :] ** 2
            w = np.outer(0.5 * (hi - lo) * wq, 2.0 * math.pi * wt) * b.Rhalf ** 3 * sh * q
            c = [1.0 / (b.Rhalf * np.sqrt(q))] * 2 + [1.0 / (b.Rhalf * sh * sth[None, :])]
        B, dB, w, c = _cuda(B), _cuda(dB), _cuda(w)[:, :, None], [_cuda(v)[:, :, None] for v in c]
        f, m = first[e], ni[e]
        at = (torch.arange(na, device=DEV)[:, None] * n + torch.arange(f, f + m, device=DEV)[None, :]).reshape(-1)
        keep = (pos[at] >= 0)
        idx = pos[at].clamp(min=0)
        args = []
        for p in ps:
            t = (p[idx][:, idx] * (keep[:, None] & keep[None, :])).reshape(na, m, na, m)
            half = torch.einsum("ambn,qn->ambq", t, B)
            Dm = torch.einsum("ambq,qm->abq", half, B)
            Em = torch.einsum("ambq,qm->abq", half, dB) if gga else None
            rho, g = 0.0, [0.0, 0.0, 0.0]
            for d, (i, j) in pt.items():
                cs, sn = _cuda(np.cos(d * phi)), _cuda(np.sin(d * phi))
                cd = torch.einsum("xq,xt->qt", Dm[i, j], tt[d])[:, :, None]
                rho = rho + cd * cs
                if gga:
                    g[0] = g[0] + 2.0 * torch.einsum("xq,xt->qt", Em[i, j], tt[d])[:, :, None] * cs
                    g[1] = g[1] + torch.einsum("xq,xt->qt", Dm[i, j], td[d])[:, :, None] * cs
                    g[2] = g[2] - d * cd * sn
            args.append((rho, [c[x] * g[x] for x in range(3)] if gga else None))
        if len(args) == 1:
            rho, g = args[0]
            args = [(0.5 * rho, [0.5 * v for v in g] if gga else None)] * 2
        (ra, ga), (rb, gb) = args
        dot = lambda u, v: u[0] * v[0] + u[1] * v[1] + u[2] * v[2]  # noqa: E731
        sig = (dot(ga, ga), dot(ga, gb), dot(gb, gb)) if gga else None
        en = torch.sum(w * _energy(case["xc"], ra, rb, sig, case["pol"]))
        for G, dG in zip(grads, torch.autograd.grad(en, ps)):
            G += dG
        exc += float(en.detach())
        nel += float(torch.sum(w * (ra + rb)).detach())
    return [0.5 * (G + G.T) for G in grads], exc, nel


def _energy(name, ra, rb, sig, pol):
    """Exchange-correlation energy per volume, zero below the density threshold: Slater and
    VWN5, or PBE on PW92."""
    rho = ra + rb
    live = rho >= THR
    one = torch.ones_like(rho)
    a, b = torch.where(live, ra, one), torch.where(live, rb, one)
    n = a + b
    z = torch.clamp((a - b) / n, -1.0, 1.0)
    rs = (3.0 / (4.0 * math.pi) / n) ** (1.0 / 3.0)
    opz, omz = torch.clamp(1.0 + z, min=2.2e-16), torch.clamp(1.0 - z, min=2.2e-16)
    fz = (opz ** (4.0 / 3.0) + omz ** (4.0 / 3.0) - 2.0) / (2.0 ** (4.0 / 3.0) - 2.0)
    cx = -0.75 * (6.0 / math.pi) ** (1.0 / 3.0)
    z4 = z ** 4
    floor = THR if name == "pbe" and pol else 0.0

    def spin(v, F):
        ok = v > floor if floor == 0.0 else v >= floor
        u = torch.where(ok, v, one)
        return torch.where(ok, cx * u ** (4.0 / 3.0) * F(u), torch.zeros_like(v))

    if name == "lda":
        def vwn(A, p, q, x0):
            x = torch.sqrt(rs)
            Q, X, X0 = math.sqrt(4 * q - p * p), x * x + p * x + q, x0 * x0 + p * x0 + q
            at = torch.atan(Q / (2 * x + p))
            return A * (torch.log(x * x / X) + 2 * p / Q * at
                        - p * x0 / X0 * (torch.log((x - x0) ** 2 / X) + 2 * (p + 2 * x0) / Q * at))
        eP, eF = vwn(0.0310907, 3.72744, 12.9352, -0.10498), vwn(0.01554535, 7.06042, 18.0578, -0.325)
        eA = vwn(-1.0 / (6.0 * math.pi ** 2), 1.13107, 13.0045, -0.0047584)
        fpp = 4.0 / (9.0 * (2.0 ** (1.0 / 3.0) - 1.0))
        ec = eP + eA * fz * (1.0 - z4) / fpp + (eF - eP) * fz * z4
        e = n * ec + spin(a, lambda u: 1.0) + spin(b, lambda u: 1.0)
        return torch.where(live, e, torch.zeros_like(e))

    def pw(A, a1, b1, b2, b3, b4):
        s = torch.sqrt(rs)
        return -2.0 * A * (1.0 + a1 * rs) * torch.log(1.0 + 1.0 / (2.0 * A * (b1 * s + b2 * rs + b3 * rs * s + b4 * rs * rs)))

    g0 = pw(0.0310907, 0.21370, 7.5957, 3.5876, 1.6382, 0.49294)
    g1 = pw(0.01554535, 0.20548, 14.1189, 6.1977, 3.3662, 0.62517)
    g2 = pw(0.0168869, 0.11125, 10.357, 3.6231, 0.88026, 0.49671)
    ec = g0 + z4 * fz * (g1 - g0 + g2 / 1.709920934161365617563962776245) - fz * g2 / 1.709920934161365617563962776245
    beta, gamma, kappa = 0.06672455060314922, (1.0 - math.log(2.0)) / math.pi ** 2, 0.804
    mu = beta * math.pi ** 2 / 3.0
    saa, sab, sbb = (torch.where(live, s, one) for s in sig)

    def enh(s):
        # spin scaling: the unpolarised factor at density 2u and gradient 4s
        return lambda u: 1.0 + kappa - kappa / (1.0 + mu / kappa * 4.0 * s / (
            4.0 * (3.0 * math.pi ** 2) ** (2.0 / 3.0) * (2.0 * u) ** (8.0 / 3.0)))

    ex = spin(a, enh(saa)) + spin(b, enh(sbb))
    saa, sbb = torch.clamp(saa, min=1e-40), torch.clamp(sbb, min=1e-40)
    av = 0.5 * (saa + sbb)
    sab = torch.minimum(torch.maximum(sab, -av), av) if pol else sab
    ph = 0.5 * (opz ** (2.0 / 3.0) + omz ** (2.0 / 3.0))
    ks2 = 4.0 / math.pi * (3.0 * math.pi ** 2 * n) ** (1.0 / 3.0)
    t2 = (saa + 2.0 * sab + sbb) / (4.0 * ph * ph * ks2 * n * n)
    A = beta / gamma / torch.expm1(-ec / (gamma * ph ** 3))
    Hc = gamma * ph ** 3 * torch.log(1.0 + beta / gamma * t2 * (1.0 + A * t2) / (1.0 + A * t2 + (A * t2) ** 2))
    e = ex + n * (ec + Hc)
    return torch.where(live, e, torch.zeros_like(e))
