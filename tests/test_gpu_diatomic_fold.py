"""The in-element diatomic exchange with folded operators at every shape of its
tiles: element sizes from one function to a full 16 x 16 tile (row tiles, inner
extents and their splits over the waves all follow the size), units with one
and two rows, and the forms it stands in for.  FP32 takes it on elements of at
least 7 functions and at most 2.6 long in mu.

Bar: FP64 1e-12 of max|K| against the oracle (src/diatomic/basis.cpp:1818-2089),
as the other parity tests; FP32 1.25 times the Cholesky-form kernel's error on
the same inputs, or where an element holds so few functions that no sum
averages the roundings out, the four of one product (density, both weights and
operator, 2^-24 each): 2.4e-7."""
import numpy as np
import pytest

import helfem_amd as H
import oracle as O
from helfem_amd._lib import check, lib
from helfem_amd.synthetic import random_symmetric

pytestmark = pytest.mark.gpu
TOL = 1e-12


def relerr(a, b):
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300))


def launched(ctx, run):
    """The result and the in-element kernels that made it."""
    check(lib().hf_ctx_set_timing(ctx.handle, 1))
    K = run().cpu().numpy()
    v, ran = np.zeros(3), {}
    for name in ("k_dia_kin_fold", "k_dia_kin_lds", "k_dia_kin_op", "k_dia_kin_gemm", "k_dia_k_in"):
        check(lib().hf_ctx_kernel_stats(ctx.handle, name.encode(), v.ctypes.data))
        ran[name] = int(v[0])
    check(lib().hf_ctx_set_timing(ctx.handle, 0))
    return K, ran


@pytest.mark.parametrize("nodes", [2, 3, 4, 6, 9, 12, 16])
def test_element_sizes(nodes, gpu_ctx, monkeypatch):
    import torch
    print(f"[gpu] folded in-element exchange, {nodes} nodes", flush=True)
    ob = O.DiatomicBasis(3, 1, 3.0, [3, 2], 2, nnodes=nodes)
    ob.compute_tei()
    b = {}
    for form in ("fold", "0"):
        if form == "0":
            monkeypatch.setenv("HFGPU_EXCHANGE_OP", "0")
        b[form] = H.DiatomicBasis(3, 1, 3.0, [3, 2], 2, nnodes=nodes, ctx=gpu_ctx)
        b[form].compute_tei()
        b[form].exchange(torch.zeros((ob.Nbf, ob.Nbf), dtype=torch.float64, device="cuda"))  # the form is fixed here
    S = random_symmetric(ob.Nbf, seed=2101)
    G = S + 0.3 * np.triu(random_symmetric(ob.Nbf, seed=2102))
    for P in (S, G):
        Kr = ob.exchange(P)
        Pd = torch.as_tensor(P, device="cuda")
        e64 = {f: relerr(x.exchange(Pd).cpu().numpy(), Kr) for f, x in b.items()}
        e32 = {f: relerr(x.exchange(Pd, precision="fp32").cpu().numpy(), Kr) for f, x in b.items()}
        print(e64, e32, flush=True)
        assert e64["fold"] <= TOL and e64["0"] <= TOL
        ran = {f: launched(gpu_ctx, lambda: x.exchange(Pd))[1] for f, x in b.items()}
        # 16 functions: a rank beyond the LDS of k_dia_kin_lds
        assert ran["fold"]["k_dia_kin_fold"] == 1 and ran["0"]["k_dia_kin_lds"] + ran["0"]["k_dia_k_in"] == 1
        assert e32["fold"] <= max(1.25 * e32["0"], 4 * 2.0 ** -24)


def test_one_element_and_density_holes(gpu_ctx):
    """A single element (no cross-element launch) and a density without some
    of its shell blocks (runs of tiles with gaps)."""
    import torch
    print("[gpu] folded in-element exchange, one element, sparse density", flush=True)
    for nel in (1, 2):
        ob = O.DiatomicBasis(2, 1, 1.5, [4, 3], nel, nnodes=6)
        ob.compute_tei()
        hb = H.DiatomicBasis(2, 1, 1.5, [4, 3], nel, nnodes=6, ctx=gpu_ctx)
        hb.compute_tei()
        P = random_symmetric(ob.Nbf, seed=2103)
        sh = np.asarray(hb.pure_idx) // hb.Nrad
        rng = np.random.default_rng(2104)
        keep = rng.random((hb.Nang, hb.Nang)) < 0.6
        keep = keep & keep.T
        P = P * keep[sh][:, sh]
        assert relerr(hb.exchange(torch.as_tensor(P, device="cuda")).cpu().numpy(), ob.exchange(P)) <= TOL


@pytest.mark.parametrize("lmm,top", [([2, 3, 4, 5, 6, 7, 8, 9], 7), (list(range(11)), 10)], ids=["m7", "m10"])
def test_fp32_high_m(lmm, top, gpu_ctx):
    """|m| where the in-element operators ((L+M)!/(L-M)!: 1e40 at M = 14, 1e58 at
    M = 20) and the coupling factors, their inverse, leave FP32's range: every
    block, and those that the largest M alone feeds (the density of m = -top in the
    output of m = top), at the FP32 exchange's bar of the other tests, 2e-6 of the
    largest entry."""
    import torch
    print(f"[gpu] FP32 diatomic exchange at |m| = {top}", flush=True)
    hb = H.DiatomicBasis(7, 7, 2.074, lmm, 3, nnodes=8, ctx=gpu_ctx)
    hb.compute_tei()
    m = np.asarray(hb.mval)[np.asarray(hb.pure_idx) // hb.Nrad]
    P = random_symmetric(hb.Nbf, seed=2105)
    low = np.where((m[:, None] == -top) & (m[None, :] == -top), P, 0.0)
    out = np.ix_(m == top, m == top)
    for X, sel in ((P, np.ix_(m == m, m == m)), (low, out)):
        Xd = torch.as_tensor(np.ascontiguousarray(X), device="cuda")
        K64 = hb.exchange(Xd).cpu().numpy()[sel]
        K32 = hb.exchange(Xd, precision="fp32").cpu().numpy()[sel]
        assert np.max(np.abs(K64)) > 0.0 and np.all(np.isfinite(K32))
        print(f"fp32 error {relerr(K32, K64):.2e}", flush=True)
        assert relerr(K32, K64) <= 2e-6


@pytest.mark.parametrize("nel", [3, 6])
def test_sums_no_further_off(nel, gpu_ctx, monkeypatch):
    """Long sums (15 functions, 465 products, channels that cancel): the error of
    the folded FP32 form against FP64, over several smooth densities, is at most the
    Cholesky form's.  Both round the same inputs; a single FP32 chain is 1.6 to 1.9
    times as far off, sums of 16 products 0.7 times."""
    import torch
    print(f"[gpu] folded FP32 sums, {nel} elements", flush=True)
    args, kw = (7, 7, 6.0, [3, 2, 2], nel), dict(nnodes=15, ctx=gpu_ctx)
    fold = H.DiatomicBasis(*args, **kw)
    fold.compute_tei()
    fold.exchange(torch.zeros((fold.Nbf, fold.Nbf), dtype=torch.float64, device="cuda"))  # the form is fixed here
    monkeypatch.setenv("HFGPU_EXCHANGE_OP", "0")
    chol = H.DiatomicBasis(*args, **kw)
    chol.compute_tei()
    S = np.asarray(fold.overlap())
    sh = np.asarray(fold.pure_idx) // fold.Nrad
    m, rad = np.asarray(fold.mval)[sh], np.asarray(fold.pure_idx) % fold.Nrad
    mu = np.linspace(0.0, fold.bval[-1], fold.Nrad)[rad]
    e = []
    for seed in range(4):
        rng = np.random.default_rng(2106 + seed)
        P = np.zeros((fold.Nbf, fold.Nbf))
        for k in (-1, 0, 0, 0, 1):
            c = np.zeros(fold.Nbf)
            for a in np.flatnonzero(np.asarray(fold.mval) == k):
                z = 0.3 + 6.0 * rng.random()
                c[sh == a] = (rng.standard_normal() * np.sinh(mu) ** abs(k) * np.exp(-3.0 * z * (np.cosh(mu) - 1.0)))[sh == a]
            P += np.outer(c, c) / (c @ S @ c)
        Pd = torch.as_tensor(P, device="cuda")
        ref = chol.exchange(Pd)
        e.append([float(torch.linalg.norm(b.exchange(Pd, precision="fp32") - ref)) for b in (fold, chol)])
    ratio = np.array(e)[:, 0] / np.array(e)[:, 1]
    print("folded / Cholesky form error", ratio, flush=True)
    assert np.exp(np.mean(np.log(ratio))) <= 1.0


def test_operators_of_one_precision_only(gpu_ctx, monkeypatch):
    """A budget that holds the FP32 operators and not the FP64 ones: FP64 takes the
    Cholesky form, FP32 the folded one, in turn on one handle and over two screening
    patterns; with no room at all both take the Cholesky form."""
    import torch
    print("[gpu] folded operators under a memory budget", flush=True)
    n, nel = 9, 3
    s, a = n * (n + 1) // 2, n * (n - 1) // 2
    per = sum((p + 15) // 16 * 16 * ((2 * p + n * n + 15) // 16 * 16) for p in (s, a))
    ob = O.DiatomicBasis(3, 1, 3.0, [3, 2], nel, nnodes=n)
    ob.compute_tei()
    hb, none = (H.DiatomicBasis(3, 1, 3.0, [3, 2], nel, nnodes=n, ctx=gpu_ctx) for _ in range(2))
    sizes = np.zeros(7, dtype=np.int64)
    check(lib().hf_diatomic_sizes(hb._h, sizes.ctypes.data))
    gib = 6.0 * per * nel * int(sizes[5]) / 2.0 ** 30  # bytes between four and eight per entry
    for b in (hb, none):
        b.compute_tei()
    S = random_symmetric(ob.Nbf, seed=2110)
    sh = np.asarray(hb.pure_idx) // hb.Nrad
    D = np.where((sh[:, None] == 0) | (sh[None, :] == 0), 0.0, S)
    for P in (S, D, S):
        Kr = ob.exchange(P)
        Pd = torch.as_tensor(P, device="cuda")
        for b, env, forms in ((hb, gib, ("k_dia_kin_lds", "k_dia_kin_fold")), (none, 0.0, ("k_dia_kin_lds",) * 2)):
            monkeypatch.setenv("HFGPU_EXCHANGE_FOLD_GIB", repr(env))
            for prec, form, tol in (("fp64", forms[0], TOL), ("fp32", forms[1], 2e-6), ("fp64", forms[0], TOL)):
                K, ran = launched(gpu_ctx, lambda: b.exchange(Pd, precision=prec))
                assert ran[form] == 1 and sum(ran.values()) == 1
                assert relerr(K, Kr) <= tol


@pytest.mark.parametrize("lmm,nel,nodes,R,form", [
    ([3, 2, 2], 3, 5, 6.0, "k_dia_kin_lds"),   # few functions: 1.7 times the Cholesky form's error when folded
    ([3, 2, 2], 3, 7, 6.0, "k_dia_kin_lds"),   # the last element has 6
    ([3, 2, 2], 3, 8, 6.0, "k_dia_kin_fold"),
    ([4], 1, 8, 1.0, "k_dia_kin_lds"),         # one element of mu 0 .. 5.1: 2.0 times
    ([4], 3, 15, 1.0, "k_dia_kin_lds"),        # longest element 2.75: 1.4 times
    ([6, 6], 3, 15, 2.0, "k_dia_kin_fold"),    # 2.31
])
def test_fp32_form_by_basis(lmm, nel, nodes, R, form, gpu_ctx):
    import torch
    print(f"[gpu] FP32 in-element form {lmm} {nel} {nodes} R {R}", flush=True)
    hb = H.DiatomicBasis(7, 7, R, lmm, nel, nnodes=nodes, ctx=gpu_ctx)
    hb.compute_tei()
    Pd = torch.as_tensor(random_symmetric(hb.Nbf, seed=2111), device="cuda")
    K64, r64 = launched(gpu_ctx, lambda: hb.exchange(Pd))
    K32, r32 = launched(gpu_ctx, lambda: hb.exchange(Pd, precision="fp32"))
    assert r64["k_dia_kin_fold"] == 1 and r32[form] == 1 and sum(r32.values()) == 1
    assert relerr(K32, K64) <= 2e-6
    K64b, _ = launched(gpu_ctx, lambda: hb.exchange(Pd))  # the lists serve both forms
    assert relerr(K64b, K64) <= TOL
