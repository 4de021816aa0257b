"""The two-step cross-element diatomic exchange at the edges of its lists:
columns with more rows than one workgroup holds, (L,|M|) groups whose slots do
not fit the LDS tiles together, elements of the smallest and the full tile
size, and densities the shared sums must not see (infinities).

Bars: FP64 1e-12 of max|K| against the oracle (src/diatomic/basis.cpp:
1818-2089), as the other parity tests.  FP32: the one-step kernel's own error
on the same inputs (both round the density, the weights and the factors to 24
bits, 6e-8 each, and differ in the order of their sums: 1.25 times it), which
scales with the cancellation in a random dense density, not with the kernel."""
import numpy as np
import pytest

import helfem_amd as H
import oracle as O
from helfem_amd._lib import check, lib
from helfem_amd.synthetic import random_symmetric

pytestmark = pytest.mark.gpu
TOL = 1e-12

CASES = {
    # ragged angular basis, odd element count, 16-node elements (full tiles)
    "l531-3el-order16": ([5, 3, 2], 3, 16),
    # one l per m: single-row waves, single-slot groups
    "l0-2el": ([0], 2, 15),
    "l1-m1-4el-order3": ([1, 1], 4, 3),
}


def relerr(a, b):
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300))


def launched(ctx, run):
    """The result and how often the two-step and the one-step kernel made it."""
    check(lib().hf_ctx_set_timing(ctx.handle, 1))
    K = run().cpu().numpy()
    v, ran = np.zeros(3), []
    for name in ("k_dia_k2_off", "k_dia_k_off"):
        check(lib().hf_ctx_kernel_stats(ctx.handle, name.encode(), v.ctypes.data))
        ran.append(int(v[0]))
    check(lib().hf_ctx_set_timing(ctx.handle, 0))
    return K, tuple(ran)


@pytest.mark.parametrize("name", list(CASES))
def test_lists_at_their_edges(name, gpu_ctx, monkeypatch):
    import torch
    print(f"[gpu] two-step diatomic exchange: {name}", flush=True)
    lmm, nel, nodes = CASES[name]
    ob = O.DiatomicBasis(7, 6, 2.1, lmm, nel, nnodes=nodes)
    ob.compute_tei()
    hb = H.DiatomicBasis(7, 6, 2.1, lmm, nel, nnodes=nodes, ctx=gpu_ctx)
    hb.compute_tei()
    one = H.DiatomicBasis(7, 6, 2.1, lmm, nel, nnodes=nodes, ctx=gpu_ctx)
    one.compute_tei()
    S = random_symmetric(ob.Nbf, seed=2001)
    G = S + 0.3 * np.triu(random_symmetric(ob.Nbf, seed=2002))
    # m-diagonal and with one shell empty: sparse lists
    D = S.copy()
    sh = np.asarray(hb.pure_idx) // hb.Nrad
    m = np.asarray(hb.mval)[sh]
    D[m[:, None] != m[None, :]] = 0.0
    D[sh == 0, :] = 0.0
    D[:, sh == 0] = 0.0
    for P in (S, G, D):
        Kr = ob.exchange(P)
        Pd = torch.as_tensor(P, device="cuda")
        K, ran = launched(gpu_ctx, lambda: hb.exchange(Pd))
        assert relerr(K, Kr) <= TOL
        K32, ran32 = launched(gpu_ctx, lambda: hb.exchange(Pd, precision="fp32"))
        if np.any(Kr):  # else no block is coupled
            assert ran == (1, 0) and ran32 == (1, 0)
        e32 = relerr(K32, Kr)
        monkeypatch.setenv("HFGPU_EXCHANGE_TWOSTEP", "0")
        K32, ran32 = launched(gpu_ctx, lambda: one.exchange(Pd, precision="fp32"))
        if np.any(Kr):
            assert ran32 == (0, 1)
        o32 = relerr(K32, Kr)
        monkeypatch.delenv("HFGPU_EXCHANGE_TWOSTEP")
        print(f"fp32 error {e32:.2e}, one-step {o32:.2e}", flush=True)
        assert e32 <= 1.25 * o32


def test_more_rows_and_slots_than_fit(gpu_ctx, monkeypatch):
    """53 rows per column of a general density (three workgroups) and 34 slots
    in the |M| = 1 groups: equal to the one-step kernel (HFGPU_EXCHANGE_TWOSTEP=0),
    which the oracle pins on the small bases (its own build takes minutes here)."""
    import torch
    print("[gpu] two-step diatomic exchange: 53 rows, 34 slots", flush=True)
    K = []
    for two in ("1", "0"):
        monkeypatch.setenv("HFGPU_EXCHANGE_TWOSTEP", two)
        hb = H.DiatomicBasis(7, 6, 2.1, [17, 17], 2, nnodes=4, ctx=gpu_ctx)
        hb.compute_tei()
        S = random_symmetric(hb.Nbf, seed=2005)
        G = S + 0.3 * np.triu(random_symmetric(hb.Nbf, seed=2006))
        K.append([])
        for P in (S, G):
            Pd = torch.as_tensor(P, device="cuda")
            X, ran = launched(gpu_ctx, lambda: hb.exchange(Pd))
            assert ran == ((1, 0) if two == "1" else (0, 1))
            K[-1].append(X)
    for a, b in zip(*K):
        assert relerr(a, b) <= TOL


def test_infinite_density_stays_in_its_blocks(gpu_ctx, monkeypatch):
    """An infinite entry reaches only the output blocks coupled to its own
    density block: the non-finite pattern is the one-step kernels'."""
    import torch
    print("[gpu] two-step diatomic exchange: infinite entry", flush=True)
    K = []
    for two in ("1", "0"):
        monkeypatch.setenv("HFGPU_EXCHANGE_TWOSTEP", two)
        hb = H.DiatomicBasis(7, 7, 2.074, [5, 4], 3, ctx=gpu_ctx)
        hb.compute_tei()
        P = random_symmetric(hb.Nbf, seed=2003)
        P[3, 5] = P[5, 3] = np.inf
        Pd = torch.as_tensor(P, device="cuda")
        hb.exchange(torch.as_tensor(random_symmetric(hb.Nbf, seed=2004), device="cuda"))
        X, ran = launched(gpu_ctx, lambda: hb.exchange(Pd))
        assert ran == (0, 1)  # not finite: one step either way
        K.append(X)
    assert np.array_equal(np.isfinite(K[0]), np.isfinite(K[1]))
    ok = np.isfinite(K[0])
    assert relerr(K[0][ok], K[1][ok]) <= TOL
