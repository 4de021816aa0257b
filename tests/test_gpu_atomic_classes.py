"""The cross-element atomic exchange by density classes (k_atomic_kc_off), forced
on bases of every shape (HFGPU_EXCHANGE_CLASSES=1; by itself it takes large
angular bases only) against the oracle and the one-block-at-a-time kernel (=0).

Bar: FP64 1e-12 of max|K| against the oracle (src/atomic/TwoDBasis.cpp:880-999);
FP32 1.25 times the other kernel's error on the same inputs or the roundings of
one product (density, two weights, factor: 2^-24 each)."""
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
    """The result and how often the class and the block kernel made it."""
    check(lib().hf_ctx_set_timing(ctx.handle, 1))
    K = run()
    v, ran = np.zeros(3), []
    for name in ("k_atomic_kc_off", "k_atomic_k_off"):
        check(lib().hf_ctx_kernel_stats(ctx.handle, name.encode(), v.ctypes.data))
        ran.append(int(v[0]))
    check(lib().hf_ctx_set_timing(ctx.handle, 0))
    return K, tuple(ran)


def _bases(monkeypatch, ctx, args, kw):
    """The basis with the kernel on and off; the choice is made at the first build."""
    import torch
    out = []
    for env in ("1", "0"):
        monkeypatch.setenv("HFGPU_EXCHANGE_CLASSES", env)
        b = H.AtomicBasis(*args, ctx=ctx, **kw)
        b.compute_tei()
        out.append(b)
    return out, lambda b, P, **k: b.exchange(torch.as_tensor(P, device="cuda"), **k).cpu().numpy()


@pytest.mark.parametrize("lmax,mmax,nel,nodes", [(0, 0, 2, 15), (2, 2, 3, 16), (3, 1, 2, 5), (4, 2, 2, 3)])
def test_against_oracle(lmax, mmax, nel, nodes, gpu_ctx, monkeypatch):
    print(f"[gpu] class exchange lmax={lmax} mmax={mmax}, {nel} elements, {nodes} nodes", flush=True)
    (on, off), K = _bases(monkeypatch, gpu_ctx, (10, lmax, mmax, nel), dict(nnodes=nodes))
    ob = O.AtomicBasis(10, lmax, mmax, nel, nnodes=nodes)
    ob.compute_tei()
    S = random_symmetric(ob.Nbf, seed=2201)
    G = S + 0.3 * np.triu(random_symmetric(ob.Nbf, seed=2202))
    sh = np.arange(ob.Nbf) // on.Nrad
    rng = np.random.default_rng(2203)
    keep = rng.random((on.Nang, on.Nang)) < 0.5
    D = S * (keep & keep.T)[sh][:, sh]  # runs of tiles with gaps
    for P in (S, G, D):
        Kr = ob.exchange(P)
        monkeypatch.setenv("HFGPU_EXCHANGE_CLASSES", "1")
        K1, ran = launched(gpu_ctx, lambda: K(on, P))
        assert relerr(K1, Kr) <= TOL and ran == (1, 0)
        K1, ran = launched(gpu_ctx, lambda: K(on, P, precision="fp32"))
        assert ran == (1, 0)
        e1 = relerr(K1, Kr)
        monkeypatch.setenv("HFGPU_EXCHANGE_CLASSES", "0")
        K0, ran = launched(gpu_ctx, lambda: K(off, P))
        assert relerr(K0, Kr) <= TOL and ran == (0, 1)
        e0 = relerr(K(off, P, precision="fp32"), Kr)
        print(f"fp32 error {e1:.2e}, other kernel {e0:.2e}", flush=True)
        assert e1 <= max(1.25 * e0, 4 * 2.0 ** -24)


@pytest.mark.parametrize("lmax,nel,nodes", [(2, 4, 10), (3, 6, 15)])
@pytest.mark.parametrize("ldiag", [True, False])
def test_fp32_no_further_off(lmax, nel, nodes, ldiag, gpu_ctx, monkeypatch):
    """The FP32 error of the class kernel is at most the other kernel's: both round
    density and factors alike, and the largest product of weights once.  Geometric
    mean over four densities; 1.0007 to 1.0073 when every weight was rounded by
    itself, 0.994 to 0.999 now."""
    import torch
    print(f"[gpu] class exchange FP32 error, lmax {lmax}", flush=True)
    (on, off), K = _bases(monkeypatch, gpu_ctx, (36, lmax, lmax, nel), dict(nnodes=nodes))
    sh = np.arange(on.Nbf) // on.Nrad
    l, m = np.asarray(on.lval)[sh], np.asarray(on.mval)[sh]
    ratio = []
    for seed in range(4):
        P = random_symmetric(on.Nbf, seed=2210 + seed)
        if ldiag:
            P = np.where((l[:, None] == l[None, :]) & (m[:, None] == m[None, :]), P, 0.0)
        monkeypatch.setenv("HFGPU_EXCHANGE_CLASSES", "0")
        ref = K(off, P)
        e0 = np.linalg.norm(K(off, P, precision="fp32") - ref)
        monkeypatch.setenv("HFGPU_EXCHANGE_CLASSES", "1")
        ratio.append(np.linalg.norm(K(on, P, precision="fp32") - ref) / e0)
    print("class / block kernel error", ratio, flush=True)
    assert np.exp(np.mean(np.log(ratio))) <= 1.0


def test_several_stages(gpu_ctx, monkeypatch):
    """lmax = 9: 167 tiles of one class, three stages of LDS, runs of five
    sources; the oracle takes minutes here, the other kernel stands in."""
    print("[gpu] class exchange in several stages", flush=True)
    (on, off), K = _bases(monkeypatch, gpu_ctx, (10, 9, 9, 2), dict(nnodes=3))
    P = random_symmetric(on.Nbf, seed=2204)
    m = np.repeat(on.mval, on.Nrad)
    P[m[:, None] != m[None, :]] = 0.0
    monkeypatch.setenv("HFGPU_EXCHANGE_CLASSES", "1")
    K1, ran = launched(gpu_ctx, lambda: K(on, P))
    assert ran == (1, 0)
    monkeypatch.setenv("HFGPU_EXCHANGE_CLASSES", "0")
    K0, ran = launched(gpu_ctx, lambda: K(off, P))
    assert ran == (0, 1)
    assert relerr(K1, K0) <= TOL


def test_batches_and_single_builds_in_turn(gpu_ctx, monkeypatch):
    """Batched launches do not read the class lists and do not build them: a single
    build of the same handle, pattern and precision does, before and after a batch."""
    import torch
    print("[gpu] class exchange between batched builds", flush=True)
    (on, off), K = _bases(monkeypatch, gpu_ctx, (10, 3, 2, 3), dict(nnodes=8))
    P = random_symmetric(on.Nbf, seed=2206)
    sh = np.arange(on.Nbf) // on.Nrad
    D = np.where((sh[:, None] == 1) | (sh[None, :] == 1), 0.0, P)
    monkeypatch.setenv("HFGPU_EXCHANGE_CLASSES", "0")
    ref = {k: (K(off, X), K(off, X, precision="fp32")) for k, X in (("P", P), ("D", D))}
    monkeypatch.setenv("HFGPU_EXCHANGE_CLASSES", "1")
    bt = H.AtomicBatch([on], gpu_ctx)
    for k, X in (("P", P), ("D", D), ("P", P)):
        Xd = torch.as_tensor(X, device="cuda")
        for prec, r, tol in (("fp32", ref[k][1], 2e-6), ("fp64", ref[k][0], TOL)):
            out = torch.empty_like(Xd)
            _, ran = launched(gpu_ctx, lambda: bt.exchange([Xd], [out], fp32=[prec == "fp32"]))
            assert ran == (0, 0) and relerr(out.cpu().numpy(), r) <= tol  # its own kernels
            K1, ran = launched(gpu_ctx, lambda: K(on, X, precision=prec))
            assert ran == (1, 0) and relerr(K1, r) <= tol


def test_yukawa_and_infinite_density(gpu_ctx, monkeypatch):
    """The Yukawa exchange through its own factors, and an infinite entry that
    reaches only the blocks coupled to its own."""
    import torch
    print("[gpu] class exchange, Yukawa factors and an infinite entry", flush=True)
    (on, off), K = _bases(monkeypatch, gpu_ctx, (4, 3, 2, 3), dict(nnodes=8))
    P = random_symmetric(on.Nbf, seed=2205)
    R, N = [], []
    Q = P.copy()
    Q[2, 3] = Q[3, 2] = np.inf
    for env, b in (("1", on), ("0", off)):
        monkeypatch.setenv("HFGPU_EXCHANGE_CLASSES", env)
        b.compute_yukawa(0.4)
        R.append(b.rs_exchange(torch.as_tensor(P, device="cuda")).cpu().numpy())
        N.append(K(b, Q))
    assert relerr(R[0], R[1]) <= TOL
    assert np.array_equal(np.isfinite(N[0]), np.isfinite(N[1]))
