"""J is written in whole columns, zeros included: 8- and 16-byte aligned targets,
padded leading dimensions, one to many elements of few or 15 functions, shells
without their first function, shells without any (one element of two nodes, m != 0),
and density pairs that do not fill a wave's run.

Bar: the oracle's J agrees to the rounding of sums over at most Nbf^2 products of
which a J entry sees a few thousand; 1e-12 of the largest entry covers 4500 * 2^-52.
Outside the matrix nothing may be written.
"""
import numpy as np
import pytest

import helfem_amd as H
import oracle as O
from helfem_amd._lib import check, lib
from helfem_amd.synthetic import random_symmetric

pytestmark = pytest.mark.gpu
TOL, MARK = 1e-12, -7.25

ATOMS = [(0, 0, 1, 15), (0, 0, 7, 2), (1, 1, 3, 2), (1, 0, 1, 3), (2, 2, 3, 15), (3, 1, 2, 6)]
DIATOMICS = [([1], 1, 15), ([0, 1], 2, 15), ([2, 1], 5, 3), ([3, 2, 1], 2, 8),
             ([0, 1], 1, 2), ([1, 1], 1, 2), ([2, 1], 1, 2)]


def _check(ob, hb, fn, ctx, pad, offset):
    import torch
    n, ld = ob.Nbf, ob.Nbf + pad
    P = random_symmetric(n, seed=6001)
    Jr = ob.coulomb(P)
    Pd = torch.from_numpy(P).cuda()
    buf = torch.full((offset + ld * n + 3,), MARK, dtype=torch.float64, device="cuda")
    ctx.bind_torch_stream()
    for _ in range(2):  # the second over the first's result
        check(fn(hb._h, Pd.data_ptr(), n, buf.data_ptr() + 8 * offset, ld))
    torch.cuda.synchronize()
    out = buf.cpu().numpy()
    J = out[offset:offset + ld * n].reshape(n, ld)
    assert np.max(np.abs(J[:, :n].T - Jr)) <= TOL * np.max(np.abs(Jr))
    assert np.all(out[:offset] == MARK) and np.all(out[offset + ld * n:] == MARK) and np.all(J[:, n:] == MARK)


@pytest.mark.parametrize("pad,offset", [(0, 0), (0, 1), (1, 0), (4, 1)])
@pytest.mark.parametrize("lmax,mmax,nelem,nnodes", ATOMS)
def test_atomic_columns(lmax, mmax, nelem, nnodes, pad, offset, gpu_ctx):
    print(f"[gpu] atomic J columns {lmax} {mmax} {nelem} {nnodes} +{pad} @{offset}", flush=True)
    ob = O.AtomicBasis(10, lmax, mmax, nelem, nnodes=nnodes)
    hb = H.AtomicBasis(10, lmax, mmax, nelem, nnodes=nnodes, ctx=gpu_ctx)
    ob.compute_tei()
    hb.compute_tei()
    _check(ob, hb, lib().hf_atomic_coulomb_dev, gpu_ctx, pad, offset)


@pytest.mark.parametrize("pad,offset", [(0, 0), (1, 1)])
@pytest.mark.parametrize("lmm,nelem,nnodes", DIATOMICS)
def test_diatomic_columns(lmm, nelem, nnodes, pad, offset, gpu_ctx):
    print(f"[gpu] diatomic J columns {lmm} {nelem} {nnodes} +{pad} @{offset}", flush=True)
    ob = O.DiatomicBasis(2, 1, 1.5, lmm, nelem, nnodes=nnodes)
    hb = H.DiatomicBasis(2, 1, 1.5, lmm, nelem, nnodes=nnodes, ctx=gpu_ctx)
    ob.compute_tei()
    hb.compute_tei()
    _check(ob, hb, lib().hf_diatomic_coulomb_dev, gpu_ctx, pad, offset)
