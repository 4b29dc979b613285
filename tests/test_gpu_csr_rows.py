"""The SpMV of a DG matrix, by rows below a million nonzeros and by elements without
column indices above: against the downloaded CSR arrays, on meshes whose elements
have from none to all six neighbours.

Bar: a row sums at most 875 products, so both sides differ by at most 2 * 875 eps =
4e-13 of sum |a| |x|; FP32 vectors add the rounding of the result, 6e-8 of |y|."""
import numpy as np
import pytest

import dunefem_amd as fa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1, 1, 1), (1, 1, 5), (2, 3, 1), (3, 4, 3)])
@pytest.mark.parametrize("p", [1, 2, 3, 4])
def test_dg_spmv_matches_its_arrays(ctx, n, p):
    rng = np.random.default_rng(p + sum(n))
    op = fa.GalerkinOperator(ctx, fa.OP_DG_SIPG_3D, n, p, 10.0 * p * p, (1, -.5, .25), 0.3, fa.KAPPA_CELL)
    op.set_kappa_cell(np.exp(rng.normal(size=n[0] * n[1] * n[2])))
    A = fa.SparseRowMatrix(op)
    S = A.to_scipy()
    for prec, eps in ((fa.F64, 0.0), (fa.F32, 6e-8)):
        x = rng.normal(size=op.N).astype(np.float64 if prec == fa.F64 else np.float32)
        X, Y = fa.DofVector(ctx, op.N, prec), fa.DofVector(ctx, op.N, prec)
        X.upload(x)
        Y.fill(np.nan)
        A(X, Y)
        ref = S @ x.astype(np.float64)
        bar = 4e-13 * (abs(S) @ np.abs(x.astype(np.float64))) + eps * np.abs(ref)
        err = np.abs(Y.download() - ref)
        print("csr", n, p, prec, (err / bar).max(), flush=True)
        assert (err <= bar).all()


@pytest.mark.parametrize("p,n", [
    # a million nonzeros and more, from where on the element kernel is taken: rows of
    # elements with one, two, three and up to six neighbours
    (1, (1, 1, 5500)), (1, (70, 60, 1)), (1, (13, 15, 16)),
    (2, (480, 1, 1)), (2, (2, 3, 70)), (2, (7, 6, 8)),
    (3, (1, 90, 1)), (3, (4, 3, 5)), (4, (1, 1, 24)), (4, (3, 3, 2)),
])
def test_large_dg_spmv_matches_its_arrays(ctx, p, n):
    test_dg_spmv_matches_its_arrays(ctx, n, p)
