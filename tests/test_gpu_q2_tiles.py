"""The 2D Q2 apply where its tiles end: meshes of one element, of whole tiles,
and with a remainder of one in each direction, with and without a reaction.

Bar: 1e-12 (FP64) and 2e-5 (FP32) of max |w|: a value sums the results of four
elements, each 2 * 27 products of up to four factors, whose rounding stays below
300 eps = 7e-14 and 4e-5 / 2 of the largest term."""
import numpy as np
import pytest

import dunefem_amd as fa
import pyoracle as ora

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1, 1), (1, 16), (15, 15), (16, 15), (14, 31), (46, 17)])
@pytest.mark.parametrize("c", [0.0, 0.7])
@pytest.mark.parametrize("kind", ["qp", "const"])
def test_q2_apply_at_tile_edges(ctx, n, c, kind):
    rng = np.random.default_rng(n[0] + 100 * n[1])
    kappa = np.exp(rng.normal(size=(n[0] * n[1], 9))) if kind == "qp" else 1.3
    oop = ora.CGOperator(n, c=c, kappa=kappa)
    u = rng.normal(size=(2 * n[0] + 1) * (2 * n[1] + 1))
    ref = oop.apply(u)
    for prec, tol in ((fa.F64, 1e-12), (fa.F32, 2e-5)):
        op = fa.GalerkinOperator(ctx, fa.OP_CG_Q2_2D, n, 2, c=c, kappa_mode=fa.KAPPA_QP if kind == "qp" else fa.KAPPA_CONST,
                                 kappa_const=1.0 if kind == "qp" else kappa, precision=prec)
        if kind == "qp":
            op.set_kappa_qp(kappa)
        U, W = op.vector(u), op.vector()
        W.fill(np.nan)
        op(U, W)
        err = np.abs(W.download() - ref).max() / np.abs(ref).max()
        print("q2", n, c, kind, prec, err, flush=True)
        assert err < tol


@pytest.mark.parametrize("n", [(2, 2), (16, 15), (46, 17)])
def test_q2_cg_with_the_applys_partials(ctx, n):
    """CG takes <q, A q> from the apply's workgroups.  u vanishes on the boundary:
    only there is the operator with its identity rows symmetric."""
    rng = np.random.default_rng(n[0] + 100 * n[1])
    kappa = np.exp(rng.normal(size=(n[0] * n[1], 9)))
    u = np.zeros((2 * n[1] + 1, 2 * n[0] + 1))
    u[1:-1, 1:-1] = rng.normal(size=(2 * n[1] - 1, 2 * n[0] - 1))
    u = u.ravel()
    op = fa.GalerkinOperator(ctx, fa.OP_CG_Q2_2D, n, 2, c=0.0, kappa_mode=fa.KAPPA_QP)
    op.set_kappa_qp(kappa)
    F, X = op.vector(ora.CGOperator(n, kappa=kappa).apply(u)), op.vector()
    inv = fa.InverseOperator(ctx, method=fa.CG, tolerance=1e-12, errormeasure=fa.RELATIVE, maxiterations=5000)
    inv.bind(op, fa.Preconditioner(op, fa.PRE_JACOBI))
    inv(F, X)
    assert inv.info()["converged"]
    # 1e-12 of |F| times the condition of the Jacobi-scaled operator, below 1e5
    # on these meshes and coefficients
    assert np.abs(X.download() - u).max() < 1e-6 * np.abs(u).max()


@pytest.mark.parametrize("use_graph", [True, False])
def test_batch_steps_over_uneven_instances(ctx, use_graph):
    """Instances of one tile and of many, one with a zero load (done at its
    first step), two solves with different step limits: a limit of one step
    per refinement must hold in a replayed graph as well."""
    sides = [(1, 1), (15, 15), (31, 46), (64, 3), (16, 16)]
    rng = np.random.default_rng(4)
    kv = [np.exp(rng.normal(size=(a * b, 9))) for a, b in sides]
    fq = [rng.normal(size=(a * b, 9)) * (i != 4) for i, (a, b) in enumerate(sides)]
    B = fa.Batch(ctx, sides)
    B.set_kappa_qp(np.concatenate(kv))
    F = B.rhs(np.concatenate(fq))
    X = B.vector()
    info = B.solve(F, X, tol=1e-10, use_graph=use_graph)
    assert info["converged"] == len(sides) and info["iterations"][4] == 0
    x, f = X.download(), F.download()
    for i, s in enumerate(sides):
        lo, hi = B.offsets[i], B.offsets[i + 1]
        r = f[lo:hi] - ora.CGOperator(s, kappa=kv[i]).apply(x[lo:hi])
        assert np.linalg.norm(r) <= 1.01e-10 * np.linalg.norm(f[lo:hi])
    Y = B.vector()
    info = B.solve(F, Y, tol=1e-10, inner_maxit=1, max_outer=3, use_graph=use_graph)
    assert info["outer_iterations"] == 3 and info["max_inner_iterations"] == 3
    assert all(n <= 3 for n in info["iterations"])
