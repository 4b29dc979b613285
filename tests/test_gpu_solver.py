"""GPU Krylov solvers and preconditioners against the oracle (through the C ABI).

CG follows LinearSolver::cg exactly (same recurrence and stopping rule), so the
iteration count matches the oracle's up to rounding (+-1) and the solutions
agree to the solver tolerance.  GMRES/FGMRES are checked against the oracle's
restatement and a dense solve.  Every solve is also checked by its FP64 true
relative residual.
"""
import numpy as np
import pytest

import dunefem_amd as fa
import pyoracle as ora
from dunefem_amd import workloads as wl

pytestmark = pytest.mark.gpu


def cg_problem(ctx, n=(64, 64)):
    P = wl.problem0(n=n[0])
    gop = fa.GalerkinOperator(ctx, fa.OP_CG_Q2_2D, n, 2, c=1.0)
    oop = ora.CGOperator(n, c=1.0)
    return P, gop, oop


def test_cg_jacobi_problem0_matches_oracle(ctx):
    P, gop, oop = cg_problem(ctx)
    F = oop.rhs(P["fq"])
    xo, ito = ora.cg(oop, F, pre=ora.jacobi(1.0 / oop.diag()), tol=1e-10, maxit=5000, criteria=1)
    B = gop.rhs(P["fq"])
    assert np.abs(B.download() - F).max() < 1e-12 * np.abs(F).max()
    X = gop.vector()
    pre = fa.Preconditioner(gop, fa.PRE_JACOBI)
    inv = fa.InverseOperator(ctx, method=fa.CG, tolerance=1e-10, errormeasure=fa.RELATIVE, maxiterations=5000)
    inv.bind(gop, pre)
    inv(B, X)
    info = inv.info()
    print("problem0 CG+Jacobi: gpu its", info["iterations"], "oracle its", ito, "true rel res",
          info["true_rel_residual"], "time", info["timing"], flush=True)
    assert info["converged"] and abs(info["iterations"] - ito) <= 1
    x = X.download()
    assert np.abs(x - xo).max() < 1e-8 * np.abs(xo).max()
    assert info["true_rel_residual"] < 1e-9


def test_cg_unpreconditioned_and_maxit(ctx):
    P, gop, oop = cg_problem(ctx, (24, 20))
    F = oop.rhs(np.random.default_rng(1).normal(size=(480, 9)))
    xo, ito = ora.cg(oop, F, tol=1e-9, maxit=5000, criteria=1)
    B, X = gop.vector(F), gop.vector()
    inv = fa.InverseOperator(ctx, method=fa.CG, tolerance=1e-9, errormeasure=fa.RELATIVE, maxiterations=5000)
    inv.bind(gop)
    inv(B, X)
    assert abs(inv.iterations() - ito) <= 1
    assert np.abs(X.download() - xo).max() < 1e-7 * np.abs(xo).max()
    # non-convergence is a negative count, not an error (cg.hh:116)
    inv2 = fa.InverseOperator(ctx, method=fa.CG, tolerance=1e-14, errormeasure=fa.RELATIVE, maxiterations=7)
    inv2.bind(gop)
    X.clear()
    inv2(B, X)
    assert inv2.iterations() == -7 and not inv2.info()["converged"]


def dg_small(ctx, n, p, kappa, b=(0, 0, 0), prec=fa.F64):
    if kappa[0] == "cell":
        op = fa.GalerkinOperator(ctx, fa.OP_DG_SIPG_3D, n, p, 10.0 * p * p, b, 0.0, fa.KAPPA_CELL, precision=prec)
        op.set_kappa_cell(kappa[1])
    else:
        op = fa.GalerkinOperator(ctx, fa.OP_DG_SIPG_3D, n, p, 10.0 * p * p, b, 0.0, fa.KAPPA_QP, precision=prec)
        op.set_kappa_qp(kappa[1], kappa[2])
    return op


@pytest.mark.parametrize("method", ["gmres", "fgmres"])
def test_gmres_matches_oracle_and_dense(ctx, method):
    rng = np.random.default_rng(2)
    n, p = (4, 3, 3), 2
    E = 36
    kc = rng.uniform(0.5, 5.0, size=E)
    oop = ora.DGOperator(n, p, 40.0, (1, .5, .25), 0.0, kappa=("cell", kc))
    gop = dg_small(ctx, n, p, ("cell", kc), b=(1, .5, .25))
    b = rng.normal(size=oop.N)
    f = ora.gmres if method == "gmres" else ora.fgmres
    xo, ito = f(oop, b, tol=1e-10, maxit=2000, criteria=1, restart=15)
    B, X = gop.vector(b), gop.vector()
    inv = fa.InverseOperator(ctx, method=fa.GMRES if method == "gmres" else fa.FGMRES, tolerance=1e-10,
                             errormeasure=fa.RELATIVE, maxiterations=2000, restart=15)
    inv.bind(gop)
    inv(B, X)
    info = inv.info()
    print(method, "gpu its", info["iterations"], "oracle its", ito, "res", info["true_rel_residual"], flush=True)
    assert info["converged"] and abs(info["iterations"] - ito) <= 2
    assert info["true_rel_residual"] < 1.5e-10
    assert np.abs(X.download() - xo).max() < 1e-7 * np.abs(xo).max()


def test_block_jacobi_is_exact_element_inverse(ctx):
    # cellwise kappa, b = 0: the tensor-product eigen-decomposition gives A_KK^-1 exactly
    rng = np.random.default_rng(3)
    n, p = (3, 2, 4), 2
    kc = 10.0 ** rng.integers(0, 5, size=24).astype(float)
    oop = ora.DGOperator(n, p, 40.0, kappa=("cell", kc))
    blocks = oop.block_diag()
    gop = dg_small(ctx, n, p, ("cell", kc))
    pre = fa.Preconditioner(gop, fa.PRE_BLOCK_JACOBI)
    x = rng.normal(size=oop.N)
    X, Y = gop.vector(x), gop.vector()
    pre(X, Y)
    nb = 27
    ref = np.linalg.solve(blocks, x.reshape(-1, nb)[..., None])[..., 0].ravel()
    err = np.abs(Y.download() - ref).max() / np.abs(ref).max()
    print("block jacobi rel err", err, flush=True)
    assert err < 1e-11


@pytest.mark.parametrize("n,p", [((12, 12, 12), 2), ((8, 6, 5), 3)])
def test_cg_block_jacobi_matches_oracle(ctx, n, p):
    # CG + block Jacobi on DG operators: the apply and the preconditioner
    # hand the solver per-workgroup partials of its dots (Q2: the high-
    # contrast channel problem at 12^3; Q3: random cellwise kappa)
    if p == 2:
        P = wl.problem3(n=n[0])
        kcell, fq, beta = P["kcell"], P["fq"], P["beta"]
    else:
        rng = np.random.default_rng(31)
        E = n[0] * n[1] * n[2]
        kcell = rng.uniform(0.1, 10.0, size=E)
        fq = rng.normal(size=(E, (p + 1) ** 3))
        beta = 10.0 * p * p
    gop = fa.GalerkinOperator(ctx, fa.OP_DG_SIPG_3D, n, p, beta, (0, 0, 0), 0.0, fa.KAPPA_CELL)
    gop.set_kappa_cell(kcell)
    pre = fa.Preconditioner(gop, fa.PRE_BLOCK_JACOBI)
    F = gop.rhs(fq)
    X = gop.vector()
    inv = fa.InverseOperator(ctx, method=fa.CG, tolerance=1e-8, errormeasure=fa.RELATIVE, maxiterations=5000)
    inv.bind(gop, pre)
    inv(F, X)
    info = inv.info()
    oop = ora.DGOperator(n, p, beta, kappa=("cell", kcell))
    inv_blocks = np.linalg.inv(oop.block_diag())
    xo, ito = ora.cg(oop, F.download(), pre=ora.block_jacobi(inv_blocks), tol=1e-8, maxit=5000, criteria=1)
    print("CG+BJ", n, p, "gpu its", info["iterations"], "oracle its", ito, "res", info["true_rel_residual"], flush=True)
    assert info["converged"] and ito > 0
    assert abs(info["iterations"] - ito) <= 2
    assert np.abs(X.download() - xo).max() < 1e-6 * np.abs(xo).max()


def test_cg_block_jacobi_nonzero_initial_guess(ctx):
    # x is the initial guess on entry (inverseoperatorinterface.hh operator()(u, w))
    rng = np.random.default_rng(43)
    n, p = (5, 4, 4), 3
    E = n[0] * n[1] * n[2]
    kcell = rng.uniform(0.2, 5.0, size=E)
    gop = fa.GalerkinOperator(ctx, fa.OP_DG_SIPG_3D, n, p, 90.0, (0, 0, 0), 0.0, fa.KAPPA_CELL)
    gop.set_kappa_cell(kcell)
    pre = fa.Preconditioner(gop, fa.PRE_BLOCK_JACOBI)
    F = gop.rhs(rng.normal(size=(E, (p + 1) ** 3)))
    x0 = rng.normal(size=gop.N)
    X = gop.vector(x0)
    inv = fa.InverseOperator(ctx, method=fa.CG, tolerance=1e-9, errormeasure=fa.RELATIVE, maxiterations=5000)
    inv.bind(gop, pre)
    inv(F, X)
    info = inv.info()
    oop = ora.DGOperator(n, p, 90.0, kappa=("cell", kcell))
    xo, ito = ora.cg(oop, F.download(), x0=x0, pre=ora.block_jacobi(np.linalg.inv(oop.block_diag())), tol=1e-9,
                     maxit=5000, criteria=1)
    print("CG+BJ x0", "gpu its", info["iterations"], "oracle its", ito, flush=True)
    assert info["converged"] and abs(info["iterations"] - ito) <= 2
    assert np.abs(X.download() - xo).max() < 1e-6 * np.abs(xo).max()


def test_fgmres_block_jacobi_problem3_small(ctx):
    # the high-contrast channel problem at 12^3: FGMRES(30) + block Jacobi to 1e-8
    P = wl.problem3(n=12)
    gop = dg_small(ctx, P["n"], P["p"], ("cell", P["kcell"]))
    pre = fa.Preconditioner(gop, fa.PRE_BLOCK_JACOBI)
    F = gop.rhs(P["fq"])
    X = gop.vector()
    inv = fa.InverseOperator(ctx, method=fa.FGMRES, tolerance=1e-8, errormeasure=fa.RELATIVE,
                             maxiterations=5000, restart=30)
    inv.bind(gop, pre)
    inv(F, X)
    info = inv.info()
    print("problem3 12^3 FGMRES+BJ", info, flush=True)
    assert info["converged"] and info["true_rel_residual"] < 1.01e-8
    # the oracle reaches the same residual with the same iteration count (+-2)
    oop = ora.DGOperator(P["n"], P["p"], P["beta"], kappa=("cell", P["kcell"]))
    inv_blocks = np.linalg.inv(oop.block_diag())
    xo, ito = ora.fgmres(oop, F.download(), pre=ora.block_jacobi(inv_blocks), tol=1e-8, maxit=5000,
                         criteria=1, restart=30)
    assert abs(info["iterations"] - ito) <= 2
    assert np.abs(X.download() - xo).max() < 1e-6 * np.abs(xo).max()


@pytest.mark.parametrize("method", [fa.CG, fa.FGMRES])
def test_mixed_precision_refinement_reaches_fp64_residual(ctx, method):
    P = wl.problem3(n=12)
    op64 = dg_small(ctx, P["n"], P["p"], ("cell", P["kcell"]))
    op32 = dg_small(ctx, P["n"], P["p"], ("cell", P["kcell"]), prec=fa.F32)
    pre32 = fa.Preconditioner(op32, fa.PRE_BLOCK_JACOBI)
    F = op64.rhs(P["fq"])
    X = op64.vector()
    inv = fa.InverseOperator(ctx, method=method, tolerance=1e-8, errormeasure=fa.RELATIVE, maxiterations=20000,
                             restart=30, refinement=1, inner_tolerance=1e-3, inner_maxiterations=2000)
    inv.bind(op64, None, op32, pre32)
    inv(F, X)
    info = inv.info()
    print("IR", method, info, flush=True)
    assert info["converged"] and info["true_rel_residual"] <= 1e-8
    assert info["outer_iterations"] >= 2


def bicgstab_count_slack(ito):
    # BiCGStab's residual is not monotone and the reference's stopping value
    # sqrt(<s,s> - w(2<r,s> - w<r,r>)) cancels near convergence, so the
    # order of the dot-product sums moves the step at which it first falls
    # below the tolerance (measured: 215 vs 204, 146 vs 149 steps). The
    # iterates themselves are compared step by step in
    # bicgstab_iterates_agree.
    return max(2, ito // 10)


def bicgstab_iterates_agree(ctx, op, oop, b, pre=False):
    # after a fixed number of steps (the solver stops at maxiterations and
    # reports a negative count) the GPU iterate equals the oracle's to
    # rounding: a dropped term or a wrong sign in any update shows here
    inv_blocks = np.linalg.inv(oop.block_diag()) if pre else None
    for k in (1, 2, 5, 12):
        xo, ito = ora.bicgstab(oop, b, pre=ora.block_jacobi(inv_blocks) if pre else None, tol=1e-15, maxit=k,
                               criteria=1, nthreads=8)
        inv = fa.InverseOperator(ctx, method=fa.BICGSTAB, tolerance=1e-15, errormeasure=fa.RELATIVE, maxiterations=k)
        inv.bind(op, fa.Preconditioner(op, fa.PRE_BLOCK_JACOBI) if pre else None)
        X = op.vector(np.zeros(op.N))
        inv(op.vector(b), X)
        assert ito == -k and inv.iterations() == -k
        x = X.download()
        err = np.abs(x - xo).max() / np.abs(xo).max()
        print("bicgstab step", k, "iterate rel diff", err, flush=True)
        assert err < 1e-10, (k, err)


def test_bicgstab_matches_oracle(ctx):
    # LinearSolver::bicgstab restated (bicgstab.hh:56-222): nonsymmetric SIPG
    # with advection, unpreconditioned; iteration count and solution against
    # the oracle
    rng = np.random.default_rng(12)
    n, p = (5, 4, 3), 2
    kc = rng.uniform(0.5, 2.0, size=60)
    oop = ora.DGOperator(n, p, 40.0, (1.0, -0.5, 0.25), 0.0, kappa=("cell", kc))
    b = rng.normal(size=oop.N)
    xo, ito = ora.bicgstab(oop, b, tol=1e-10, maxit=3000, criteria=1)
    op = fa.GalerkinOperator(ctx, fa.OP_DG_SIPG_3D, n, p, 40.0, (1.0, -0.5, 0.25), 0.0, fa.KAPPA_CELL)
    op.set_kappa_cell(kc)
    inv = fa.InverseOperator(ctx, method=fa.BICGSTAB, tolerance=1e-10, errormeasure=fa.RELATIVE, maxiterations=3000)
    inv.bind(op)
    X = op.vector()
    inv(op.vector(b), X)
    info = inv.info()
    print("bicgstab gpu its", info["iterations"], "oracle its", ito, "true rel res", info["true_rel_residual"], flush=True)
    assert info["converged"] and info["true_rel_residual"] < 1e-9
    assert abs(info["iterations"] - ito) <= bicgstab_count_slack(ito)
    assert np.abs(X.download() - xo).max() <= 1e-7 * np.abs(xo).max()
    bicgstab_iterates_agree(ctx, op, oop, b)
    # non-convergence is a negative count
    inv2 = fa.InverseOperator(ctx, method=fa.BICGSTAB, tolerance=1e-14, errormeasure=fa.RELATIVE, maxiterations=3)
    inv2.bind(op)
    X.clear()
    inv2(op.vector(b), X)
    assert inv2.iterations() == -3 and not inv2.info()["converged"]


def test_bicgstab_block_jacobi_diffusion_matches_oracle(ctx):
    rng = np.random.default_rng(13)
    n, p = (5, 4, 3), 3
    kc = 10.0 ** rng.uniform(-1, 1, size=60)
    oop = ora.DGOperator(n, p, 90.0, (0, 0, 0), 0.0, kappa=("cell", kc))
    b = rng.normal(size=oop.N)
    xo, ito = ora.bicgstab(oop, b, pre=ora.block_jacobi(np.linalg.inv(oop.block_diag())), tol=1e-10, maxit=3000,
                           criteria=1, nthreads=8)
    op = fa.GalerkinOperator(ctx, fa.OP_DG_SIPG_3D, n, p, 90.0, (0, 0, 0), 0.0, fa.KAPPA_CELL)
    op.set_kappa_cell(kc)
    inv = fa.InverseOperator(ctx, method=fa.BICGSTAB, tolerance=1e-10, errormeasure=fa.RELATIVE, maxiterations=3000)
    inv.bind(op, fa.Preconditioner(op, fa.PRE_BLOCK_JACOBI))
    X = op.vector(np.zeros(op.N))
    inv(op.vector(b), X)
    info = inv.info()
    print("bicgstab+bj gpu its", info["iterations"], "oracle its", ito, flush=True)
    assert info["converged"] and abs(info["iterations"] - ito) <= bicgstab_count_slack(ito)
    assert np.abs(X.download() - xo).max() <= 1e-7 * np.abs(xo).max()
    bicgstab_iterates_agree(ctx, op, oop, b, pre=True)


@pytest.mark.parametrize("method", ["gmres", "fgmres"])
@pytest.mark.parametrize("n,restart", [((1, 1, 1), 5), ((3, 2, 2), 1), ((3, 3, 3), 9), ((7, 6, 5), 33), ((23, 9, 8), 64)])
def test_gmres_steps_minimise_the_residual(ctx, method, n, restart):
    # after k steps the estimate |g_k| is the norm of b - A x over the Krylov
    # space: the true residual of the returned iterate equals it.  Sizes: fewer
    # DoFs than a slice of the dots, one and several groups of 8 basis vectors,
    # the longest cycle.  Classical Gram-Schmidt loses orthogonality like the
    # condition of the Krylov basis, far below 1e-8 of |b| over these few steps
    rng = np.random.default_rng(restart)
    op = fa.GalerkinOperator(ctx, fa.OP_DG_SIPG_3D, n, 2, 40.0, (1.0, -0.5, 0.25), 0.5, fa.KAPPA_CELL)
    op.set_kappa_cell(rng.uniform(0.5, 2.0, size=n[0] * n[1] * n[2]))
    b = rng.normal(size=op.N)
    last = None
    for k in (1, restart // 2 + 1, restart):
        inv = fa.InverseOperator(ctx, method=getattr(fa, method.upper()), tolerance=1e-14, errormeasure=fa.RELATIVE,
                                 maxiterations=k, restart=restart)
        inv.bind(op, fa.Preconditioner(op, fa.PRE_JACOBI))
        B, X, W = op.vector(b), op.vector(np.zeros(op.N)), op.vector()
        inv(B, X)
        assert abs(inv.iterations()) <= k
        op(X, W)
        r = np.linalg.norm(W.download() - b) / np.linalg.norm(b)
        assert abs(r - inv.info()["true_rel_residual"]) < 1e-8
        assert r < 1.0 + 1e-8 and (last is None or r <= last + 1e-8)
        # the minimum over the same space, by dense least squares (small cases)
        if op.N <= 800 and k <= 9:
            A = np.empty((op.N, op.N))
            e = np.zeros(op.N)
            for i in range(op.N):
                e[:] = 0
                e[i] = 1
                op(op.vector(e), W)
                A[:, i] = W.download()
            dinv = 1.0 / np.diag(A)
            V = [b / np.linalg.norm(b)]
            for _ in range(k - 1):
                V.append(A @ (dinv * V[-1]))
                V[-1] /= np.linalg.norm(V[-1])
            M = np.array([A @ (dinv * v) for v in V]).T
            y = np.linalg.lstsq(M, b, rcond=None)[0]
            assert abs(r - np.linalg.norm(b - M @ y) / np.linalg.norm(b)) < 1e-7
        last = r


@pytest.mark.parametrize("case", ["none", "one_element", "jacobi", "jacobi_many_partials", "lagrange_jacobi", "bj",
                                  "bj_fp32_inner", "mg", "mg32", "bf16"])
@pytest.mark.parametrize("graph", [0, 1])
def test_cg_steps_match_the_recurrence(ctx, case, graph):
    # the iterate after k steps against the recurrence of cg.hh:19-117 on the
    # host with the same apply and preconditioner.  Each way a step takes its
    # dots: from the apply, from the preconditioner, from passes over the
    # vectors, from more partials than a workgroup sums.  The recurrences differ
    # by the rounding of the dots, about 1e-16 sqrt(N) per step, amplified by
    # less than the condition number (below 1e5 here): 1e-8 in FP64, 1e-2 in
    # FP32 and BF16
    rng = np.random.default_rng(3)
    n, p, prec, kind = (7, 6, 5), 2, fa.F64, fa.KAPPA_CELL
    if case == "one_element":
        n = (1, 1, 1)
    if case == "jacobi_many_partials":
        n, p, kind = (16, 66, 65), 1, fa.KAPPA_QP
    if case == "bj_fp32_inner":
        prec = fa.F32
    if case == "bf16":
        prec = fa.BF16MFMA
    if case == "lagrange_jacobi":
        op = fa.GalerkinOperator(ctx, fa.OP_CG_Q2_2D, (37, 29), 2, c=1.0)
    else:
        m, E = p + 1, n[0] * n[1] * n[2]
        op = fa.GalerkinOperator(ctx, fa.OP_DG_SIPG_3D, n, p, 10.0 * p * p, (0, 0, 0), 0.0, kind, precision=prec)
        if kind == fa.KAPPA_CELL:
            op.set_kappa_cell(rng.uniform(0.5, 2.0, size=E))
        else:
            op.set_kappa_qp(np.full((E, m ** 3), 1.5),
                            [np.full(((n[0] + (d == 0)) * (n[1] + (d == 1)) * (n[2] + (d == 2)), m * m), 1.5)
                             for d in range(3)])
    pre = None
    if "jacobi" in case:
        pre = fa.Preconditioner(op, fa.PRE_JACOBI)
    elif "bj" in case or case == "bf16":
        pre = fa.Preconditioner(op, fa.PRE_BLOCK_JACOBI)
    elif case == "mg":
        pre = fa.Preconditioner(op, fa.PRE_MULTIGRID)
    elif case == "mg32":
        op32 = fa.GalerkinOperator(ctx, fa.OP_DG_SIPG_3D, n, p, 10.0 * p * p, (0, 0, 0), 0.0, kind, precision=fa.F32)
        op32.set_kappa_cell(np.random.default_rng(3).uniform(0.5, 2.0, size=E))
        pre = fa.Preconditioner(op32, fa.PRE_MULTIGRID)
    U, W = op.vector(), op.vector()
    P32 = (op32.vector(), op32.vector()) if case == "mg32" else None

    def A(v):
        U.upload(v)
        op(U, W)
        return W.download()

    def M(v):
        if pre is None:
            return v.copy()
        a, b = P32 or (U, W)
        a.upload(v)
        pre(a, b)
        return b.download()

    b = rng.normal(size=op.N)
    if case == "lagrange_jacobi":
        b = A(b)
    for k in (1, 2, 6):
        x = np.zeros(op.N)
        r = b - A(x)
        q = M(r)
        s, res = q.copy(), np.dot(r, q)
        for it in range(k):
            if it:
                q = s + beta * q
            h = A(q)
            alpha = res / np.dot(q, h)
            x, r = x + alpha * q, r - alpha * h
            s = M(r)
            new = np.dot(r, s)
            beta, res = new / res, new
        inv = fa.InverseOperator(ctx, method=fa.CG, tolerance=1e-30, errormeasure=fa.RELATIVE, maxiterations=k, graph=graph)
        inv.bind(op, pre)
        X = op.vector(np.zeros(op.N))
        inv(op.vector(b), X)
        assert inv.iterations() == -k
        err = np.linalg.norm(X.download() - x) / np.linalg.norm(x)
        print("cg", case, k, err, flush=True)
        assert err < (1e-8 if prec == fa.F64 else 1e-2)


@pytest.mark.parametrize("prec", [fa.F64, fa.F32])
def test_cg_steps_with_many_block_jacobi_partials(ctx, prec):
    # 64 x 65 x 65 Q1 elements: 4420 workgroups of the apply and 4225 of block
    # Jacobi, so both of its lists and that of <q, A q> are first brought down to
    # fewer.  Bars as in test_cg_steps_match_the_recurrence
    n, rng = (64, 65, 65), np.random.default_rng(5)
    op = fa.GalerkinOperator(ctx, fa.OP_DG_SIPG_3D, n, 1, 10.0, (0, 0, 0), 0.0, fa.KAPPA_CELL, precision=prec)
    op.set_kappa_cell(rng.uniform(0.5, 2.0, size=n[0] * n[1] * n[2]))
    pre = fa.Preconditioner(op, fa.PRE_BLOCK_JACOBI)
    U, W = op.vector(), op.vector()

    def on_device(call, v):
        U.upload(v)
        call(U, W)
        return W.download().astype(np.float64)

    b = rng.normal(size=op.N)
    for k in (1, 2, 6):
        x, r = np.zeros(op.N), b
        q = s = on_device(pre, r)
        res = np.dot(r, s)
        for it in range(k):
            q = s + beta * q if it else s
            h = on_device(op, q)
            alpha = res / np.dot(q, h)
            x, r = x + alpha * q, r - alpha * h
            s = on_device(pre, r)
            new = np.dot(r, s)
            beta, res = new / res, new
        inv = fa.InverseOperator(ctx, method=fa.CG, tolerance=1e-30, errormeasure=fa.RELATIVE, maxiterations=k)
        inv.bind(op, pre)
        X = op.vector(np.zeros(op.N))
        inv(op.vector(b), X)
        assert inv.iterations() == -k
        err = np.linalg.norm(X.download() - x) / np.linalg.norm(x)
        print("cg many", k, err, flush=True)
        assert err < (1e-8 if prec == fa.F64 else 1e-2)
