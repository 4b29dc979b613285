"""The modal apply and sweep (kappa constant per element): parity with the
oracle where tiles, walks and rows end unevenly.

Bar: as in test_gpu_apply.py, 1e-12 (FP64) and 2e-5 (FP32) of max |w|: both
sides sum about 10 K^2 terms per value, whose rounding stays below K^2 10 eps =
6e-14 and 3e-5 / 2 of the largest term at K = 5.
"""
import time

import numpy as np
import pytest

import dunefem_amd as fa
import mg_oracle as mgo
import pyoracle as ora

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


def operator(ctx, n, p, b, c, kappa, prec=fa.F64):
    cell = not np.isscalar(kappa)
    op = fa.GalerkinOperator(ctx, fa.OP_DG_SIPG_3D, n, p, 10.0 * p * p, b, c, fa.KAPPA_CELL if cell else fa.KAPPA_CONST,
                             1.0 if cell else kappa, precision=prec)
    if cell:
        op.set_kappa_cell(kappa)
    return op


@pytest.mark.parametrize("n,p,b,c,kind", [
    # one element, and one element thick in each direction
    ((1, 1, 1), 2, (1, -.5, .25), 0.3, "cell"),
    ((9, 1, 1), 3, (1, -.5, .25), 0.0, "cell"),
    ((1, 9, 1), 4, (0, 0, 0), 0.0, "cell"),
    ((1, 1, 9), 4, (-1, .5, .25), 0.2, "const"),
    ((1, 7, 6), 1, (1, .5, .25), 0.0, "cell"),
    # tiles and rows with a remainder in both directions
    ((6, 17, 5), 1, (1, -.5, .25), 0.0, "cell"),
    ((5, 9, 13), 2, (0, 0, 0), 0.4, "cell"),
    ((4, 7, 11), 3, (-1, .5, -.25), 0.0, "cell"),
    ((3, 5, 7), 4, (1, .5, .25), 0.0, "cell"),
    # walks of two steps, the last of them shorter
    ((41, 40, 60), 2, (1, .5, .25), 0.0, "cell"),
    ((41, 33, 33), 3, (0, 0, 0), 0.0, "cell"),
    ((41, 21, 33), 4, (1, -.5, .25), 0.1, "cell"),
])
def test_modal_apply_matches_oracle(ctx, n, p, b, c, kind):
    rng = np.random.default_rng(sum(n) + p)
    kappa = np.exp(rng.normal(size=n[0] * n[1] * n[2])) if kind == "cell" else 1.3
    oop = ora.DGOperator(n, p, 10.0 * p * p, b, c, kappa=("cell", kappa) if kind == "cell" else kappa)
    u = rng.normal(size=oop.N)
    ref = oop.apply(u)
    for prec, tol in ((fa.F64, 1e-12), (fa.F32, 2e-5)):
        op = operator(ctx, n, p, b, c, kappa, prec)
        U, W = op.vector(u), op.vector()
        W.fill(np.nan)
        op(U, W)
        err = rel(W.download(), ref)
        print("modal", n, p, kind, prec, err, flush=True)
        assert err < tol


@pytest.mark.parametrize("n,p", [((7, 5, 6), 1), ((9, 6, 5), 2), ((5, 7, 4), 3), ((7, 6, 5), 4)])
def test_sweep_equals_apply_and_block_inverse(ctx, n, p):
    """One V-cycle smooths with fused sweeps; the block inverse of the oracle's
    element blocks gives the same Krylov solve, and two V-cycles agree bit for
    bit (a sweep's workgroups exchange data through LDS)."""
    rng = np.random.default_rng(5 + p)
    op = operator(ctx, n, p, (0, 0, 0), 0.0, np.exp(rng.normal(size=n[0] * n[1] * n[2])))
    mg = fa.Preconditioner(op, fa.PRE_MULTIGRID)
    R = op.vector(rng.normal(size=op.N))
    Z = [op.vector(), op.vector()]
    for z in Z:
        mg(R, z)
    assert np.array_equal(Z[0].download(), Z[1].download())
    F = op.vector(rng.normal(size=op.N))
    X = [op.vector(), op.vector()]
    for x, pre in zip(X, (mg, fa.Preconditioner(op, fa.PRE_BLOCK_JACOBI))):
        inv = fa.InverseOperator(ctx, method=fa.CG, tolerance=1e-11, errormeasure=fa.RELATIVE, maxiterations=5000)
        inv.bind(op, pre)
        inv(F, x)
        assert inv.info()["converged"]
    # both stop at 1e-11 of |F|; the operator's smallest eigenvalue bounds the
    # distance of the two solutions by 2e-11 times its condition, about 1e4
    assert rel(X[0].download(), X[1].download()) < 1e-6


@pytest.mark.parametrize("n,p", [((1, 1, 1), 2), ((6, 17, 5), 1), ((5, 9, 13), 2), ((4, 7, 11), 3), ((3, 5, 7), 4)])
def test_reaction_apply_matches_oracle(ctx, n, p):
    """The pass to the Gauss points and back, at rows with a remainder."""
    rng = np.random.default_rng(sum(n) + p)
    E = n[0] * n[1] * n[2]
    kappa, cvol = np.exp(rng.normal(size=E)), rng.uniform(0.5, 2.0, size=(E, (p + 1) ** 3))
    oop = ora.DGOperator(n, p, 10.0 * p * p, (1, -.5, .25), 0.3, kappa=("cell", kappa))
    oop.set_reaction_qp(cvol)
    u = rng.normal(size=oop.N)
    ref = oop.apply(u)
    for prec, tol in ((fa.F64, 1e-12), (fa.F32, 2e-5)):
        op = operator(ctx, n, p, (1, -.5, .25), 0.3, kappa, prec)
        op.set_reaction_qp(cvol)
        U, W = op.vector(u), op.vector()
        W.fill(np.nan)
        op(U, W)
        err = rel(W.download(), ref)
        print("reaction", n, p, prec, err, flush=True)
        assert err < tol


@pytest.mark.parametrize("n,p,reaction", [
    # one to three vertex levels, vertex counts with a remainder of the
    # wavefront, even and odd last coarse cells, one cell in a direction
    ((1, 30, 23), 1, True), ((6, 17, 9), 1, False), ((18, 23, 21), 1, True),
    ((12, 9, 13), 2, True), ((9, 12, 6), 3, False),
])
def test_vcycle_matches_oracle_on_odd_lattices(ctx, n, p, reaction):
    """Bars as in test_gpu_multigrid.py: the cycle's sums are those of its
    levels' applies, 1e-12 of max |z| (FP64) and 1e-4 of |z| (FP32)."""
    rng = np.random.default_rng(sum(n) + p)
    E = n[0] * n[1] * n[2]
    kappa, cvol = np.exp(rng.normal(size=E)), rng.uniform(0.5, 2.0, size=(E, (p + 1) ** 3)) if reaction else None
    M = mgo.MGOracle(n, p, 10.0 * p * p, ("cell", kappa), **({"cvol": cvol} if reaction else {}))
    r = rng.normal(size=E * (p + 1) ** 3)
    ref = M.apply(r)
    for prec in (fa.F64, fa.F32):
        op = operator(ctx, n, p, (0, 0, 0), 0.0, kappa, prec)
        if reaction:
            op.set_reaction_qp(cvol)
        R, Z = op.vector(r), op.vector()
        Z.fill(np.nan)
        fa.Preconditioner(op, fa.PRE_MULTIGRID)(R, Z)
        z = Z.download()
        print("vcycle", n, p, prec, rel(z, ref), flush=True)
        if prec == fa.F64:
            assert rel(z, ref) < 1e-12
        else:
            assert np.linalg.norm(z - ref) < 1e-4 * np.linalg.norm(ref)


@pytest.mark.parametrize("n", [(1, 1, 1), (13, 3, 1), (801, 1, 1), (773, 2, 1), (775, 1, 2)])
@pytest.mark.parametrize("p", [2, 3, 4])
def test_meshes_thin_in_y_and_z(ctx, n, p):
    """Apply, and CG with the apply's partials of <q, A q>, on meshes that fill less
    than half of a tile."""
    rng = np.random.default_rng(sum(n) + p)
    kappa = np.exp(rng.normal(size=n[0] * n[1] * n[2]))
    oop = ora.DGOperator(n, p, 10.0 * p * p, (1, -.5, .25), 0.3, kappa=("cell", kappa))
    u = rng.normal(size=oop.N)
    ref = oop.apply(u)
    for prec, tol in ((fa.F64, 1e-12), (fa.F32, 2e-5)):
        op = operator(ctx, n, p, (1, -.5, .25), 0.3, kappa, prec)
        U, W = op.vector(u), op.vector()
        W.fill(np.nan)
        op(U, W)
        assert rel(W.download(), ref) < tol
    # two steps of CG with Jacobi: alpha by the apply's partials
    op = operator(ctx, n, p, (0, 0, 0), 0.0, kappa)
    U, W, D = op.vector(), op.vector(), op.vector()

    def A(v):
        U.upload(v)
        op(U, W)
        return W.download()

    op.diagonal(D)
    dinv, b = 1.0 / D.download(), rng.normal(size=op.N)
    q = s = dinv * b
    x, r, res = np.zeros(op.N), b, np.dot(b, s)
    for _ in range(2):
        h = A(q)
        alpha = res / np.dot(q, h)
        x, r = x + alpha * q, r - alpha * h
        s = dinv * r
        new = np.dot(r, s)
        q, res = s + new / res * q, new
    inv = fa.InverseOperator(ctx, method=fa.CG, tolerance=1e-30, errormeasure=fa.RELATIVE, maxiterations=2)
    inv.bind(op, fa.Preconditioner(op, fa.PRE_JACOBI))
    X = op.vector(np.zeros(op.N))
    inv(op.vector(b), X)
    # both recurrences round alike, 1e-16 sqrt(N) per dot
    assert np.linalg.norm(X.download() - x) < 1e-11 * np.linalg.norm(x)


@pytest.mark.parametrize("p", [2, 3])
def test_vcycle_on_a_thin_mesh(ctx, p):
    """The residual on the next level's modes by rows.  The element blocks' condition
    is about 10 (801 / 1)^2, so 1e-16 per term becomes 1e-9 of max |z|."""
    n = (801, 1, 1)
    rng = np.random.default_rng(p)
    kappa, r = np.exp(rng.normal(size=801)), rng.normal(size=801 * (p + 1) ** 3)
    ref = mgo.MGOracle(n, p, 10.0 * p * p, ("cell", kappa)).apply(r)
    op = operator(ctx, n, p, (0, 0, 0), 0.0, kappa)
    R, Z = op.vector(r), op.vector()
    Z.fill(np.nan)
    fa.Preconditioner(op, fa.PRE_MULTIGRID)(R, Z)
    print("thin vcycle", p, rel(Z.download(), ref), flush=True)
    assert rel(Z.download(), ref) < 1e-9


def test_direction_of_a_thin_mesh_does_not_matter_for_time(ctx):
    """The same elements in a row along x and along z: the walk along x took
    almost five times as long (46 us and 9.8 us), the rows take 10.6 us."""
    t = []
    for n in ((20000, 1, 1), (1, 1, 20000)):
        op = operator(ctx, n, 3, (0, 0, 0), 0.0, np.ones(20000))
        U, W = op.vector(np.ones(op.N)), op.vector()
        best = np.inf
        for _ in range(10):
            ctx.synchronize()
            t0 = time.perf_counter()
            for _ in range(100):
                op(U, W)
            ctx.synchronize()
            best = min(best, time.perf_counter() - t0)
        t.append(best)
    print("thin", [round(1e4 * v, 1) for v in t], flush=True)
    assert t[0] < 2.5 * t[1]


# meshes whose walks take three steps (the last two) and sixteen (the last
# fifteen), with a remainder of the tile in y and in z
WALKS = [((11, 103, 107), 2), ((11, 81, 85), 3), ((11, 57, 59), 4),
         ((47, 135, 137), 2), ((47, 101, 105), 3), ((47, 71, 75), 4)]


@pytest.mark.parametrize("prec,tol", [(fa.F64, 1e-12), (fa.F32, 2e-5)])
@pytest.mark.parametrize("n,p", WALKS)
def test_long_walks_equal_rows(ctx, n, p, prec, tol):
    """A pointwise reaction of zeros sends the same operator by rows, without a walk:
    the same lines, added in another order."""
    rng = np.random.default_rng(p)
    E = n[0] * n[1] * n[2]
    op = operator(ctx, n, p, (1, -.5, .25), 0.3, np.exp(rng.normal(size=E)), prec)
    u = rng.standard_normal(op.N, dtype=np.float64 if prec == fa.F64 else np.float32)
    U, W = op.vector(u), op.vector()
    W.fill(np.nan)
    op(U, W)
    walk = W.download()
    op.set_reaction_qp(np.zeros((E, (p + 1) ** 3)))
    W.fill(np.nan)
    op(U, W)
    err = rel(walk, W.download())
    print("walk", n, p, prec, err, flush=True)
    assert err < tol


@pytest.mark.parametrize("n,p", WALKS[:3])
def test_residual_of_a_long_walk_equals_rows(ctx, n, p):
    """V-cycles of the same operator, its reaction once as the constant c (the
    residual by a walk on every level above Q1) and once as values at the points
    (the finest residual by rows, the coarser ones by a walk with a reaction per
    element).  Bars as in test_gpu_multigrid.py."""
    rng = np.random.default_rng(p)
    E = n[0] * n[1] * n[2]
    kappa, c = np.exp(rng.normal(size=E)), 7.0
    r = rng.normal(size=E * (p + 1) ** 3)
    for prec in (fa.F64, fa.F32):
        z = []
        for points in (False, True):
            op = operator(ctx, n, p, (0, 0, 0), 0.0 if points else c, kappa, prec)
            if points:
                op.set_reaction_qp(np.full((E, (p + 1) ** 3), c))
            R, Z = op.vector(r), op.vector()
            Z.fill(np.nan)
            fa.Preconditioner(op, fa.PRE_MULTIGRID)(R, Z)
            z.append(Z.download())
        print("residual", n, p, prec, rel(*z), flush=True)
        if prec == fa.F64:
            assert rel(*z) < 1e-12
        else:
            assert np.linalg.norm(z[0] - z[1]) < 1e-4 * np.linalg.norm(z[1])
