"""The calls a user of this library makes, with their real sizes.

A case is one call of a public entry point: an operator apply, a
preconditioner apply, an assembled matrix-vector product, or a whole linear,
Newton or batched solve.  ``listed`` names twelve of them, ``draw`` gives more
of the same ranges.  ``exact`` restates the discretisation (SIPG DG on
hexahedra with the orthonormal Legendre basis, continuous Q2 on quads) in
64-bit torch, without the library.

DoF vectors are torch tensors in device memory that the library views in
place, as a program does that already holds its unknowns on the GPU.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("dune-fem_amd"))

import dunefem_amd as fa  # noqa: E402

DEV = "cuda"
PREC = {"f64": fa.F64, "f32": fa.F32, "bf16": fa.BF16MFMA}


# ---- cases ------------------------------------------------------------------
def listed():
    return [
        # one operator apply on a mesh of a few elements, as in a time step or
        # a unit test of a small model: latency
        {"name": "apply_q2_small", "kind": "apply", "p": 2, "nx": 5, "ny": 4, "nz": 6, "kappa": "cell",
         "adv": False, "dtype": "f64"},
        # the benchmark's headline apply: advection-diffusion, coefficient
        # given at the quadrature points, 16.8 M unknowns
        {"name": "apply_q3_64_qp", "kind": "apply", "p": 3, "nx": 64, "ny": 64, "nz": 64, "kappa": "qp",
         "adv": True, "dtype": "f64"},
        # the same operator in single precision (inner operator of iterative
        # refinement) on a mesh with no round numbers
        {"name": "apply_q3_ragged_qp_f32", "kind": "apply", "p": 3, "nx": 45, "ny": 38, "nz": 51, "kappa": "qp",
         "adv": True, "dtype": "f32"},
        # the largest problem of the benchmark: 110.6 M unknowns, one
        # log-normal coefficient per element
        {"name": "apply_q4_96_cell", "kind": "apply", "p": 4, "nx": 96, "ny": 96, "nz": 96, "kappa": "cell",
         "adv": False, "dtype": "f64"},
        # continuous Q2 in 2D with a pointwise coefficient, ragged mesh
        {"name": "apply2d_qp", "kind": "apply2d", "nx": 517, "ny": 386, "kappa": "qp", "dtype": "f64"},
        # one multigrid V-cycle, the preconditioner step of every Krylov
        # iteration on the high-contrast problem
        {"name": "vcycle_q2_48", "kind": "pre", "pre": "mg", "p": 2, "nx": 48, "ny": 48, "nz": 48, "dtype": "f64"},
        # the recommended solve: FP64 CG, FP32 V-cycle, steps replayed as a
        # graph, Q4
        {"name": "cg_mg32_q4_32", "kind": "solve", "method": "cg", "pre": "mg32", "p": 4, "nx": 32, "ny": 32,
         "nz": 32, "kappa": "cell", "adv": False},
        # the plain solve: CG with the exact element block Jacobi, odd sizes
        {"name": "cg_bj_q2_ragged", "kind": "solve", "method": "cg", "pre": "bj", "p": 2, "nx": 23, "ny": 20,
         "nz": 27, "kappa": "cell", "adv": False},
        # a nonsymmetric solve: upwind advection, pointwise coefficient,
        # restarted GMRES with Jacobi
        {"name": "gmres_q3_adv", "kind": "solve", "method": "gmres", "pre": "jacobi", "p": 3, "nx": 12, "ny": 10,
         "nz": 9, "kappa": "qp", "adv": True},
        # Newton on -div(kappa grad u) + c u^3 = f, a V-cycle built on each
        # Jacobian
        {"name": "newton_q2_24", "kind": "newton", "p": 2, "nx": 24, "ny": 24, "nz": 24},
        # many independent 2D problems of different sizes in one call
        {"name": "batch_24", "kind": "batch", "count": 24, "smin": 32, "smax": 128},
        # the assembled Jacobian: one sparse matrix-vector product
        {"name": "csr_q2", "kind": "csr", "p": 2, "nx": 18, "ny": 16, "nz": 20},
    ]


def _mesh(rng, elements, lo=2):
    """three sides of about `elements` in all, none more than about twice another"""
    s = max(lo, elements ** (1.0 / 3.0))
    return [max(lo, int(round(s * math.exp(rng.uniform(-0.35, 0.35))))) for _ in range(3)]


def draw(rng):
    kind = rng.choices(["apply", "apply2d", "pre", "solve", "newton", "batch", "csr"],
                       [40, 12, 16, 16, 6, 5, 5])[0]
    if kind == "apply":
        p = rng.choice([1, 2, 3, 4])
        kappa = rng.choice(["const", "cell", "qp", "qp"])
        top = 1.2e7 if kappa == "qp" else 4.0e7
        n = _mesh(rng, math.exp(rng.uniform(math.log(2e3), math.log(top))) / (p + 1) ** 3)
        return {"kind": kind, "p": p, "nx": n[0], "ny": n[1], "nz": n[2], "kappa": kappa,
                "adv": rng.random() < 0.5, "dtype": rng.choices(["f64", "f32", "bf16"], [6, 3, 1])[0]}
    if kind == "apply2d":
        s = math.exp(rng.uniform(math.log(16), math.log(1000)))
        return {"kind": kind, "nx": max(4, int(s * rng.uniform(0.7, 1.4))), "ny": max(4, int(s * rng.uniform(0.7, 1.4))),
                "kappa": rng.choice(["const", "qp"]), "dtype": rng.choice(["f64", "f64", "f32"])}
    if kind == "pre":
        p = rng.choice([1, 2, 3, 4])
        pre = rng.choice(["mg", "mg", "bj"])
        n = _mesh(rng, math.exp(rng.uniform(math.log(2e4), math.log(1.5e7))) / (p + 1) ** 3, 4)
        return {"kind": kind, "pre": pre, "p": p, "nx": n[0], "ny": n[1], "nz": n[2], "dtype": rng.choice(["f64", "f32"])}
    if kind == "solve":
        method, pre = rng.choice([("cg", "mg"), ("cg", "mg32"), ("cg", "mg32"), ("cg", "bj"), ("fgmres", "mg"),
                                  ("gmres", "jacobi")])
        p = rng.choice([1, 2, 3, 4])
        adv = method == "gmres"
        top = 2.5e5 if pre == "bj" else 5e4 if adv else 3e6
        n = _mesh(rng, math.exp(rng.uniform(math.log(1e4), math.log(top))) / (p + 1) ** 3, 4)
        return {"kind": kind, "method": method, "pre": pre, "p": p, "nx": n[0], "ny": n[1], "nz": n[2],
                "kappa": "qp" if adv else "cell", "adv": adv}
    if kind == "newton":
        p = rng.choice([1, 2, 3])
        n = _mesh(rng, math.exp(rng.uniform(math.log(1e4), math.log(3.5e5))) / (p + 1) ** 3, 4)
        return {"kind": kind, "p": p, "nx": n[0], "ny": n[1], "nz": n[2]}
    if kind == "batch":
        return {"kind": kind, "count": rng.randint(4, 24), "smin": rng.randint(20, 40), "smax": rng.randint(60, 120)}
    p = rng.choice([1, 2, 3])
    n = _mesh(rng, math.exp(rng.uniform(math.log(5e3), math.log(1.5e5))) / (p + 1) ** 3, 3)
    return {"kind": "csr", "p": p, "nx": n[0], "ny": n[1], "nz": n[2]}


# ---- inputs -----------------------------------------------------------------
_CTX = []


def _ctx():
    if not _CTX:
        _CTX.append(fa.Context(0))
    return _CTX[0]


def _gauss(m):
    x, w = np.polynomial.legendre.leggauss(m)
    return 0.5 * (x + 1.0), 0.5 * w


def _points(n, m):
    return ((np.arange(n)[:, None] + _gauss(m)[0][None, :]) / n).ravel()


class _Sines:
    """sum_m a_m prod_d sin(k_md pi x_d + s_md): a smooth random field"""

    def __init__(self, seed, dim, modes=12, kmax=4, sigma=1.0):
        r = np.random.default_rng(seed)
        self.k = r.integers(1, kmax + 1, size=(modes, dim))
        self.s = r.uniform(0.0, np.pi, size=(modes, dim))
        self.a = r.normal(0.0, sigma / math.sqrt(modes), size=modes) * math.sqrt(2.0) ** dim

    def grid(self, *coords):
        """on the tensor grid of the coordinate lists, indexed [.., y, x]"""
        T = [torch.from_numpy(np.sin(np.pi * self.k[:, d:d + 1] * c[None, :] + self.s[:, d:d + 1])).to(DEV)
             for d, c in enumerate(coords)]
        T[0] = T[0] * torch.from_numpy(self.a).to(DEV)[:, None]
        if len(coords) == 2:
            return T[1].t().contiguous() @ T[0]
        M = T[0].shape[0]
        zy = (T[2][:, :, None] * T[1][:, None, :]).reshape(M, -1)
        return (zy.t().contiguous() @ T[0]).reshape(len(coords[2]), len(coords[1]), len(coords[0]))


def _n3(c):
    return c["nx"], c["ny"], c["nz"]


def _vol3(G, n, m):
    nx, ny, nz = n
    return G.reshape(nz, m, ny, m, nx, m).permute(0, 2, 4, 1, 3, 5).reshape(nx * ny * nz, m ** 3)


def _faces3(fn, n, m):
    """fn on the points of the faces normal to x, y and z: [faces][m^2]"""
    nx, ny, nz = n
    q = [_points(k, m) for k in n]
    f = [np.arange(k + 1) / k for k in n]
    return [fn(f[0], q[1], q[2]).reshape(nz, m, ny, m, nx + 1).permute(0, 2, 4, 1, 3).reshape(-1, m * m),
            fn(q[0], f[1], q[2]).reshape(nz, m, ny + 1, nx, m).permute(0, 2, 3, 1, 4).reshape(-1, m * m),
            fn(q[0], q[1], f[2]).reshape(nz + 1, ny, m, nx, m).permute(0, 1, 3, 2, 4).reshape(-1, m * m)]


def _kappa(c, seed):
    """the coefficient data of a case, on the GPU in 64 bits: ("const", v),
    ("cell", [E]) or ("qp", [E][m^3], three face arrays)"""
    n, m = _n3(c), c["p"] + 1
    kind = c.get("kappa", "cell")
    if kind == "const":
        return ("const", 0.5 + (seed % 97) / 97.0)
    if kind == "cell":
        # log-normal, correlated over a few elements, sigma 1.2
        g = _Sines(seed, 3, modes=24, kmax=9, sigma=1.2)
        return ("cell", torch.exp(g.grid(*[(np.arange(k) + 0.5) / k for k in n])).reshape(-1))
    g = _Sines(seed, 3, modes=16, kmax=4, sigma=0.6)

    def kap(x, y, z):
        return torch.clip(torch.exp(g.grid(x, y, z)), 0.1, 10.0)

    return ("qp", _vol3(kap(*[_points(k, m) for k in n]), n, m).contiguous(), [f.contiguous() for f in _faces3(kap, n, m)])


def _beta(c):
    return 10.0 * c["p"] ** 2


def _b(c):
    return (1.0, 0.5, 0.25) if c.get("adv") else (0.0, 0.0, 0.0)


def _operator(c, kap, prec):
    mode = {"const": fa.KAPPA_CONST, "cell": fa.KAPPA_CELL, "qp": fa.KAPPA_QP}[kap[0]]
    op = fa.GalerkinOperator(_ctx(), fa.OP_DG_SIPG_3D, _n3(c), c["p"], _beta(c), _b(c), 0.0, mode,
                             kap[1] if kap[0] == "const" else 1.0, precision=prec)
    if kap[0] == "cell":
        op.set_kappa_cell(kap[1].cpu().numpy())
    elif kap[0] == "qp":
        op.set_kappa_qp(kap[1].cpu().numpy(), [f.cpu().numpy() for f in kap[2]])
    return op


def _view(t):
    """the library's vector on a torch tensor's memory"""
    return fa.DofVector(_ctx(), t.numel(), fa.F64 if t.dtype == torch.float64 else fa.F32, device_ptr=t.data_ptr())


def _normal(n, seed, dtype):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000003 * seed + 17)
    return torch.randn(n, generator=g, device=DEV, dtype=torch.float64 if dtype == "f64" else torch.float32)


def _source(c, seed):
    """the source term at the volume points, a smooth random field"""
    n, m = _n3(c), c["p"] + 1
    return _vol3(_Sines(seed + 5, 3, modes=16, kmax=4).grid(*[_points(k, m) for k in n]), n, m).contiguous()


def _newton_coefficient(c):
    return 1.0e3


def _batch_inputs(c, seed):
    """per instance: side lengths, log-normal coefficient and source at the points"""
    r, sides = np.random.default_rng(seed), np.random.default_rng(c["count"] + 100 * c["smax"])
    out = []
    for _ in range(c["count"]):
        nx, ny = (int(v) for v in sides.integers(c["smin"], c["smax"] + 1, size=2))
        q = _points(nx, 3), _points(ny, 3)
        s = int(r.integers(1 << 30))

        def lay(G):
            return G.reshape(ny, 3, nx, 3).permute(0, 2, 1, 3).reshape(nx * ny, 9)

        out.append((nx, ny, lay(torch.exp(_Sines(s, 2, modes=16, kmax=8).grid(*q))), lay(_Sines(s + 1, 2, modes=8).grid(*q))))
    return out


def _apply2d_inputs(c, seed):
    n = c["nx"], c["ny"]
    N = (2 * n[0] + 1) * (2 * n[1] + 1)
    kq = None
    if c["kappa"] == "qp":
        G = torch.exp(_Sines(seed, 2, modes=16, kmax=8).grid(_points(n[0], 3), _points(n[1], 3)))
        kq = G.reshape(n[1], 3, n[0], 3).permute(0, 2, 1, 3).reshape(n[0] * n[1], 9).contiguous()
    return n, kq, _normal(N, seed, c["dtype"])


def prepare(case, seed):
    c, ctx, kind = case, _ctx(), case["kind"]
    st = {"kind": kind}
    if kind == "apply2d":
        n, kq, u = _apply2d_inputs(c, seed)
        op = fa.GalerkinOperator(ctx, fa.OP_CG_Q2_2D, n, 2, c=1.0, kappa_mode=fa.KAPPA_CONST if kq is None else fa.KAPPA_QP,
                                 precision=PREC[c["dtype"]])
        if kq is not None:
            op.set_kappa_qp(kq.cpu().numpy())
        st.update(call=op, src=u, out=torch.empty_like(u))
    elif kind == "batch":
        insts = _batch_inputs(c, seed)
        B = fa.Batch(ctx, [(i[0], i[1]) for i in insts])
        B.set_kappa_qp(torch.cat([i[2] for i in insts]).cpu().numpy())
        F = B.rhs(torch.cat([i[3] for i in insts]).cpu().numpy())
        x = torch.zeros(int(B.N), device=DEV, dtype=torch.float64)
        st.update(batch=B, F=F, out=x)
    else:
        dt = c.get("dtype", "f64")
        kap = _kappa(c, seed)
        op = _operator(c, kap, PREC[dt])
        vd = "f64" if dt == "f64" else "f32"
        if kind == "apply":
            u = _normal(op.N, seed, vd)
            st.update(call=op, src=u, out=torch.empty_like(u))
        elif kind == "csr":
            u = _normal(op.N, seed, vd)
            st.update(call=fa.SparseRowMatrix(op), src=u, out=torch.empty_like(u))
        elif kind == "pre":
            u = _normal(op.N, seed, vd)
            pre = fa.Preconditioner(op, fa.PRE_MULTIGRID if c["pre"] == "mg" else fa.PRE_BLOCK_JACOBI)
            st.update(call=pre, op=op, src=u, out=torch.empty_like(u))
        elif kind == "solve":
            F = op.rhs(_source(c, seed).cpu().numpy())
            pop = _operator(c, kap, fa.F32) if c["pre"] == "mg32" else op
            pre = fa.Preconditioner(pop, {"mg": fa.PRE_MULTIGRID, "mg32": fa.PRE_MULTIGRID, "bj": fa.PRE_BLOCK_JACOBI,
                                          "jacobi": fa.PRE_JACOBI}[c["pre"]])
            inv = fa.InverseOperator(ctx, method={"cg": fa.CG, "gmres": fa.GMRES, "fgmres": fa.FGMRES}[c["method"]],
                                     tolerance=1e-11, errormeasure=fa.RELATIVE, maxiterations=20000, restart=30,
                                     graph=1 if c["method"] == "cg" and c["pre"] != "bj" else 0)
            inv.bind(op, pre)
            st.update(inv=inv, F=F, op=op, out=torch.zeros(op.N, device=DEV, dtype=torch.float64))
        else:
            op.set_reaction_law(_newton_coefficient(c), 2)
            F = op.rhs(20.0 * _source(c, seed).cpu().numpy())
            fn = math.sqrt(F.normSquaredDofs())
            inv = fa.NewtonInverseOperator(ctx, {"nonlinear.tolerance": 1e-10 * fn},
                                           linear=dict(method=fa.CG, tolerance=1e-7, errormeasure=fa.REDUCTION,
                                                       maxiterations=20000, preconditioning=fa.PRE_MULTIGRID))
            inv.bind(op)
            st.update(inv=inv, F=F, op=op, out=torch.zeros(op.N, device=DEV, dtype=torch.float64))
    if "src" in st:
        st["u"] = _view(st["src"])
    st["w"] = _view(st["out"])
    ctx.synchronize()
    torch.cuda.synchronize()
    return st


def run(state):
    w = state["w"]
    if "call" in state:
        state["call"](state["u"], w)
    else:
        w.clear()
        if "batch" in state:
            state["batch"].solve(state["F"], w, tol=1e-11)
        else:
            state["inv"](state["F"], w)
    return state["out"]


# ---- work -------------------------------------------------------------------
def _coefficients(c):
    """coefficient values an apply of the case needs"""
    n, m = _n3(c), c["p"] + 1
    E = n[0] * n[1] * n[2]
    if c.get("kappa", "cell") == "const":
        return 0
    if c.get("kappa", "cell") == "cell":
        return E
    return E * m ** 3 + sum((n[0] + (d == 0)) * (n[1] + (d == 1)) * (n[2] + (d == 2)) for d in range(3)) * m * m


def work(case):
    """Bytes: inputs read and outputs written once per operator use.  Iterative
    calls count a nominal number of steps of their kind, each with one operator
    use and the vectors of the recurrence.  Flops: the multiplications and
    additions of sum-factorised contractions."""
    c, kind = case, case["kind"]
    if kind == "apply2d":
        E, N = c["nx"] * c["ny"], (2 * c["nx"] + 1) * (2 * c["ny"] + 1)
        s = 8 if c["dtype"] == "f64" else 4
        return {"bytes": s * (2 * N + (9 * E if c["kappa"] == "qp" else 0)), "flops": 300 * E}
    if kind == "batch":
        side = 0.5 * (c["smin"] + c["smax"])
        N = c["count"] * (2 * side + 1) ** 2
        steps = 2000
        return {"bytes": steps * (4 * 8 * N + 4 * 9 * N / 4), "flops": steps * 90 * N}
    n, k = _n3(c), c["p"] + 1
    E = n[0] * n[1] * n[2]
    N = E * k ** 3
    s = 4 if c.get("dtype", "f64") != "f64" else 8
    if kind == "csr":
        nnz = (7 * E - 2 * (n[0] * n[1] + n[1] * n[2] + n[0] * n[2])) * k ** 6
        return {"bytes": 12 * nnz + 24 * N, "flops": 2 * nnz}
    apply_b, apply_f = s * (2 * N + _coefficients(c)), (12 * k if c.get("kappa", "cell") != "qp" else 30 * k) * N
    if kind == "apply":
        return {"bytes": apply_b, "flops": apply_f}
    if kind == "pre":
        if c["pre"] == "bj":
            return {"bytes": s * (2 * N + E), "flops": 12 * k * N}
        # the V-cycle: five operator uses on the fine level, a fixed share more on the coarser ones
        return {"bytes": 6 * apply_b, "flops": 6 * apply_f}
    if kind == "newton":
        return {"bytes": 60 * (7 * apply_b + 8 * 9 * N), "flops": 60 * 7 * apply_f}
    steps, uses, vecs = {"mg": (30, 7, 9), "mg32": (30, 4, 9), "bj": (400, 2, 9), "jacobi": (400, 1, 32)}[c["pre"]]
    return {"bytes": steps * (uses * apply_b + 8 * vecs * N), "flops": steps * uses * apply_f}


# ---- the same numbers from plain 64-bit torch ---------------------------------
def _along(M, T, axis):
    """contraction of axis `axis` of T with the columns of M"""
    return torch.tensordot(T, M, dims=([axis], [1])).movedim(-1, axis)


class _Sipg:
    """The SIPG form on an nx x ny x nz mesh of the unit cube: tensors indexed
    [z, y, x, mode or point x, y, z]; the element axis of direction d is 2 - d,
    its mode axis 3 + d."""

    def __init__(self, c, kap):
        self.n, self.K = _n3(c), c["p"] + 1
        n, K = self.n, self.K
        self.beta, self.b = _beta(c), _b(c)
        x, w = _gauss(K)
        leg = [np.polynomial.legendre.Legendre.basis(a, domain=[0, 1]) * math.sqrt(2 * a + 1) for a in range(K)]

        def table(pts, d):
            return torch.from_numpy(np.array([[(f.deriv() if d else f)(t) for f in leg] for t in pts])).to(DEV)

        self.B, self.Bd = table(x, 0), table(x, 1)
        self.P, self.dP = table([0.0, 1.0], 0), table([0.0, 1.0], 1)
        w = torch.from_numpy(w).to(DEV)
        self.w3, self.w2 = w[:, None, None] * w[:, None] * w, w[:, None] * w
        self.h = [1.0 / v for v in n]
        sh = (n[2], n[1], n[0])
        one = torch.ones(1, device=DEV, dtype=torch.float64)
        if kap[0] == "qp":
            self.kv = kap[1].reshape(*sh, K, K, K).permute(0, 1, 2, 5, 4, 3)
            # the face arrays hold one layer more in their direction, points [q2][q1]
            self.kf = [kap[2][d].reshape([v + (a == 2 - d) for a, v in enumerate(sh)] + [K, K]).transpose(-1, -2)
                       for d in range(3)]
            self.cell = None
        else:
            self.cell = (kap[1] if kap[0] == "cell" else one.expand(n[0] * n[1] * n[2]) * kap[1]).reshape(*sh, 1, 1, 1)
            self.kv, self.kf = self.cell, None
        self.cvol = None

    def points(self, U):
        for d in range(3):
            U = _along(self.B, U, 3 + d)
        return U

    def test(self, R):
        for d in range(3):
            R = _along(self.B.t(), R, 3 + d)
        return R

    def vector(self, u):
        K = self.K
        return u.to(torch.float64).reshape(self.n[2], self.n[1], self.n[0], K, K, K)

    def load(self, fq):
        K = self.K
        f = fq.reshape(self.n[2], self.n[1], self.n[0], K, K, K).permute(0, 1, 2, 5, 4, 3)
        return self.test(f * self.w3 * (self.h[0] * self.h[1] * self.h[2]))

    def __call__(self, U):
        h, vol = self.h, self.h[0] * self.h[1] * self.h[2]
        out = torch.zeros_like(U)
        uq = self.points(U)
        for d in range(3):
            g = U
            for e in range(3):
                g = _along(self.Bd if e == d else self.B, g, 3 + e)
            f = (self.kv * g / h[d] - self.b[d] * uq) * self.w3 * (vol / h[d])
            for e in range(3):
                f = _along((self.Bd if e == d else self.B).t(), f, 3 + e)
            out += f
            del g, f
        if self.cvol is not None:
            out += self.test(self.cvol * uq * self.w3 * vol)
        del uq
        for d in range(3):
            self._faces(U, d, out)
        return out

    def _faces(self, U, d, out):
        h, ax = self.h[d], 2 - d
        oth = [e for e in range(3) if e != d]
        T = U
        for e in oth:
            T = _along(self.B, T, 3 + e)
        val = [torch.tensordot(T, self.P[s], dims=([3 + d], [0])) for s in (0, 1)]
        der = [torch.tensordot(T, self.dP[s], dims=([3 + d], [0])) / h for s in (0, 1)]
        del T
        W = self.w2 * (self.h[oth[0]] * self.h[oth[1]])
        pen, bd, n = self.beta / h, self.b[d], U.shape[ax]

        def cut(t, lo, cnt):
            return t.narrow(ax, lo, cnt)

        c0 = [torch.zeros_like(val[0]) for _ in (0, 1)]
        c1 = [torch.zeros_like(val[0]) for _ in (0, 1)]
        if n > 1:
            ul, ur, gl, gr = cut(val[1], 0, n - 1), cut(val[0], 1, n - 1), cut(der[1], 0, n - 1), cut(der[0], 1, n - 1)
            if self.cell is not None:
                kc = self.cell.squeeze(-1)
                kl, kr = cut(kc, 0, n - 1), cut(kc, 1, n - 1)
                kp = 0.5 * (kl + kr)
            else:
                kl = kr = kp = cut(self.kf[d], 1, n - 1)
            jump = ul - ur
            flux = W * (kp * pen * jump - 0.5 * (kl * gl + kr * gr) + max(bd, 0.0) * ul - max(-bd, 0.0) * ur)
            cut(c0[1], 0, n - 1).copy_(flux)
            cut(c0[0], 1, n - 1).copy_(-flux)
            cut(c1[1], 0, n - 1).copy_(-0.5 * W * kl * jump)
            cut(c1[0], 1, n - 1).copy_(-0.5 * W * kr * jump)
        for s in (0, 1):
            at, nrm = (n - 1 if s else 0), (1.0 if s else -1.0)
            k = cut(self.cell.squeeze(-1), at, 1) if self.cell is not None else cut(self.kf[d], n if s else 0, 1)
            u, g = cut(val[s], at, 1), cut(der[s], at, 1) * nrm
            cut(c0[s], at, 1).copy_(W * ((k * pen + max(bd * nrm, 0.0)) * u - k * g))
            cut(c1[s], at, 1).copy_(-W * k * u * nrm)
        for s in (0, 1):
            lift = c0[s].unsqueeze(3 + d) * _shape(self.P[s], 3 + d) + c1[s].unsqueeze(3 + d) * _shape(self.dP[s] / h, 3 + d)
            for e in oth:
                lift = _along(self.B.t(), lift, 3 + e)
            out += lift

    def blocks(self):
        """element blocks by applying the form to one mode of every eighth
        element (parity colours), as a dense batch"""
        K3 = self.K ** 3
        sh = (self.n[2], self.n[1], self.n[0])
        z, y, x = (torch.arange(v, device=DEV) % 2 for v in sh)
        col = (z[:, None, None] * 4 + y[None, :, None] * 2 + x).reshape(-1)
        E = col.numel()
        out = torch.empty(E, K3, K3, device=DEV, dtype=torch.float64)
        for k in range(8):
            at = col == k
            for j in range(K3):
                u = torch.zeros(E, K3, device=DEV, dtype=torch.float64)
                u[at, j] = 1.0
                out[at, :, j] = self(self.vector(u)).reshape(E, K3)[at]
        return out


def _shape(v, axis):
    s = [1] * 6
    s[axis] = v.numel()
    return v.reshape(s)


def _pcg(A, b, Minv, tol=1e-14, most=4000):
    x, r = torch.zeros_like(b), b.clone()
    z = Minv(r)
    p, rz, stop = z.clone(), torch.sum(r * z), tol * float(b.norm())
    for k in range(most):
        q = A(p)
        a = rz / torch.sum(p * q)
        x += a * p
        r -= a * q
        if k % 10 == 9 and float(r.norm()) <= stop:
            break
        z = Minv(r)
        new = torch.sum(r * z)
        p = z + (new / rz) * p
        rz = new
    return x


def _bicgstab(A, b, Minv, tol=1e-14, most=4000):
    x, r = torch.zeros_like(b), b.clone()
    rs, p, rho, stop = r.clone(), r.clone(), torch.sum(r * r), tol * float(b.norm())
    for k in range(most):
        y = Minv(p)
        v = A(y)
        a = rho / torch.sum(rs * v)
        s = r - a * v
        z = Minv(s)
        t = A(z)
        om = torch.sum(t * s) / torch.sum(t * t)
        x += a * y + om * z
        r = s - om * t
        if k % 10 == 9 and float(r.norm()) <= stop:
            break
        new = torch.sum(rs * r)
        p = r + (new / rho) * (a / om) * (p - om * v)
        rho = new
    return x


class _Lagrange2d:
    """Continuous Q2 on nx x ny quads, or on several independent meshes with
    their nodes one after another: node lattices [2 ny + 1][2 nx + 1], local
    index 3 iy + ix, rows of the boundary nodes the identity."""

    def __init__(self, meshes, c):
        idx, mats, edge, off = [], [], [], 0
        for n, kq in meshes:
            nx, ny = n
            lat = torch.arange((2 * nx + 1) * (2 * ny + 1), device=DEV).reshape(2 * ny + 1, 2 * nx + 1) + off
            idx.append(lat.unfold(0, 3, 2).unfold(1, 3, 2).reshape(-1, 9))
            K = _lagrange2d_matrices(n, kq, c)
            mats.append(K if K.dim() == 3 else K.expand(nx * ny, 9, 9))
            m = torch.ones_like(lat, dtype=torch.bool)
            m[1:-1, 1:-1] = False
            edge.append(m.reshape(-1))
            off += lat.numel()
        self.idx, self.K, self.edge, self.N = torch.cat(idx), torch.cat(mats), torch.cat(edge), off

    def _sum(self, el):
        return torch.zeros(self.N, device=DEV, dtype=torch.float64).index_add_(0, self.idx.reshape(-1), el.reshape(-1))

    def __call__(self, u):
        return torch.where(self.edge, u, self._sum(torch.matmul(self.K, u[self.idx].unsqueeze(2))))

    def diagonal(self):
        return torch.where(self.edge, 1.0, self._sum(torch.diagonal(self.K, dim1=1, dim2=2)))

    def load(self, meshes, sources):
        L, _, W = _lagrange2d_tables()
        phi = torch.from_numpy(np.einsum("qj,pi->qpji", L, L).reshape(9, 9) * W[:, None]).to(DEV)
        el = torch.cat([torch.matmul(f, phi) / (n[0] * n[1]) for (n, _), f in zip(meshes, sources)])
        return torch.where(self.edge, 0.0, self._sum(el))


def _lagrange2d_tables():
    x, w = _gauss(3)
    L = np.array([[(1 - t) * (1 - 2 * t), 4 * t * (1 - t), t * (2 * t - 1)] for t in x])
    D = np.array([[4 * t - 3, 4 - 8 * t, 4 * t - 1] for t in x])
    W = np.outer(w, w).ravel()                            # [qy qx]
    return L, D, W


def _lagrange2d_matrices(n, kq, c):
    """element matrices [E][9][9], local index 3 iy + ix"""
    L, D, W = _lagrange2d_tables()
    phi, gx, gy = (np.einsum("qj,pi->qpji", a, b).reshape(9, 9) for a, b in ((L, L), (L, D), (D, L)))
    S = (np.einsum("qi,qj->qij", gx, gx) * n[0] / n[1] + np.einsum("qi,qj->qij", gy, gy) * n[1] / n[0]) * W[:, None, None]
    M = np.einsum("q,qi,qj->ij", W, phi, phi) / (n[0] * n[1])
    S, M = torch.from_numpy(S).to(DEV), torch.from_numpy(M).to(DEV)
    if kq is None:
        return S.sum(0) + c * M
    return torch.matmul(kq, S.reshape(9, 81)).reshape(-1, 9, 9) + c * M


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "apply2d":
        n, kq, u = _apply2d_inputs(c, seed)
        return _Lagrange2d([(n, kq)], 1.0)(u.to(torch.float64))
    if kind == "batch":
        insts = _batch_inputs(c, seed)
        meshes = [(i[:2], i[2]) for i in insts]
        A = _Lagrange2d(meshes, 0.0)
        d = A.diagonal()
        return _pcg(A, A.load(meshes, [i[3] for i in insts]), lambda v: v / d, most=20000)
    A = _Sipg(c, _kappa(c, seed))
    K3 = A.K ** 3
    N = A.n[0] * A.n[1] * A.n[2] * K3
    if kind in ("apply", "csr"):
        return A(A.vector(_normal(N, seed, "f64" if c.get("dtype", "f64") == "f64" else "f32"))).reshape(-1)
    if kind == "pre":
        if c["pre"] == "mg" or N * K3 > 4e8:
            return None                     # a V-cycle is defined by its own hierarchy
        u = _normal(N, seed, c["dtype"]).to(torch.float64).reshape(-1, K3, 1)
        return torch.linalg.solve(A.blocks(), u).reshape(-1)
    if N * K3 > 4e7 or N > 4e5:
        return None                         # too long

    def inverse():
        inv = torch.linalg.inv(A.blocks())
        return lambda r: torch.matmul(inv, r.reshape(-1, K3, 1)).reshape(r.shape)

    if kind == "solve":
        F = A.load(_source(c, seed))
        return (_bicgstab if c["adv"] else _pcg)(A, F, inverse()).reshape(-1)
    F = A.load(20.0 * _source(c, seed))
    c3, u = _newton_coefficient(c), torch.zeros_like(F)
    for _ in range(40):
        uq = A.points(u)
        A.cvol = c3 * uq * uq
        R = A(u) - F
        if float(R.norm()) <= 1e-13 * float(F.norm()):
            break
        A.cvol = 3.0 * A.cvol
        u = u - _pcg(A, R, inverse(), tol=1e-6)
    return u.reshape(-1)
