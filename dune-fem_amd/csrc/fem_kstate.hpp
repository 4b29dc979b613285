// Scalars of one Krylov solve and who may read and write its flags.
//
// A kernel's workgroups start one after another, so a flag that a kernel reads
// at its entry must not be written by that kernel: workgroups, and the
// wavefronts of one workgroup, would take different ways.  Every flag therefore
// has a kernel that finds it out and a later kernel that passes it on, and the
// functions below are what the kernels (fem_solver.hip) call for it.  Host code
// as well as device code, so that the order can be checked without a GPU.
#pragma once

#include <cstddef>

#if defined(__HIPCC__)
#define FEM_HD __host__ __device__ __forceinline__
#else
#define FEM_HD inline
#endif

namespace femamd {

constexpr int GM_MAX = 64;   // maximum GMRES restart length

// scalars of one solve, resident in device memory; kernels read and update
// them so that the iteration loop needs no host round trip per step
struct KState {
    double res, prev, qh, alpha, beta, tol, bnorm2, scale;
    int it, done, maxit, criteria;
    int crit_res;      // stop on ||r||^2 instead of <r, M^-1 r>
    double rr;         // ||r||^2 of the current residual
    // CG: the scalars after the step just reduced, whether no step has been
    // made yet, and whether the step just reduced was the last one
    double n_res, n_rr;
    int n_it, fresh, end;
    // GMRES
    double gtol;
    double gres;     // the cycle's last residual estimate |g[jlast]|
    int jlast;       // inner steps done in the current cycle
    int converged;   // cycle ended by |g| < tol
    int cycle_end;   // the step just scaled was the cycle's last (converged or maxit)
    int cycle_done;  // the same, a kernel later
    // BiCGStab
    double nu, omega, bres;
    int fin;         // the iteration just reduced is the last one
    // GMRES work (from here on never copied to the host)
    double H[(GM_MAX + 1) * GM_MAX];
    double g[GM_MAX + 1], cs[GM_MAX], sn[GM_MAX], y[GM_MAX];
};
// the part of KState that travels between host and device
constexpr size_t KSTATE_HEAD = offsetof(KState, H);

// ---- CG -------------------------------------------------------------------------
// A step is: direction, apply, update, preconditioner.  The direction kernel sums
// <p, s> and <p, p> of the step before and keeps them in n_*, and `end`; the
// kernels after it enter by `end`; the update kernel makes the kept scalars
// current and passes `end` on as `done`, by which the direction kernel and the
// host enter.
FEM_HD bool cg_skip_dir(const KState &st) { return st.done || st.fresh; }
FEM_HD bool cg_skip_step(const KState &st) { return st.end; }

FEM_HD bool cg_stops(const KState &st, double r, double rr)
{
    return !((st.crit_res ? rr : r) > st.tol) || st.it + 1 >= st.maxit;
}

// by one thread of the direction kernel
FEM_HD void cg_keep(KState &st, double r, double rr)
{
    const bool stops = cg_stops(st, r, rr);
    st.n_res = r;
    st.n_rr = rr;
    st.n_it = st.it + 1;
    if (stops) st.end = 1;
}

// by one thread of the update kernel, also where it skips the step
FEM_HD void cg_pass_on(KState &st)
{
    st.res = st.n_res;
    st.rr = st.n_rr;
    st.it = st.n_it;
    st.fresh = 0;
    if (st.end) st.done = 1;
}

// ---- GMRES ----------------------------------------------------------------------
// A step is: preconditioner, apply, multi-dot, orthogonalisation, scaling.  The
// scaling kernel finishes column j and finds out whether the cycle ends; the
// kernels after it enter by `cycle_end`; the orthogonalisation passes it on as
// `cycle_done`, by which the scaling enters.  At the start of a cycle (j < 0) the
// scaling always runs.
FEM_HD bool gm_skip_scale(const KState &st, int j) { return j >= 0 && st.cycle_done; }
FEM_HD bool gm_skip_step(const KState &st) { return st.cycle_end; }

// by one thread of the scaling at the start of a cycle, nrm = ||r||
FEM_HD void gm_begin(KState &st, double nrm)
{
    st.res = nrm;
    st.jlast = 0;
    st.gres = nrm;
    st.converged = nrm <= st.gtol * (1 + 1e-15);
    st.cycle_end = st.cycle_done = st.converged || st.it >= st.maxit;
    if (!st.converged) st.g[0] = -nrm;
}

// by one thread of the scaling, gl = g[j + 1] after the rotation of column j
FEM_HD void gm_keep(KState &st, int j, int m, double gl)
{
    const double e = gl < 0 ? -gl : gl;
    st.gres = e;
    st.it += 1;
    st.jlast = j + 1;
    if (e < st.gtol) st.converged = 1;
    if (st.converged || st.it >= st.maxit || j + 1 == m) st.cycle_end = 1;
}

// by one thread of the orthogonalisation, where it skips the step
FEM_HD void gm_pass_on(KState &st) { st.cycle_done = 1; }

}  // namespace femamd
