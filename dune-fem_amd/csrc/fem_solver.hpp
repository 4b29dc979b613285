// Device-driven Krylov solvers behind the InverseOperator interface.
#pragma once

#include <functional>
#include <memory>

#include "fem_kstate.hpp"
#include "fem_op.hpp"

namespace femamd {

struct Solver {
    Context *ctx = nullptr;
    fem_solver_params prm{};
    Operator *op = nullptr, *iop = nullptr;
    Precond *pre = nullptr, *ipre = nullptr;
    // preconditioners built at bind from fem.solver.preconditioning.method
    // when the caller passes none
    std::unique_ptr<Precond> own_pre, own_ipre;
    std::unique_ptr<Precond> widened;   // an FP32 preconditioner serving the FP64 solve
    DevBuf state, partials, counters;
    KState *hstate = nullptr;   // pinned mirror
    std::vector<DevBuf *> work;
    // CG: called with the device iterate and residual every snap_chunk steps
    std::function<void(const void *x, const void *r)> snapshot;
    int snap_chunk = 0;
    int fallback_used = 0;

    void init(Context *c, const fem_solver_params &p);
    void bind(Operator *o, Precond *p, Operator *io, Precond *ip);
    void unbind();
    void solve(const Vec &b, Vec &x, fem_solver_info &info);
    ~Solver();

    // one Krylov solve in precision of `o` on raw pointers; returns signed iterations
    int krylov(int method, Operator *o, Precond *p, const void *b, void *x, double tol, int criteria, int maxit,
               int restart, int64_t N, int prec);
    void *workbuf(int i, size_t bytes);
    void fetch_state();
    double true_residual(const Vec &b, const Vec &x, Vec &r);
};

}  // namespace femamd

struct fem_solver { femamd::Solver s; femamd::Context *held = nullptr; };
