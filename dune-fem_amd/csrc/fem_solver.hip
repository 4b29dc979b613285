// Device-driven Krylov solvers.
//
//   CG     LinearSolver::cg (dune/fem/solver/linear/cg.hh:19-117): the same
//          recurrence (r = Ax - b, p = b - Ax, q = M^-1 p, ...), the same
//          stopping rule on <p, M^-1 p> against eps^2 * (1 | ||b||^2 | r0)
//          and the signed iteration count.
//   GMRES  LinearSolver::gmres (dune/fem/solver/linear/gmres.hh:117-299):
//          restarted, right preconditioned, classical Gram-Schmidt, Givens
//          rotations, M^-1 applied once to V y at the end of a cycle.
//   FGMRES flexible variant storing z_j = M^-1 v_j (no in-tree counterpart;
//          dune-istl's RestartedFlexibleGMResSolver is reached through
//          dune/fem/solver/istlinverseoperators.hh:176-178).
//
// All scalars (alpha, beta, Hessenberg matrix, rotations) live in device
// memory, so a Krylov step needs no host round trip.  CG and GMRES leave a
// reduction's partials to the kernel that needs the sum, whose first workgroup
// keeps the scalars; BiCGStab has the last block of a reduction update them.
// Every kernel reads a device flag of the end and returns at once when the
// solve has finished; the host launches steps in batches and reads the state
// back once per batch (CG, BiCGStab) or once per restart cycle (GMRES).
#include <chrono>
#include <cmath>
#include <cstdio>

#include "fem_blas.hpp"
#include "fem_learned.hpp"
#include "fem_solver.hpp"

namespace femamd {

constexpr int GRP = 8;   // vectors per register group in the multi-dot
// partials that every workgroup of the next kernel sums in CG at most, and
// what more are brought down to
constexpr int CG_PARTS = 4096, CG_FEWER = 256;
// partials of a square sum at most (after the multi-dot's in the workspace)
constexpr int NORM_PARTS = 1024;

// Reductions of CG and GMRES: a reduction leaves one partial per workgroup,
// and the kernel that needs the result sums the partials itself, each
// workgroup all of them in the same order.  A kernel boundary orders the two,
// where a finish by the last workgroup to arrive waits for a chain of atomics
// (69 k DoFs, restart 30: multi-dot 37 us and orthogonalisation 15 us with
// that finish on 512 workgroups, 7.6 and 7.4 us so).  The grids grow with the
// vector, so that few partials are left where the sums are short.

// the sum of n partials, in every thread, for every workgroup alike: thread t
// takes t, t + 256, ..., then a tree over the workgroup
__device__ __forceinline__ double sum_parts(const double *__restrict__ part, int n, double *lds)
{
    double v = 0;
#pragma unroll 4
    for (int k = threadIdx.x; k < n; k += RED_THREADS) v += part[k];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0;
#pragma unroll
    for (int w = 0; w < RED_THREADS / 64; ++w) s += lds[w];
    return s;
}

// ---- CG kernels ---------------------------------------------------------------
template <typename T>
__global__ void k_cg_setup(const T *__restrict__ b, const T *__restrict__ h, T *__restrict__ r, T *__restrict__ p,
                           int64_t n)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const T hb = h[i], bb = b[i];
        r[i] = hb - bb;
        p[i] = bb - hb;
    }
}

__global__ void k_cg_init(KState *st, double eps, int criteria, int maxit, int crit_res)
{
    const double r0 = crit_res ? st->rr : st->res;
    const double ref = criteria == FEM_ERRMEASURE_RELATIVE ? st->bnorm2 : criteria == FEM_ERRMEASURE_REDUCTION ? r0 : 1.0;
    st->tol = eps * eps * ref;
    st->it = 0;
    st->maxit = maxit;
    st->crit_res = crit_res;
    st->done = st->end = !(r0 > st->tol) || maxit <= 0;
    st->fresh = 1;
    st->n_res = st->res;
    st->n_rr = st->rr;
    st->n_it = 0;
}

// A CG step is: direction (k_cg_dir), apply with the partials of <q, h>,
// update (k_cg_update), preconditioner with the partials of <p, s> and
// <p, p>.  The direction kernel sums the latter, forms beta and the stopping
// test, and its first workgroup keeps the new scalars; the update kernel sums
// <q, h>, forms alpha and makes them current.  No kernel reads what one of its
// own workgroups writes (fem_kstate.hpp has the flags).

// two sums at once, of part[0..n) and part[n..2n)
__device__ __forceinline__ void sum_parts2(const double *__restrict__ part, int n, double *lds, double &s0, double &s1)
{
    double v = 0, u = 0;
#pragma unroll 4
    for (int k = threadIdx.x; k < n; k += RED_THREADS) {
        v += part[k];
        u += part[n + k];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        v += __shfl_xor(v, off, 64);
        u += __shfl_xor(u, off, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        lds[threadIdx.x >> 6] = v;
        lds[RED_THREADS / 64 + (threadIdx.x >> 6)] = u;
    }
    __syncthreads();
    s0 = s1 = 0;
#pragma unroll
    for (int w = 0; w < RED_THREADS / 64; ++w) {
        s0 += lds[w];
        s1 += lds[RED_THREADS / 64 + w];
    }
}

// the same test after the last step of a batch, for the host to read, by one
// workgroup (the next direction kernel repeats it if the solve goes on)
__global__ void __launch_bounds__(RED_THREADS) k_cg_check(KState *st, const double *__restrict__ pp, int np)
{
    if (cg_skip_dir(*st)) return;
    __shared__ double lds[2 * (RED_THREADS / 64)];
    double r, rr;
    sum_parts2(pp, np, lds, r, rr);   // (its barrier: every wavefront has entered)
    if (threadIdx.x == 0) {
        cg_keep(*st, r, rr);
        if (st->end) cg_pass_on(*st);
    }
}

// q = beta q + sg a: a = s, sg = 1 (TA = float: the result of an FP32
// preconditioner as it is), without a preconditioner a = r, sg = -1
template <typename T, typename TA>
__global__ void __launch_bounds__(RED_THREADS)
    k_cg_dir(T *__restrict__ q, const TA *__restrict__ a, double sg, int64_t n, KState *st,
             const double *__restrict__ pp, int np)
{
    if (cg_skip_dir(*st)) return;
    __shared__ double lds[2 * (RED_THREADS / 64)];
    double r, rr;
    sum_parts2(pp, np, lds, r, rr);
    if (blockIdx.x == 0 && threadIdx.x == 0) cg_keep(*st, r, rr);
    if (cg_stops(*st, r, rr)) return;
    const double beta = r / st->res;
    const int64_t stride = (int64_t)gridDim.x * RED_THREADS;
    int64_t i = blockIdx.x * (int64_t)RED_THREADS + threadIdx.x;
    // four independent elements in flight per thread
    for (; i + 3 * stride < n; i += 4 * stride) {
        T vq[4];
        TA va[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            vq[k] = q[i + k * stride];
            va[k] = a[i + k * stride];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) q[i + k * stride] = (T)(beta * (double)vq[k] + sg * (double)va[k]);
    }
    for (; i < n; i += stride) q[i] = (T)(beta * (double)q[i] + sg * (double)a[i]);
}

// MODE 0: x += a q, p -= a h (a general preconditioner follows; p32, may be
//         null: p rounded for an FP32 preconditioner)
// MODE 1: the same, s = dinv p and the partials of <p, s>, <p, p> (Jacobi)
// MODE 2: x += a q, r += a h and the partials of <r, r>, twice (no
//         preconditioner; p is r here)
template <typename T, int MODE>
__global__ void __launch_bounds__(RED_THREADS)
    k_cg_update(T *__restrict__ x, T *__restrict__ p, const T *__restrict__ q, const T *__restrict__ h,
                T *__restrict__ s, const T *__restrict__ dinv, int64_t n, KState *st, const double *__restrict__ qp,
                int nq, double *__restrict__ pp, float *__restrict__ p32)
{
    const bool keeper = blockIdx.x == 0 && threadIdx.x == 0;
    if (cg_skip_step(*st)) {
        if (keeper) cg_pass_on(*st);
        return;
    }
    __shared__ double lds[RED_THREADS / 64];
    const double qh = sum_parts(qp, nq, lds);
    const double alpha = st->n_res / qh;
    if (keeper) {
        st->qh = qh;
        st->alpha = alpha;
        cg_pass_on(*st);
    }
    double acc = 0, acc2 = 0;
    auto one = [&](int64_t i, T xv, T pv, T qv, T hv, T dv) {
        x[i] = (T)((double)xv + alpha * (double)qv);
        const T pn = (T)((double)pv + (MODE == 2 ? alpha : -alpha) * (double)hv);
        p[i] = pn;
        if (MODE == 0 && p32) p32[i] = (float)pn;
        if (MODE == 1) {
            const T sv = dv * pn;
            s[i] = sv;
            acc += (double)pn * (double)sv;
        }
        if (MODE != 0) acc2 += (double)pn * (double)pn;
    };
    const int64_t stride = (int64_t)gridDim.x * RED_THREADS;
    int64_t i = blockIdx.x * (int64_t)RED_THREADS + threadIdx.x;
    for (; i + 3 * stride < n; i += 4 * stride) {
        T xv[4], pv[4], qv[4], hv[4], dv[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int64_t o = i + k * stride;
            xv[k] = x[o];
            pv[k] = p[o];
            qv[k] = q[o];
            hv[k] = h[o];
            dv[k] = MODE == 1 ? dinv[o] : T(0);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) one(i + k * stride, xv[k], pv[k], qv[k], hv[k], dv[k]);
    }
    for (; i < n; i += stride) one(i, x[i], p[i], q[i], h[i], MODE == 1 ? dinv[i] : T(0));
    if (MODE == 0) return;
    __syncthreads();
    const double b2 = block_sum(acc2, lds);
    __syncthreads();
    const double b = MODE == 1 ? block_sum(acc, lds) : b2;
    if (threadIdx.x == 0) {
        pp[blockIdx.x] = b;
        pp[gridDim.x + blockIdx.x] = b2;
    }
}

// partials of <a, b> and (NQ = 2) of <a, a>
template <typename T, int NQ, typename TB = T>
__global__ void __launch_bounds__(RED_THREADS)
    k_cg_dots(const T *__restrict__ a, const TB *__restrict__ b, int64_t n, const KState *__restrict__ st,
              double *__restrict__ out)
{
    if (cg_skip_step(*st)) return;
    __shared__ double lds[RED_THREADS / 64];
    double acc = 0, acc2 = 0;
    const int64_t stride = (int64_t)gridDim.x * RED_THREADS;
    int64_t i = blockIdx.x * (int64_t)RED_THREADS + threadIdx.x;
    for (; i + 3 * stride < n; i += 4 * stride) {
        T va[4];
        TB vb[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            va[k] = a[i + k * stride];
            vb[k] = b[i + k * stride];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            acc += (double)va[k] * (double)vb[k];
            if (NQ == 2) acc2 += (double)va[k] * (double)va[k];
        }
    }
    for (; i < n; i += stride) {
        acc += (double)a[i] * (double)b[i];
        if (NQ == 2) acc2 += (double)a[i] * (double)a[i];
    }
    const double s = block_sum(acc, lds);
    __syncthreads();
    const double s2 = NQ == 2 ? block_sum(acc2, lds) : 0.0;
    if (threadIdx.x == 0) {
        out[blockIdx.x] = s;
        if (NQ == 2) out[gridDim.x + blockIdx.x] = s2;
    }
}

// many partials to fewer: workgroup b sums its part of each of the nq lists
// in[k * n ..] into out[k * gridDim.x + b]
__global__ void __launch_bounds__(RED_THREADS)
    k_cg_fewer(const double *__restrict__ in, int64_t n, int nq, double *__restrict__ out, const KState *__restrict__ st)
{
    if (cg_skip_step(*st)) return;
    __shared__ double lds[RED_THREADS / 64];
    const int64_t lo = n * blockIdx.x / gridDim.x, hi = n * (blockIdx.x + 1) / gridDim.x;
    for (int k = 0; k < nq; ++k) {
        const double t = sum_parts(in + k * n + lo, (int)(hi - lo), lds);
        if (threadIdx.x == 0) out[(int64_t)k * gridDim.x + blockIdx.x] = t;
    }
}

// ---- GMRES kernels --------------------------------------------------------------
// v0 -= b (v0 = A x on entry), partials of ||v0||^2
template <typename T>
__global__ void __launch_bounds__(RED_THREADS)
    k_gm_start(T *__restrict__ v0, const T *__restrict__ b, int64_t n, double *__restrict__ part)
{
    __shared__ double lds[RED_THREADS / 64];
    double acc = 0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const T v = (T)((double)v0[i] - (double)b[i]);
        v0[i] = v;
        acc += (double)v * (double)v;
    }
    const double bs = block_sum(acc, lds);
    if (threadIdx.x == 0) part[blockIdx.x] = bs;
}

// partials of <v_l, w>, l = 0..j: workgroup (s, q) takes slice s of the
// vectors and the GRP basis vectors from q GRP on, into mpart[l * slices + s]
template <typename T>
__global__ void __launch_bounds__(RED_THREADS)
    k_gm_multidot(const T *__restrict__ V, const T *__restrict__ w, int64_t n, int j, const KState *__restrict__ st,
                  double *__restrict__ mpart)
{
    if (gm_skip_step(*st)) return;
    __shared__ double lds[GRP][RED_THREADS / 64];
    const int g0 = blockIdx.y * GRP, cnt = j + 1 - g0 < GRP ? j + 1 - g0 : GRP;
    const int64_t lo = n * blockIdx.x / gridDim.x, hi = n * (blockIdx.x + 1) / gridDim.x;
    double acc[GRP];
#pragma unroll
    for (int l = 0; l < GRP; ++l) acc[l] = 0;
    const T *V0 = V + (int64_t)g0 * n;
    // four elements per thread and step, so that 4 (GRP + 1) loads are in
    // flight per thread
    int64_t i = lo + threadIdx.x;
    for (; i + 3 * (int64_t)RED_THREADS < hi; i += 4 * (int64_t)RED_THREADS) {
        double wi[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) wi[u] = (double)w[i + u * RED_THREADS];
#pragma unroll
        for (int l = 0; l < GRP; ++l)
            if (l < cnt) {
                const T *vl = V0 + (int64_t)l * n + i;
                double t = 0;
#pragma unroll
                for (int u = 0; u < 4; ++u) t = fma((double)vl[u * RED_THREADS], wi[u], t);
                acc[l] += t;
            }
    }
    for (; i < hi; i += RED_THREADS) {
        const double wi = (double)w[i];
#pragma unroll
        for (int l = 0; l < GRP; ++l)
            if (l < cnt) acc[l] += (double)V0[(int64_t)l * n + i] * wi;
    }
#pragma unroll
    for (int l = 0; l < GRP; ++l) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) acc[l] += __shfl_xor(acc[l], off, 64);
        if ((threadIdx.x & 63) == 0) lds[l][threadIdx.x >> 6] = acc[l];
    }
    __syncthreads();
    const int l = threadIdx.x;
    if (l < cnt) {
        double t = 0;
#pragma unroll
        for (int k = 0; k < RED_THREADS / 64; ++k) t += lds[l][k];
        mpart[(size_t)(g0 + l) * gridDim.x + blockIdx.x] = t;
    }
}

__device__ __forceinline__ void rot(double &x, double &y, double c, double s)
{
    const double a = x, b = y;
    x = c * a + s * b;
    y = c * b - s * a;
}

// w -= sum_l h_l v_l with h_l from the multi-dot's partials (kept as column j
// of H), partials of ||w||^2
template <typename T>
__global__ void __launch_bounds__(RED_THREADS)
    k_gm_orth(const T *__restrict__ V, T *__restrict__ w, int64_t n, int j, KState *__restrict__ st,
              const double *__restrict__ mpart, int slices, double *__restrict__ part, int m)
{
    if (gm_skip_step(*st)) {
        if (blockIdx.x == 0 && threadIdx.x == 0) gm_pass_on(*st);
        return;
    }
    __shared__ double lds[RED_THREADS / 64];
    __shared__ double h[GM_MAX + 1];
    {
        // one wavefront per dot
        const int lane = threadIdx.x & 63;
        for (int l = threadIdx.x >> 6; l <= j; l += RED_THREADS / 64) {
            double v = 0;
            for (int k = lane; k < slices; k += 64) v += mpart[(size_t)l * slices + k];
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
            if (lane == 0) {
                h[l] = v;
                if (blockIdx.x == 0) st->H[l * m + j] = v;
            }
        }
    }
    __syncthreads();
    double acc = 0;
    // a quarter of a slice of the multi-dot, by the workgroup whose number
    // equals the slice's modulo 8: the same XCD (see there)
    const int sl = blockIdx.x % slices, sub = 4 * sl + blockIdx.x / slices;
    const int64_t lo = n * sub / (4 * slices), hi = n * (sub + 1) / (4 * slices);
    for (int64_t i = lo + threadIdx.x; i < hi; i += RED_THREADS) {
        double v = (double)w[i];
        // unrolled so that several basis-vector loads are in flight
#pragma unroll 16
        for (int l = 0; l <= j; ++l) v -= h[l] * (double)V[(int64_t)l * n + i];
        const T vt = (T)v;
        w[i] = vt;
        acc += (double)vt * (double)vt;
    }
    const double bs = block_sum(acc, lds);
    if (threadIdx.x == 0) part[blockIdx.x] = bs;
}

// v /= ||v|| from the partials of its square sum; the first workgroup also
// keeps the scalars.  j >= 0: column j of H is finished (subdiagonal, Givens
// rotations, residual estimate, convergence); j < 0: a cycle begins with the
// residual v (j = -1 the first of a solve, -2 a later one).  z (may be null):
// the Jacobi preconditioner's z = dinv v in the same pass
template <typename T>
__global__ void __launch_bounds__(RED_THREADS)
    k_gm_scale(T *__restrict__ v, int64_t n, int j, KState *__restrict__ st, const double *__restrict__ part,
               int nparts, int m, const T *__restrict__ dinv, T *__restrict__ z)
{
    if (gm_skip_scale(*st, j)) return;
    __shared__ double lds[RED_THREADS / 64];
    __shared__ double col[GM_MAX + 1], cs[GM_MAX], sn[GM_MAX];
    const bool keeper = blockIdx.x == 0;
    if (keeper && j >= 0)
        for (int i = threadIdx.x; i <= j; i += RED_THREADS) {
            col[i] = st->H[i * m + j];
            if (i < j) {
                cs[i] = st->cs[i];
                sn[i] = st->sn[i];
            }
        }
    const double nrm = sqrt(sum_parts(part, nparts, lds));
    if (nrm > 0) {
        const double a = 1.0 / nrm;
        for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
            const T t = (T)((double)v[i] * a);
            v[i] = t;
            if (z) z[i] = dinv[i] * t;
        }
    }
    if (!keeper || threadIdx.x != 0) return;
    if (j < 0) {
        if (j == -1 && st->criteria == FEM_ERRMEASURE_REDUCTION) st->gtol *= nrm;
        gm_begin(*st, nrm);
        return;
    }
    double x = col[0];   // H[i][j] while the rotations pass down the column
    for (int i = 0; i < j; ++i) {
        double below = col[i + 1];
        rot(below, x, cs[i], sn[i]);
        st->H[i * m + j] = x;
        x = below;
    }
    const double a = x, b = nrm;
    const double r = sqrt(a * a + b * b);
    const double c = a / r, s = -b / r;
    st->cs[j] = c;
    st->sn[j] = s;
    double low = b, top = a;
    rot(low, top, c, s);
    st->H[j * m + j] = top;
    double gl = 0.0, gt = st->g[j];
    rot(gl, gt, c, s);
    st->g[j] = gt;
    st->g[j + 1] = gl;
    gm_keep(*st, j, m, gl);
}

// H y = g, back substitution by one wavefront, lane i holding row i
__global__ void __launch_bounds__(64) k_gm_backsolve(KState *st, int m)
{
    __shared__ double H[GM_MAX * GM_MAX];
    const int last = st->jlast, i = threadIdx.x;
    for (int k = i; k < last * last; k += 64) H[k] = st->H[(k / last) * m + k % last];
    double s = i < last ? st->g[i] : 0.0, y = 0.0;
    __syncthreads();
    for (int c = last - 1; c >= 0; --c) {
        const double yc = __shfl(s, c, 64) / H[c * last + c];
        if (i == c) y = yc;
        if (i < c) s -= H[i * last + c] * yc;
    }
    if (i < last) st->y[i] = y;
}

// u = beta_u * u + sum_{i<last} y_i Z_i
template <typename T, typename TU>
__global__ void k_gm_update(TU *__restrict__ u, const T *__restrict__ Z, int64_t n, const KState *__restrict__ st,
                            int zero_first)
{
    __shared__ double y[GM_MAX];
    const int last = st->jlast;
    for (int l = threadIdx.x; l < last; l += blockDim.x) y[l] = st->y[l];
    __syncthreads();
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        double v = zero_first ? 0.0 : (double)u[i];
        for (int l = 0; l < last; ++l) v += y[l] * (double)Z[(int64_t)l * n + i];
        u[i] = (TU)v;
    }
}

template <typename T>
__global__ void k_add(T *__restrict__ u, const T *__restrict__ z, int64_t n)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        u[i] = u[i] + z[i];
}

// ---- BiCGStab kernels --------------------------------------------------------------
// LinearSolver::bicgstab (dune/fem/solver/linear/bicgstab.hh:56-222), right
// preconditioned; the scalars stay on the device.
// nu = <r, r*>, tolerance by criterion (relative: eps ||b||, reduction:
// eps sqrt(nu), absolute: eps)
__global__ void k_bicg_init(KState *st, double eps, int criteria, int maxit)
{
    const double nu = st->nu;
    st->tol = criteria == FEM_ERRMEASURE_RELATIVE ? eps * sqrt(st->bnorm2)
            : criteria == FEM_ERRMEASURE_REDUCTION ? eps * sqrt(nu) : eps;
    st->it = 0;
    st->maxit = maxit;
    st->done = maxit <= 0;
    st->fin = 0;
}

// alpha = nu / <tmp, r*>
template <typename T>
__global__ void __launch_bounds__(RED_THREADS)
    k_bicg_alpha(const T *__restrict__ tmp, const T *__restrict__ rs, int64_t n, KState *st, double *partials,
                 unsigned *counter)
{
    if (st->done) return;
    __shared__ double lds[RED_THREADS / 64];
    double acc = 0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        acc += (double)tmp[i] * (double)rs[i];
    double own = block_sum(acc, lds);
    __shared__ double res[1];
    if (finish_reduction(0.0, partials, counter, res, 1, &own) && threadIdx.x == 0) st->alpha = st->nu / res[0];
}

// s = r - alpha tmp
template <typename T>
__global__ void k_bicg_s(const T *__restrict__ r, const T *__restrict__ tmp, T *__restrict__ s, int64_t n,
                         const KState *__restrict__ st)
{
    if (st->done) return;
    const double a = st->alpha;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        s[i] = (T)((double)r[i] - a * (double)tmp[i]);
}

// the five inner products of scalarProductVecs (bicgstab.hh:19-54) and the
// scalars of the step: omega, the residual estimate, beta, nu; fin marks the
// last iteration (res < tol or it >= maxit)
template <typename T>
__global__ void __launch_bounds__(RED_THREADS)
    k_bicg_dots(const T *__restrict__ r, const T *__restrict__ s, const T *__restrict__ rs, int64_t n, KState *st,
                double *partials, unsigned *counter)
{
    if (st->done) return;
    __shared__ double lds[RED_THREADS / 64];
    double a[5] = { 0, 0, 0, 0, 0 };
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const double ri = (double)r[i], si = (double)s[i], ti = (double)rs[i];
        a[0] += ri * si;
        a[1] += ri * ri;
        a[2] += si * si;
        a[3] += si * ti;
        a[4] += ri * ti;
    }
    double own[5];
    for (int k = 0; k < 5; ++k) {
        own[k] = block_sum(a[k], lds);
        __syncthreads();
    }
    __shared__ double g[5];
    if (finish_reduction(0.0, partials, counter, g, 5, own) && threadIdx.x == 0) {
        const double omega = g[0] / g[1];
        const double res = sqrt(g[2] - omega * (2.0 * g[0] - omega * g[1]));
        const double beta = (g[3] - omega * g[4]) * st->alpha / (omega * st->nu);
        st->nu = g[3] - omega * g[4];
        st->omega = omega;
        st->beta = beta;
        st->bres = res;
        st->it += 1;
        st->fin = !(res >= st->tol) || st->it >= st->maxit;
    }
}

// x += alpha p + omega s; unless this was the last iteration:
// r = s - omega r, p = beta (p - omega tmp) + r
template <typename T>
__global__ void k_bicg_update(T *__restrict__ x, T *__restrict__ p, T *__restrict__ r, const T *__restrict__ s,
                              const T *__restrict__ tmp, int64_t n, const KState *__restrict__ st)
{
    if (st->done) return;
    const double a = st->alpha, w = st->omega, b = st->beta;
    const bool last = st->fin;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const double pi = (double)p[i], si = (double)s[i];
        x[i] = (T)((double)x[i] + a * pi + w * si);
        if (!last) {
            const double rn = si - w * (double)r[i];
            r[i] = (T)rn;
            p[i] = (T)(b * (pi - w * (double)tmp[i]) + rn);
        }
    }
}

// r = b - r
template <typename T>
__global__ void k_bicg_res(const T *__restrict__ b, T *__restrict__ r, int64_t n)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        r[i] = (T)((double)b[i] - (double)r[i]);
}

__global__ void k_bicg_commit(KState *st)
{
    if (!st->done && st->fin) st->done = 1;
}

// ---- refinement helpers -----------------------------------------------------------
// r64 = b - h (h = A x in FP64), partial ||r||^2 -> out
__global__ void __launch_bounds__(RED_THREADS)
    k_residual64(const double *__restrict__ b, const double *__restrict__ h, double *__restrict__ r, int64_t n,
                 double *partials, unsigned *counter, double *out)
{
    __shared__ double lds[RED_THREADS / 64];
    double acc = 0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const double v = b[i] - h[i];
        r[i] = v;
        acc += v * v;
    }
    double bs = block_sum(acc, lds);
    finish_reduction(0.0, partials, counter, out, 1, &bs);
}

__global__ void k_scale_to32(const double *__restrict__ r, float *__restrict__ r32, int64_t n, double a)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        r32[i] = (float)(r[i] * a);
}

__global__ void k_update64(double *__restrict__ x, const float *__restrict__ d, int64_t n, double a)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        x[i] += a * (double)d[i];
}

// ---------------------------------------------------------------------------------
void Solver::init(Context *c, const fem_solver_params &p)
{
    ctx = c;
    prm = p;
    FEM_CHECK(p.method >= FEM_SOLVER_CG && p.method <= FEM_SOLVER_BICGSTAB, FEM_ERR_ARG, "solver method");
    FEM_CHECK(p.restart >= 1 && p.restart <= GM_MAX, FEM_ERR_ARG, "gmres restart must be in 1..64");
    state.alloc(sizeof(KState));
    partials.alloc(sizeof(double) * (RED_BLOCKS * (GM_MAX + 2) + NORM_PARTS));
    counters.alloc(sizeof(unsigned) * 8);
    FEM_HIP(hipMemset(counters.p, 0, counters.bytes));
    FEM_HIP(hipHostMalloc((void **)&hstate, sizeof(KState), hipHostMallocDefault));
}

Solver::~Solver()
{
    if (hstate) (void)hipHostFree(hstate);
    for (DevBuf *b : work) delete b;
}

void Solver::bind(Operator *o, Precond *p, Operator *io, Precond *ip)
{
    op = iop = nullptr;
    pre = ipre = nullptr;
    FEM_CHECK(o, FEM_ERR_ARG, "bind: null operator");
    FEM_CHECK(!o->nonlinear() && (!io || !io->nonlinear()), FEM_ERR_STATE,
              "bind: the operator is nonlinear (bind its Jacobian; the Newton solve does)");
    FEM_CHECK(!p || p->op == o || p->op->N == o->N, FEM_ERR_ARG, "preconditioner does not match the operator");
    // an FP32 preconditioner may serve an FP64 solve (rounded in, widened
    // out); otherwise the precisions agree
    FEM_CHECK(!p || p->prec == o->vec_prec || (p->prec == FEM_F32 && o->vec_prec == FEM_F64 && !prm.refinement),
              FEM_ERR_ARG, "preconditioner precision does not match the operator");
    // the learned preconditioner is nonlinear in its argument (the coarse
    // scaling depends on it): only the flexible GMRES, which stores
    // z_j = M(v_j), stays a valid Krylov method with it
    auto flexible_only = [&](const Precond *q) {
        FEM_CHECK(!q || !q->learned_part() || prm.method == FEM_SOLVER_FGMRES, FEM_ERR_UNSUPPORTED,
                  "the learned preconditioner is nonlinear: it needs fem.solver.method = fgmres");
    };
    flexible_only(p);
    if (prm.refinement) {
        FEM_CHECK(io, FEM_ERR_ARG, "refinement needs an inner operator");
        FEM_CHECK(io->N == o->N, FEM_ERR_ARG, "inner operator size");
        FEM_CHECK(o->vec_prec == FEM_F64, FEM_ERR_ARG, "refinement: the outer operator must be FP64");
        // the inner Krylov solve runs in FP32 on FP32 work vectors
        FEM_CHECK(io->vec_prec == FEM_F32, FEM_ERR_ARG, "refinement: the inner operator must be FP32 or BF16-MFMA");
        FEM_CHECK(!ip || ip->prec == io->vec_prec, FEM_ERR_ARG, "inner preconditioner precision");
        FEM_CHECK(!ip || ip->op->N == io->N, FEM_ERR_ARG, "inner preconditioner size");
        flexible_only(ip);
    }
    // fem.solver.preconditioning.method: built here when no preconditioner
    // object is passed (KrylovInverseOperator::bind creates its own the same
    // way, krylovinverseoperators.hh:86-97).  Binding the same operator again
    // (a Newton solve binds each Jacobian S'(w) to the one solver) updates
    // the one built before in place: the same result as a new one, without
    // building the hierarchy and its buffers again.
    widened.reset();
    if (p && p->prec == FEM_F32 && o->vec_prec == FEM_F64) {
        widened.reset(new Precond());
        widened->init_widening(o, p);
        p = widened.get();
    }
    auto own = [&](std::unique_ptr<Precond> &mine, Operator *target) {
        if (mine && mine->updatable_for(target, prm.preconditioning)) {
            mine->update();
        } else {
            mine.reset();
            mine.reset(new Precond());
            mine->init(target, prm.preconditioning);
        }
        return mine.get();
    };
    if (!p && prm.preconditioning != FEM_PRE_NONE && !prm.refinement) p = own(own_pre, o);
    else own_pre.reset();
    if (prm.refinement && !ip && prm.preconditioning != FEM_PRE_NONE) ip = own(own_ipre, io);
    else own_ipre.reset();
    op = o;
    pre = p;
    iop = io;
    ipre = ip;
}

void Solver::unbind()
{
    op = iop = nullptr;
    pre = ipre = nullptr;
    own_pre.reset();
    own_ipre.reset();
    widened.reset();
    for (DevBuf *b : work) delete b;
    work.clear();
}

void *Solver::workbuf(int i, size_t bytes)
{
    while ((int)work.size() <= i) work.push_back(new DevBuf());
    if (work[i]->bytes < bytes) work[i]->alloc(bytes);
    return work[i]->p;
}

void Solver::fetch_state()
{
    FEM_HIP(hipMemcpyAsync(hstate, state.p, KSTATE_HEAD, hipMemcpyDeviceToHost, ctx->stream));
    FEM_HIP(hipStreamSynchronize(ctx->stream));
}

template <typename T>
static int run_krylov(Solver &S, int method, Operator *o, Precond *p, const T *b, T *x, double eps, int criteria,
                      int maxit, int m, int64_t N, int verbose)
{
    hipStream_t s = S.ctx->stream;
    KState *st = S.state.as<KState>();
    double *part = S.partials.as<double>();
    unsigned *cnt = S.counters.as<unsigned>();
    const unsigned G = grid_for(N, 256, 4096);
    const size_t vb = sizeof(T) * N;
    const bool haspre = p && p->kind != FEM_PRE_NONE;
    FEM_HIP(hipMemsetAsync(st, 0, sizeof(KState), s));
    if (method == FEM_SOLVER_CG) {
        T *h = (T *)S.workbuf(0, vb), *r = (T *)S.workbuf(1, vb), *pp = (T *)S.workbuf(2, vb);
        // an FP32 preconditioner of an FP64 solve: p rounded (p32) and its
        // result (s32) pass between it and the CG kernels as they are, in the
        // place of s: 20 bytes per DoF and step, 40 with passes that round and
        // widen
        const Precond *low = haspre && !S.snapshot ? p->lowp : nullptr;
        const size_t half = (sizeof(float) * N + 255) / 256 * 256;
        T *ss = haspre ? (T *)S.workbuf(3, std::max(vb, low ? 2 * half : 0)) : pp,
          *q = haspre ? (T *)S.workbuf(4, vb) : pp;
        float *s32 = low ? (float *)ss : nullptr, *p32 = low ? (float *)((char *)ss + half) : nullptr;
        o->apply_raw(x, h, nullptr);
        hipLaunchKernelGGL(k_cg_setup<T>, dim3(G), dim3(256), 0, s, b, h, r, pp, N);
        if (haspre) {
            p->apply_raw(pp, q, nullptr);   // (the first step reads q alone)
        }
        dot_async(*S.ctx, N, pp, q, &st->res, cnt + 1, part);
        dot_async(*S.ctx, N, pp, pp, &st->rr, cnt + 1, part);
        dot_async(*S.ctx, N, b, b, &st->bnorm2, cnt + 1, part);
        hipLaunchKernelGGL(k_cg_init, dim3(1), dim3(1), 0, s, st, eps, criteria, maxit, S.prm.residual_check);
        FEM_HIP(hipGetLastError());
        const T *dinv = (haspre && p->pointwise()) ? (const T *)p->dinv.p : nullptr;
        // workgroups of the vector kernels (about four elements per thread),
        // and the partials of <q, h> and of <p, s>, <p, p>: from the apply
        // and from the preconditioner where they write them, else from a pass
        // over the vectors.  Every workgroup of the kernel that follows sums
        // them, so more than CG_PARTS are first brought down to CG_FEWER
        const unsigned GU = grid_for(N, 4 * RED_THREADS, CG_PARTS / 4);
        const bool qfused = o->desc.precision != FEM_BF16MFMA;
        const bool pfused = haspre && p->fused_dot();
        const int64_t nq0 = qfused ? o->dot_blocks() : GU, np0 = pfused ? p->dot_parts() : GU;
        const int nq = (int)(nq0 > CG_PARTS ? CG_FEWER : nq0), np = (int)(np0 > CG_PARTS ? CG_FEWER : np0);
        double *dq = (double *)S.workbuf(5, sizeof(double) * (nq0 + CG_FEWER));
        double *dp = (double *)S.workbuf(6, 2 * sizeof(double) * (np0 + CG_FEWER));
        double *qparts = nq0 > CG_PARTS ? dq + nq0 : dq, *pparts = np0 > CG_PARTS ? dp + 2 * np0 : dp;
        // steps between two looks of the host: a look costs about 20 us, a
        // step past the end one idle launch per kernel, of which a multigrid
        // step has some forty
        const int most = haspre && !dinv && !pfused ? 4 : 32;
        int chunk = S.snapshot ? S.snap_chunk : 4;
        // one CG step as a HIP graph: every kernel of the step reads a device
        // flag of the end, so replays after convergence do nothing; the step
        // holds no memset node.  Captured per solve (the vectors differ).
        hipGraph_t graph = nullptr;
        hipGraphExec_t gexec = nullptr;
        struct GraphGuard {
            hipGraph_t &g;
            hipGraphExec_t &e;
            ~GraphGuard()
            {
                if (e) (void)hipGraphExecDestroy(e);
                if (g) (void)hipGraphDestroy(g);
            }
        } gguard{ graph, gexec };
        auto cg_step = [&]() {
            if (low)
                hipLaunchKernelGGL((k_cg_dir<T, float>), dim3(GU), dim3(RED_THREADS), 0, s, q, s32, 1.0, N, st, pparts, np);
            else
                hipLaunchKernelGGL((k_cg_dir<T, T>), dim3(GU), dim3(RED_THREADS), 0, s, q, haspre ? ss : r,
                                   haspre ? 1.0 : -1.0, N, st, pparts, np);
            o->apply_raw(q, h, &st->end, qfused ? dq : nullptr);
            if (!qfused)
                hipLaunchKernelGGL((k_cg_dots<T, 1>), dim3(GU), dim3(RED_THREADS), 0, s, q, h, N, st, dq);
            if (nq0 > CG_PARTS)
                hipLaunchKernelGGL(k_cg_fewer, dim3(CG_FEWER), dim3(RED_THREADS), 0, s, dq, nq0, 1, qparts, st);
            if (!haspre) {
                hipLaunchKernelGGL((k_cg_update<T, 2>), dim3(GU), dim3(RED_THREADS), 0, s, x, r, q, h, (T *)nullptr, dinv,
                                   N, st, qparts, nq, dp, (float *)nullptr);
            } else if (dinv) {
                hipLaunchKernelGGL((k_cg_update<T, 1>), dim3(GU), dim3(RED_THREADS), 0, s, x, pp, q, h, ss, dinv, N, st,
                                   qparts, nq, dp, (float *)nullptr);
            } else {
                hipLaunchKernelGGL((k_cg_update<T, 0>), dim3(GU), dim3(RED_THREADS), 0, s, x, pp, q, h, (T *)nullptr, dinv, N,
                                   st, qparts, nq, dp, p32);
                if (low) low->apply_raw(p32, s32, &st->end);
                else p->apply_raw(pp, ss, &st->end, pfused ? dp : nullptr);
                if (low)
                    hipLaunchKernelGGL((k_cg_dots<T, 2, float>), dim3(GU), dim3(RED_THREADS), 0, s, pp, s32, N, st, dp);
                else if (!pfused)
                    hipLaunchKernelGGL((k_cg_dots<T, 2>), dim3(GU), dim3(RED_THREADS), 0, s, pp, ss, N, st, dp);
            }
            if (np0 > CG_PARTS)
                hipLaunchKernelGGL(k_cg_fewer, dim3(CG_FEWER), dim3(RED_THREADS), 0, s, dp, np0, 2, pparts, st);
        };
        if (S.prm.graph && !S.snapshot) {
            FEM_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
            cg_step();
            FEM_HIP(hipStreamEndCapture(s, &graph));
            FEM_HIP(hipGraphInstantiate(&gexec, graph, nullptr, nullptr, 0));
        }
        while (true) {
            for (int c = 0; c < chunk; ++c) {
                if (gexec) FEM_HIP(hipGraphLaunch(gexec, s));
                else cg_step();
            }
            hipLaunchKernelGGL(k_cg_check, dim3(1), dim3(RED_THREADS), 0, s, st, pparts, np);
            FEM_HIP(hipGetLastError());
            S.fetch_state();
            if (verbose) { std::printf("Fem::CG it: %d : residual %g\n", S.hstate->n_it, std::sqrt(S.hstate->n_res)); std::fflush(stdout); }
            if (S.hstate->done) break;
            if (S.snapshot) S.snapshot(x, pp);
            else if (chunk < most) chunk *= 2;
        }
        const int it = S.hstate->it;
        return it < maxit ? it : -it;
    }
    if (method == FEM_SOLVER_BICGSTAB) {
        // bicgstab.hh:56-222: right preconditioning iterates on y with
        // x = M^-1 y; the initial guess enters as y (r = b - A M^-1 x) and
        // the result is mapped back at the end (x = M^-1 y)
        T *r = (T *)S.workbuf(0, vb), *rs = (T *)S.workbuf(1, vb), *pp = (T *)S.workbuf(2, vb);
        T *ss = (T *)S.workbuf(3, vb), *tmp = (T *)S.workbuf(4, vb);
        T *z = haspre ? (T *)S.workbuf(5, vb) : nullptr;
        if (haspre) {
            p->apply_raw(x, z, nullptr);
            o->apply_raw(z, r, nullptr);
        } else {
            o->apply_raw(x, r, nullptr);
        }
        hipLaunchKernelGGL(k_bicg_res<T>, dim3(G), dim3(256), 0, s, b, r, N);   // r = b - A x
        FEM_HIP(hipMemcpyAsync(pp, r, vb, hipMemcpyDeviceToDevice, s));
        FEM_HIP(hipMemcpyAsync(rs, r, vb, hipMemcpyDeviceToDevice, s));
        dot_async(*S.ctx, N, r, rs, &st->nu, cnt + 1, part);
        dot_async(*S.ctx, N, b, b, &st->bnorm2, cnt + 1, part);
        hipLaunchKernelGGL(k_bicg_init, dim3(1), dim3(1), 0, s, st, eps, criteria, maxit);
        FEM_HIP(hipGetLastError());
        const int *skip = &st->done;
        int chunk = 4;
        while (true) {
            for (int c = 0; c < chunk; ++c) {
                if (haspre) {
                    p->apply_raw(pp, z, skip);
                    o->apply_raw(z, tmp, skip);
                } else {
                    o->apply_raw(pp, tmp, skip);
                }
                hipLaunchKernelGGL(k_bicg_alpha<T>, dim3(RED_DOT_BLOCKS), dim3(RED_THREADS), 0, s, tmp, rs, N, st, part, cnt);
                hipLaunchKernelGGL(k_bicg_s<T>, dim3(G), dim3(256), 0, s, r, tmp, ss, N, st);
                if (haspre) {
                    p->apply_raw(ss, z, skip);
                    o->apply_raw(z, r, skip);
                } else {
                    o->apply_raw(ss, r, skip);
                }
                hipLaunchKernelGGL(k_bicg_dots<T>, dim3(RED_DOT_BLOCKS), dim3(RED_THREADS), 0, s, r, ss, rs, N, st, part, cnt);
                hipLaunchKernelGGL(k_bicg_update<T>, dim3(G), dim3(256), 0, s, x, pp, r, ss, tmp, N, st);
                hipLaunchKernelGGL(k_bicg_commit, dim3(1), dim3(1), 0, s, st);
            }
            FEM_HIP(hipGetLastError());
            S.fetch_state();
            if (verbose) { std::printf("Fem::BiCGstab it: %d : %g\n", S.hstate->it, S.hstate->bres); std::fflush(stdout); }
            if (S.hstate->done) break;
            if (chunk < 64) chunk *= 2;
        }
        if (haspre) {
            p->apply_raw(x, z, nullptr);
            FEM_HIP(hipMemcpyAsync(x, z, vb, hipMemcpyDeviceToDevice, s));
        }
        const int it = S.hstate->it;
        return it < maxit ? it : -it;
    }
    // GMRES / FGMRES
    const bool flex = method == FEM_SOLVER_FGMRES;
    T *V = (T *)S.workbuf(0, vb * (m + 1));
    T *Z = (flex && haspre) ? (T *)S.workbuf(1, vb * m) : nullptr;
    T *z = (!flex && haspre) ? (T *)S.workbuf(2, vb) : nullptr;
    T *tmp = (!flex && haspre) ? (T *)S.workbuf(3, vb) : nullptr;
    // tolerance: eps * ||b|| for relative (gmres.hh:143-148)
    double bnorm = 0;
    if (criteria == FEM_ERRMEASURE_RELATIVE) {
        dot_async(*S.ctx, N, b, b, part + RED_BLOCKS * (GM_MAX + 1), cnt + 1, part);
        double hb;
        FEM_HIP(hipMemcpyAsync(&hb, part + RED_BLOCKS * (GM_MAX + 1), sizeof(double), hipMemcpyDeviceToHost, s));
        FEM_HIP(hipStreamSynchronize(s));
        bnorm = std::sqrt(hb);
    }
    {
        std::memset(S.hstate, 0, KSTATE_HEAD);
        S.hstate->gtol = criteria == FEM_ERRMEASURE_RELATIVE ? eps * bnorm : eps;
        S.hstate->criteria = criteria;
        S.hstate->maxit = maxit;
        FEM_HIP(hipMemcpyAsync(st, S.hstate, KSTATE_HEAD, hipMemcpyHostToDevice, s));
    }
    // slices of the multi-dot and workgroups of the other square sums: about
    // 1024 and 256 elements each while vectors are short (a step at 69 k DoFs:
    // 33.4 us with slices of 2048, 29.6 with 1024, 31.1 with 512), and from
    // 262 k DoFs on 256 slices, a workgroup per CU and group of vectors.
    // GMRES(30) + Jacobi, FP64, a step at 69 k, 0.88 M, 4.1 M and 16.8 M DoFs: 28,
    // 74, 321 and 1249 us (67, 117, 363 and 1283 us with 512 workgroups and a
    // finish by the last one).  Workgroups
    // go to the 8 XCDs in turn, so a multiple of 8 slices puts a slice of all
    // basis vectors into one XCD's L2, for the multi-dot and the
    // orthogonalisation alike (8.8 and 8.4 us without, 7.6 and 7.4 us with)
    const unsigned slices = (unsigned)std::min<int64_t>(NORM_PARTS / 4, (N + 8191) / 8192 * 8);
    const unsigned GN = grid_for(N, RED_THREADS, NORM_PARTS);
    double *npart = part + (size_t)RED_BLOCKS * (GM_MAX + 2);
    // Jacobi: its multiplication rides on the scaling of the basis vector
    const T *gdinv = haspre && p->pointwise() ? (const T *)p->dinv.p : nullptr;
    auto zvec = [&](int j) -> T * { return !gdinv ? nullptr : flex ? Z + (int64_t)j * N : z; };
    bool first = true;
    Learned *lp = p ? p->learned_part() : nullptr;
    T *xsave = lp ? (T *)S.workbuf(4, vb) : nullptr;
    while (true) {
        if (lp && lp->active()) FEM_HIP(hipMemcpyAsync(xsave, x, vb, hipMemcpyDeviceToDevice, s));
        o->apply_raw(x, V, nullptr);
        hipLaunchKernelGGL(k_gm_start<T>, dim3(GN), dim3(RED_THREADS), 0, s, V, b, N, npart);
        hipLaunchKernelGGL(k_gm_scale<T>, dim3(GN), dim3(RED_THREADS), 0, s, V, N, first ? -1 : -2, st, npart, (int)GN, m,
                           gdinv, zvec(0));
        first = false;
        for (int j = 0; j < m; ++j) {
            T *vj = V + (int64_t)j * N, *w = V + (int64_t)(j + 1) * N;
            const int *skip = &st->cycle_end;
            if (haspre) {
                T *zj = flex ? Z + (int64_t)j * N : z;
                if (!gdinv) p->apply_raw(vj, zj, skip);
                o->apply_raw(zj, w, skip);
            } else {
                o->apply_raw(vj, w, skip);
            }
            hipLaunchKernelGGL(k_gm_multidot<T>, dim3(slices, (unsigned)(j / GRP + 1)), dim3(RED_THREADS), 0, s, V, w, N, j,
                               st, part);
            hipLaunchKernelGGL(k_gm_orth<T>, dim3(4 * slices), dim3(RED_THREADS), 0, s, V, w, N, j, st, part, (int)slices, npart, m);
            hipLaunchKernelGGL(k_gm_scale<T>, dim3(GN), dim3(RED_THREADS), 0, s, w, N, j, st, npart, (int)(4 * slices), m,
                               gdinv, j + 1 < m ? zvec(j + 1) : (T *)nullptr);
        }
        hipLaunchKernelGGL(k_gm_backsolve, dim3(1), dim3(64), 0, s, st, m);
        if (flex && haspre) {
            hipLaunchKernelGGL((k_gm_update<T, T>), dim3(G), dim3(256), 0, s, x, Z, N, st, 0);
        } else if (haspre) {
            hipLaunchKernelGGL((k_gm_update<T, T>), dim3(G), dim3(256), 0, s, tmp, V, N, st, 1);
            p->apply_raw(tmp, z, nullptr);
            hipLaunchKernelGGL(k_add<T>, dim3(G), dim3(256), 0, s, x, z, N);
        } else {
            hipLaunchKernelGGL((k_gm_update<T, T>), dim3(G), dim3(256), 0, s, x, V, N, st, 0);
        }
        FEM_HIP(hipGetLastError());
        S.fetch_state();
        const double gres = S.hstate->gres;
        if (verbose) { std::printf("Fem::%sGMRES it: %d : %g\n", flex ? "F" : "", S.hstate->it, gres); std::fflush(stdout); }
        if (lp && lp->active() && !S.hstate->converged && S.hstate->jlast > 0 && !(gres < 0.95 * S.hstate->res)) {
            // the learned correction stagnates or broke down: undo the cycle
            // and continue with block Jacobi only
            FEM_HIP(hipMemcpyAsync(x, xsave, vb, hipMemcpyDeviceToDevice, s));
            lp->mode = FEM_LEARNED_OFF;
            S.fallback_used = 1;
            continue;
        }
        if (S.hstate->converged || S.hstate->it >= maxit) break;
    }
    const int it = S.hstate->it;
    return it < maxit ? it : -it;
}

int Solver::krylov(int method, Operator *o, Precond *p, const void *b, void *x, double tol, int criteria, int maxit,
                   int restart, int64_t N, int prec)
{
    if (prec == FEM_F64)
        return run_krylov<double>(*this, method, o, p, (const double *)b, (double *)x, tol, criteria, maxit, restart, N, prm.verbose);
    return run_krylov<float>(*this, method, o, p, (const float *)b, (float *)x, tol, criteria, maxit, restart, N, prm.verbose);
}

double Solver::true_residual(const Vec &b, const Vec &x, Vec &r)
{
    // ||b - A x|| / ||b|| with FP64 accumulation
    op->apply(x, r);
    Vec &rr = r;
    vec_scal(rr, -1.0);
    vec_axpy(rr, 1.0, b);
    const double rn = vec_dot(rr, rr), bn = vec_dot(b, b);
    return bn > 0 ? std::sqrt(rn / bn) : std::sqrt(rn);
}

void Solver::solve(const Vec &b, Vec &x, fem_solver_info &info)
{
    FEM_CHECK(op, FEM_ERR_STATE, "solve before bind");
    FEM_CHECK(b.n == op->N && x.n == op->N, FEM_ERR_ARG, "solve: vector size");
    FEM_CHECK(b.prec == op->vec_prec && x.prec == op->vec_prec, FEM_ERR_ARG, "solve: vector precision");
    std::memset(&info, 0, sizeof(info));
    fallback_used = 0;
    // a stall fallback switches the learned preconditioner off for the rest
    // of this solve only: its mode is restored on return, so the next solve
    // runs the network again (and reports its own fallback)
    struct ModeGuard {
        Learned *l;
        int mode;
        ~ModeGuard() { if (l) l->mode = mode; }
    } g_outer{ pre ? pre->learned_part() : nullptr, pre && pre->learned_part() ? pre->learned_part()->mode : 0 },
        g_inner{ ipre ? ipre->learned_part() : nullptr, ipre && ipre->learned_part() ? ipre->learned_part()->mode : 0 };
    const int64_t N = op->N;
    FEM_HIP(hipStreamSynchronize(ctx->stream));
    auto t0 = std::chrono::steady_clock::now();
    Vec r;
    r.ctx = ctx;
    r.n = N;
    r.prec = op->vec_prec;
    r.data = workbuf(20, x.bytes());
    r.owner = false;
    if (!prm.refinement) {
        info.iterations = krylov(prm.method, op, pre, b.data, x.data, prm.tolerance, prm.errormeasure,
                                 prm.maxiterations, prm.restart, N, op->vec_prec);
        info.converged = info.iterations >= 0;
        // residualcheck holds CG to the true residual as well: when the
        // recursive residual has converged but b - A x has drifted above the
        // tolerance, CG restarts from x (at most twice)
        if (prm.residual_check && prm.method == FEM_SOLVER_CG && prm.errormeasure != FEM_ERRMEASURE_REDUCTION) {
            for (int rs = 0; rs < 2 && info.converged; ++rs) {
                const double rel = true_residual(b, x, r);
                const double bn = std::sqrt(vec_dot(b, b));
                const double res = prm.errormeasure == FEM_ERRMEASURE_RELATIVE ? rel : rel * (bn > 0 ? bn : 1.0);
                if (!(res > prm.tolerance)) break;
                const int left = prm.maxiterations - info.iterations;
                if (left <= 0) {
                    info.converged = 0;
                    info.iterations = -info.iterations;
                    break;
                }
                const int more = krylov(prm.method, op, pre, b.data, x.data, prm.tolerance, prm.errormeasure, left,
                                        prm.restart, N, op->vec_prec);
                info.iterations = more >= 0 ? info.iterations + more : -(info.iterations - more);
                info.converged = more >= 0;
            }
        }
    } else {
        // FP64 iterative refinement around a low-precision Krylov solve
        hipStream_t s = ctx->stream;
        double *h = (double *)workbuf(10, sizeof(double) * N);
        double *r = (double *)workbuf(11, sizeof(double) * N);
        float *r32 = (float *)workbuf(12, sizeof(float) * N);
        float *d32 = (float *)workbuf(13, sizeof(float) * N);
        double *part = partials.as<double>();
        unsigned *cnt = counters.as<unsigned>();
        double *dres = part + RED_BLOCKS * (GM_MAX + 1);
        const unsigned G = grid_for(N, 256, 4096);
        const double bn = std::sqrt(vec_dot(b, b));
        int total = 0, outer = 0;
        bool ok = false;
        double rn0 = 0;   // the first residual (residualreduction)
        while (true) {
            op->apply_raw(x.data, h, nullptr);
            hipLaunchKernelGGL(k_residual64, dim3(RED_BLOCKS), dim3(RED_THREADS), 0, s, (const double *)b.data, h, r, N, part, cnt + 2, dres);
            double rn2;
            FEM_HIP(hipMemcpyAsync(&rn2, dres, sizeof(double), hipMemcpyDeviceToHost, s));
            FEM_HIP(hipStreamSynchronize(s));
            const double rn = std::sqrt(rn2);
            const double rel = bn > 0 ? rn / bn : rn;
            if (prm.verbose) { std::printf("IR outer %d: rel residual %g (inner its %d)\n", outer, rel, total); std::fflush(stdout); }
            if (outer == 0) rn0 = rn;
            const double target = prm.errormeasure == FEM_ERRMEASURE_RELATIVE    ? prm.tolerance * bn
                                  : prm.errormeasure == FEM_ERRMEASURE_REDUCTION ? prm.tolerance * rn0
                                                                                 : prm.tolerance;
            if (rn <= target || !(rn == rn)) { ok = rn == rn; break; }
            if (outer >= 100 || total >= prm.maxiterations) break;
            hipLaunchKernelGGL(k_scale_to32, dim3(G), dim3(256), 0, s, r, r32, N, 1.0 / rn);
            FEM_HIP(hipMemsetAsync(d32, 0, sizeof(float) * N, s));
            int its = krylov(prm.method, iop, ipre, r32, d32, prm.inner_tolerance, FEM_ERRMEASURE_RELATIVE,
                             prm.inner_maxiterations, prm.restart, N, FEM_F32);
            total += its < 0 ? -its : its;
            hipLaunchKernelGGL(k_update64, dim3(G), dim3(256), 0, s, (double *)x.data, d32, N, rn);
            FEM_HIP(hipGetLastError());
            ++outer;
        }
        info.iterations = ok ? total : -total;
        info.outer_iterations = outer;
        info.converged = ok;
    }
    FEM_HIP(hipStreamSynchronize(ctx->stream));
    auto t1 = std::chrono::steady_clock::now();
    info.time_s = std::chrono::duration<double>(t1 - t0).count();
    info.true_rel_residual = true_residual(b, x, r);
    info.fallback = fallback_used;
}

}  // namespace femamd
