// Continuous Lagrange Q2 operator on structured quad meshes: matrix-free
// apply, diagonal and load vector, for one instance or a batch of
// independent instances in one launch.
//
// Reference semantics: GalerkinOperator::evaluate element loop with
// addLocalDofs scatter (dune/fem/schemes/galerkin.hh:811-917, 929-934) and
// DirichletWrapperOperator::operator() (dirichletwrapper.hh:101-105: w_D = u_D).
//
// The tile of a workgroup and the exchange between its elements: fem_cg_tile.hpp.
#include "fem_blas.hpp"
#include "fem_cg_tile.hpp"

#include <algorithm>

namespace femamd {

CGTab make_cg_tab()
{
    CGTab t;
    double x[3], w[3];
    gauss_legendre01(3, x, w);
    for (int q = 0; q < 3; ++q) {
        t.w[q] = w[q];
        for (int i = 0; i < 3; ++i) {
            t.L[q][i] = lagrange2(i, x[q]);
            t.Ld[q][i] = lagrange2_d(i, x[q]);
        }
    }
    return t;
}

// w = A u (APPLY), the diagonal, the load vector.  The apply moves 9 coefficients per
// element and two vectors, and on a few hundred thousand elements it is a single set of
// workgroups, so what counts is the chain of one of them: 517 x 386 FP64 with pointwise
// kappa 7.1 us back to back on vectors that the caches keep (27 MB; 12.2 us with FP64 tables
// converted at each use, four coloured additions into LDS with a barrier each, and
// neighbouring tiles on different XCDs, of that last 1.8 us), 8.7 us (13.5 us) where the
// vectors change from call to call; 1024^2 26 us (49.6 us).  tile_inst names the instance of a
// workgroup, one load where a search over the instances' first tiles was a chain of five
// to eight; a single instance comes with the arguments.
template <int TX, int TY, typename T, bool APPLY, bool RX>
__global__ void __launch_bounds__((TX + 1) * (TY + 1))
    k_cg(int mode, const CGInst one, const CGInst *__restrict__ insts, const int *__restrict__ tile_inst, const CGTab *__restrict__ tabp,
         const T *__restrict__ kvol, const T *__restrict__ in, T *__restrict__ out, const int *__restrict__ skip,
         const int *__restrict__ inst_done, const CGReaction<T> rx, double *__restrict__ dot)
{
    constexpr int NT = (TX + 1) * (TY + 1);
    if (skip && *skip) return;
    __shared__ T xch[5][NT];
    const int bid = (int)xcd_remap(blockIdx.x, gridDim.x);
    const int ii = tile_inst ? tile_inst[bid] : 0;
    if (inst_done && inst_done[ii]) return;   // uniform over the block
    const CGInst P = tile_inst ? insts[ii] : one;
    const CGTile t = cg_tile<TX, TY>(P, bid);
    const T *u = in + P.dof_off;
    const int64_t e = P.elem_off + (int64_t)t.ey * P.nx + t.ex;
    T wl[3][3] = {}, ul[3][3] = {};
    if (t.valid) {
        if constexpr (APPLY) {
            T kap[9], cv[9];
#pragma unroll
            for (int iy = 0; iy < 3; ++iy)
#pragma unroll
                for (int ix = 0; ix < 3; ++ix) ul[iy][ix] = u[(int64_t)(2 * t.ey + iy) * t.NX + 2 * t.ex + ix];
#pragma unroll
            for (int q = 0; q < 9; ++q) {
                kap[q] = kvol ? kvol[e * 9 + q] : (T)P.kappa_const;
                cv[q] = RX && rx.cvol ? rx.cvol[e * 9 + q] : T(0);
            }
            // the reaction c + cvol + coef u^pw (the pointwise and nonlinear
            // parts of a single instance)
            const T c = (T)P.c, dj = (T)P.detJ;
            cg_element<T, RX>(ul, kap, (T)P.sx, (T)P.sy, [&](T uq, int q) {
                T r = c + cv[q];
                if (rx.pw) {
                    T pw = rx.coef;
                    for (int n = 0; n < rx.pw; ++n) pw *= uq;
                    r += pw;
                }
                return dj * r;
            }, wl);
        } else {
            const CGTab &tb = *tabp;
            const double hx = 1.0 / P.nx, hy = 1.0 / P.ny, detJ = hx * hy;
#pragma unroll
            for (int iy = 0; iy < 3; ++iy)
#pragma unroll
                for (int ix = 0; ix < 3; ++ix) {
                    double a = 0;
                    for (int qy = 0; qy < 3; ++qy)
                        for (int qx = 0; qx < 3; ++qx) {
                            const double W = tb.w[qx] * tb.w[qy] * detJ;
                            const double k = kvol ? (double)kvol[e * 9 + qx + 3 * qy] : P.kappa_const;
                            const double lx = tb.L[qx][ix], ly = tb.L[qy][iy];
                            if (mode == CG_MODE_DIAG) {
                                const double gx = tb.Ld[qx][ix] * ly / hx, gy = lx * tb.Ld[qy][iy] / hy;
                                const double r = P.c + (rx.cvol ? (double)rx.cvol[e * 9 + qx + 3 * qy] : 0.0);
                                a += W * (k * (gx * gx + gy * gy) + r * lx * lx * ly * ly);
                            } else {
                                a += W * k * lx * ly;  // kvol carries f for the load vector
                            }
                        }
                    wl[iy][ix] = (T)a;
                }
        }
    }
    T *o = out + P.dof_off;
    double d = 0;
    cg_gather<TX, TY, T>(P, t, wl, xch, [&](int64_t node, bool bnd, int iy, int ix, T v) {
        if constexpr (APPLY) {
            if (bnd) v = ul[iy][ix];
            o[node] = v;
            d += (double)ul[iy][ix] * (double)v;
        } else if (mode == CG_MODE_RHS_ADD) {
            // accumulate into the interior rows; the Dirichlet rows keep what
            // the apply wrote there
            if (!bnd) o[node] += v;
        } else {
            o[node] = bnd ? (mode == CG_MODE_DIAG ? T(1) : T(0)) : v;
        }
    });
    if (APPLY && dot) {
        __shared__ double lds[(NT + 63) / 64];
        const double tot = block_sum(d, lds);
        if (threadIdx.x == 0) dot[bid] = tot;
    }
}

// out[e*9 + qx + 3 qy] = base + coef u(x_q)^pw (base may be null: 0): u at
// the volume quadrature points of a single instance, one thread per element
template <typename T>
__global__ void __launch_bounds__(256)
    k_cg_eval_qp(int nx, int ny, const CGTab *__restrict__ tabp, const T *__restrict__ u, const T *__restrict__ base,
                 T coef, int pw, T *__restrict__ out)
{
    const int64_t E = (int64_t)nx * ny;
    const CGTab &tb = *tabp;
    const int NX = 2 * nx + 1;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < E; e += (int64_t)gridDim.x * blockDim.x) {
        const int ex = (int)(e % nx), ey = (int)(e / nx);
        T ul[3][3];
        for (int iy = 0; iy < 3; ++iy)
            for (int ix = 0; ix < 3; ++ix) ul[iy][ix] = u[(int64_t)(2 * ey + iy) * NX + 2 * ex + ix];
        for (int qy = 0; qy < 3; ++qy)
            for (int qx = 0; qx < 3; ++qx) {
                T uq = 0;
                for (int iy = 0; iy < 3; ++iy)
                    for (int ix = 0; ix < 3; ++ix) uq += (T)tb.L[qy][iy] * (T)tb.L[qx][ix] * ul[iy][ix];
                T v = coef;
                for (int t = 0; t < pw; ++t) v *= uq;
                out[e * 9 + qx + 3 * qy] = (base ? base[e * 9 + qx + 3 * qy] : T(0)) + v;
            }
    }
}

template <typename T>
void cg_eval_qp(int nx, int ny, const CGTab *d_tab, const T *u, const T *base, T coef, int pw, T *out, hipStream_t s)
{
    const int64_t E = (int64_t)nx * ny;
    const unsigned G = (unsigned)std::min<int64_t>((E + 255) / 256, 4096);
    hipLaunchKernelGGL(k_cg_eval_qp<T>, dim3(G), dim3(256), 0, s, nx, ny, d_tab, u, base, coef, pw, out);
    FEM_HIP(hipGetLastError());
}
template void cg_eval_qp<double>(int, int, const CGTab *, const double *, const double *, double, int, double *,
                                 hipStream_t);
template void cg_eval_qp<float>(int, int, const CGTab *, const float *, const float *, float, int, float *,
                                hipStream_t);

template <int TX, int TY, typename T>
static void launch_tile(int mode, const CGInst &one, const CGInst *d_inst, const int *tile_inst, int tiles,
                        const CGTab *d_tab, const T *kvol, const T *in, T *out, const int *skip, const int *inst_done, hipStream_t s,
                        const CGReaction<T> &rx, bool reaction, double *dot)
{
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(tiles), dim3((TX + 1) * (TY + 1)), 0, s, mode, one, d_inst, tile_inst, d_tab, kvol,
                           in, out, skip, inst_done, rx, dot);
    };
    if (mode != CG_MODE_APPLY) go(k_cg<TX, TY, T, false, false>);
    else if (reaction) go(k_cg<TX, TY, T, true, true>);
    else go(k_cg<TX, TY, T, true, false>);
}

template <typename T>
void cg_launch_shape(int shape, int mode, const CGInst *inst, const int *tile_inst, int total_tiles, const CGTab *d_tab,
                     const T *kvol, const T *in, T *out, const int *skip, const int *inst_done, hipStream_t s,
                     const CGReaction<T> &rx, bool c, double *dot)
{
    FEM_CHECK(!tile_inst || (!rx.cvol && !rx.pw), FEM_ERR_ARG, "pointwise/nonlinear reaction: a single instance");
    const bool reaction = c || rx.cvol || rx.pw;
#define CGS(ID, TX, TY)                                                                                          \
    case ID:                                                                                                     \
        launch_tile<TX, TY, T>(mode, tile_inst ? CGInst{} : *inst, inst, tile_inst, total_tiles, d_tab, kvol, in, out, skip, inst_done, s, rx, \
                               reaction, dot);                                                                   \
        break;
    switch (shape) {
        CGS(0, 15, 15) CGS(1, 7, 7) CGS(2, 15, 7) CGS(3, 31, 7) CGS(4, 7, 31)
    default: throw Error(FEM_ERR_ARG, "tile shape");
    }
#undef CGS
    FEM_HIP(hipGetLastError());
}

template void cg_launch_shape<double>(int, int, const CGInst *, const int *, int, const CGTab *, const double *,
                                      const double *, double *, const int *, const int *, hipStream_t,
                                      const CGReaction<double> &, bool, double *);
template void cg_launch_shape<float>(int, int, const CGInst *, const int *, int, const CGTab *, const float *,
                                     const float *, float *, const int *, const int *, hipStream_t,
                                     const CGReaction<float> &, bool, double *);

}  // namespace femamd
