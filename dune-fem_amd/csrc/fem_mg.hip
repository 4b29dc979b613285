// Multigrid preconditioner for the SIPG DG operator (cellwise or constant
// kappa, no advection; a reaction c and a pointwise reaction cvol at the
// volume quadrature points, as the Jacobians of the nonlinear operators
// have, are taken into the levels: c as it is, cvol by its element means on
// the coarse DG levels, and from there by the Galerkin products into the
// vertex levels).  No reference counterpart: dune-fem
// reaches multigrid only through external packages (the "amg-jacobi"
// preconditioning method of dune/fem/solver/parameter.hh:48-59, an assembled-
// matrix AMG of dune-istl or PETSc).  This one is matrix-free and geometric.
//
// Levels (one symmetric V-cycle per application, so it is a fixed SPD
// operator and may precondition CG):
//   * DG levels Q_p -> Q_{p/2} -> ... -> Q_1 on the fine mesh.  The
//     orthonormal Legendre basis is hierarchical, so the prolongation embeds
//     the low modes and the restriction of a residual keeps them; with the
//     penalty factor of the fine operator the rediscretised Q_{p'} operator
//     equals the Galerkin product P^T A P exactly (the (p'+1)-point rules
//     integrate the Q_{p'} products exactly).  Smoother: damped exact
//     element-block Jacobi, nu sweeps before and after.
//   * The conforming trilinear space on the (n+1)^3 vertices, embedded in
//     DG Q1 (per element the 8 Legendre modes of the trilinear interpolant).
//     Its Galerkin operator P_c^T A_Q1 P_c is a 27-point stencil (interior
//     face terms vanish on continuous functions); it is computed on the
//     device in closed form from the Q1 level's coefficients.  Smoother:
//     damped Jacobi.
//   * Geometric vertex levels: every second vertex (and the last one) is
//     kept per direction, trilinear interpolation, Galerkin stencils
//     P^T A P formed directly from the finer stencil, down to at most 512
//     vertices, which are solved with a dense
//     inverse (Gauss-Jordan on the device; on the host, with pivoting, for
//     an indefinite operator).
// The conforming coarse space is what makes the method robust for the
// high-contrast coefficients of the configurations: element means (Q_0) as
// the coarse space of DG Q1 leave far more iterations (measured on the CPU
// on a 12^3 channel problem: 69 PCG iterations with an exact Q_0 coarse
// solve against 27 with the exact conforming one).
#include <cmath>
#include <type_traits>

#include "fem_blas.hpp"
#include "fem_mg.hpp"

namespace femamd {

namespace {

constexpr int MGT = 256;   // threads of the grid-stride level kernels
constexpr int MG_DENSE_MAX = 512;

inline unsigned mg_grid(int64_t n) { return grid_for(n, MGT, 16384); }

#define MG_SKIP \
    if (skip && *skip) return

// ---- DG levels ----------------------------------------------------------------------
// xf += P xc (embedding of the low modes), a pass of its own: a sweep that adds
// P xc as it reads its seven pencils came out slower or the same (V-cycle 64^3
// Q4 FP32 1230 us against 1172 us, 48^3 Q3 FP64 392 us against 366 us)
template <typename T>
__global__ void k_mg_prolong_modes(int64_t E, int Kf, int Kc, const T *__restrict__ xc, T *__restrict__ xf,
                                   const int *__restrict__ skip)
{
    MG_SKIP;
    const int Kc3 = Kc * Kc * Kc, Kf3 = Kf * Kf * Kf;
    const int64_t n = E * Kc3;
    const bool narrow = n < (int64_t(1) << 31);
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n; q += (int64_t)gridDim.x * blockDim.x) {
        const int64_t e = narrow ? (int64_t)((unsigned)q / (unsigned)Kc3) : q / Kc3;
        const int l = (int)(q - e * Kc3);
        const int a = l / (Kc * Kc), b = (l / Kc) % Kc, c = l % Kc;
        xf[e * Kf3 + a * Kf * Kf + b * Kf + c] += xc[q];
    }
}

// ---- conforming trilinear <-> DG Q1 ------------------------------------------------------
// The 1D nodal functions 1 - s and s in the orthonormal Legendre modes
// phi_0 = 1, phi_1 = sqrt(3) (2 s - 1): coefficient of mode a for vertex i
__device__ __forceinline__ double tq1(int a, int i)
{
    return a == 0 ? 0.5 : (i ? 0.28867513459481287 : -0.28867513459481287);   // 1 / (2 sqrt 3)
}

// rv = P_c^T (r - A x), in two passes.  First, per element, the trilinear
// functional of the residual's Q1 modes at each of its 8 vertices, c[e][q]
// with q = i + 2 j + 4 k for the vertex (cx + i, cy + j, cz + k), kept in
// FP64, by the Q1 level's residual pass (fem_dg_modal.hip); then per vertex
// the sum over the (up to) 8 elements around it.  A single per-vertex pass
// would gather 8 x 8 mode values per vertex.
template <typename T>
__global__ void k_mg_corners_to_vertex(int nx, int ny, int nz, const double *__restrict__ c, T *__restrict__ rv,
                                       const int *__restrict__ skip)
{
    MG_SKIP;
    const int nvx = nx + 1, nvy = ny + 1;
    const int64_t V = (int64_t)nvx * nvy * (nz + 1);
    for (int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; v < V; v += (int64_t)gridDim.x * blockDim.x) {
        const int vx = (int)(v % nvx), vy = (int)((v / nvx) % nvy), vz = (int)(v / ((int64_t)nvx * nvy));
        double acc = 0;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int i = q & 1, j = (q >> 1) & 1, k = q >> 2;
            const int cx = vx - i, cy = vy - j, cz = vz - k;
            const bool in = cx >= 0 && cx < nx && cy >= 0 && cy < ny && cz >= 0 && cz < nz;
            const int64_t e = in ? cx + (int64_t)nx * (cy + (int64_t)ny * cz) : 0;
            const double val = c[e * 8 + q];
            acc += in ? val : 0.0;
        }
        rv[v] = (T)acc;
    }
}

// x += P_c xv: the Q1 modes of the trilinear interpolant of the vertex values
template <typename T>
__global__ void k_mg_vertex_to_dg1(int nx, int ny, int nz, const T *__restrict__ xv, T *__restrict__ x,
                                   const int *__restrict__ skip)
{
    MG_SKIP;
    const int nvx = nx + 1, nvy = ny + 1;
    const int64_t n = (int64_t)nx * ny * nz * 8;
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n; q += (int64_t)gridDim.x * blockDim.x) {
        const int64_t e = q >> 3;
        const int l = (int)(q & 7), a = l >> 2, b = (l >> 1) & 1, c = l & 1;
        const int cx = (int)(e % nx), cy = (int)((e / nx) % ny), cz = (int)(e / ((int64_t)nx * ny));
        double acc = 0;
        for (int k = 0; k < 2; ++k)
            for (int j = 0; j < 2; ++j)
                for (int i = 0; i < 2; ++i)
                    acc += tq1(a, i) * tq1(b, j) * tq1(c, k) *
                           (double)xv[(cx + i) + (int64_t)nvx * ((cy + j) + (int64_t)nvy * (cz + k))];
        x[q] = (T)((double)x[q] + acc);
    }
}

// ---- vertex levels -------------------------------------------------------------------
struct VDims {
    int n[3];
};

// The stencil is stored by offset, A[s * V + v] with s = (dx+1) + 3 (dy+1) +
// 9 (dz+1), so each of the 27 coefficient loads is coalesced; a neighbour outside
// the lattice reads v itself with weight 0, so all loads are issued together.
//
// Vertex sweeps: three lanes per vertex, one per z-plane of its stencil (the
// block is VS vertices by 3 planes, the plane sums meet in LDS).  The levels are
// small (33^3 vertices and fewer behind a 32^3 mesh), so what bounds them is the
// chain of loads of one vertex and the workgroups in flight, not the bandwidth:
// with a thread per vertex the 27 + 27 loads of a sweep took up to 256 registers
// and 33^3 vertices made 141 workgroups (FP32 hierarchy of 33^3 vertices: down
// 8.6 us, up 9.8 us; V-cycle 48^3 Q1 FP64 143 us, now 122 us).
constexpr int VS = 64;

// the sum over the three planes of a vertex, valid in plane 1
template <typename T>
__device__ __forceinline__ T plane_sum(T (*part)[VS], T acc)
{
    const int i = threadIdx.x, p = threadIdx.y;
    __syncthreads();
    if (p != 1) part[p >> 1][i] = acc;
    __syncthreads();
    return p == 1 ? (part[0][i] + acc) + part[1][i] : T(0);
}

// down: x0 = omega dinv r and t = r - A x0 (a Jacobi sweep from zero and the
// residual it leaves) in one pass: the neighbours' x0 is formed from r
template <typename T>
__global__ void __launch_bounds__(3 * VS)
    k_mg_v_down(VDims d, const T *__restrict__ A, const T *__restrict__ dinv, const T *__restrict__ r,
                T *__restrict__ x0, T *__restrict__ t, T omega, const int *__restrict__ skip)
{
    MG_SKIP;
    __shared__ T part[2][VS];
    const int64_t V = (int64_t)d.n[0] * d.n[1] * d.n[2];
    const int64_t sy = d.n[0], sz = (int64_t)d.n[0] * d.n[1];
    const int dz = (int)threadIdx.y - 1;
    for (int64_t v0 = blockIdx.x * (int64_t)VS; v0 < V; v0 += (int64_t)gridDim.x * VS) {
        const bool ok = v0 + threadIdx.x < V;
        const int64_t v = ok ? v0 + threadIdx.x : V - 1;
        const int vx = (int)(v % d.n[0]), vy = (int)((v / d.n[0]) % d.n[1]), vz = (int)(v / sz);
        const bool inz = vz + dz >= 0 && vz + dz < d.n[2];
        T acc = 0, xv = 0, rv = 0;
#pragma unroll
        for (int q = 0; q < 9; ++q) {
            const int dx = q % 3 - 1, dy = q / 3 - 1;
            const bool in = inz && vx + dx >= 0 && vx + dx < d.n[0] && vy + dy >= 0 && vy + dy < d.n[1];
            const T a = A[(threadIdx.y * 9 + q) * V + v];
            const int64_t w = in ? v + dx + dy * sy + dz * sz : v;
            const T rw = r[w], xw = omega * dinv[w] * rw;
            if (q == 4) {
                rv = rw;   // (of the vertex itself in plane 1)
                xv = xw;
            }
            acc = fma(in ? a : T(0), xw, acc);
        }
        acc = plane_sum(part, acc);
        if (threadIdx.y == 1 && ok) {
            x0[v] = xv;
            t[v] = rv - acc;
        }
    }
}

// the stencil from one row per vertex (A[v * 27 + s]) to one row per offset
__global__ void k_mg_by_offset(int64_t V, const double *__restrict__ Av, double *__restrict__ As)
{
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < V * 27; q += (int64_t)gridDim.x * blockDim.x) {
        const int64_t v = q / 27;
        const int s = (int)(q - v * 27);
        As[s * V + v] = Av[q];
    }
}

// 1D trilinear interpolation from the coarse vertices (fine positions 0, 2,
// 4, ..., and the last fine vertex) to fine vertex i: weight of coarse J.
// The last coarse vertex, J = ceil((nf - 1) / 2), is (i >> 1) or (i >> 1) + 1
// for i = nf - 1, so the two candidates of a fine vertex always cover it.
__device__ __forceinline__ double w1(int i, int J, int nf, int nc)
{
    if (i == nf - 1) return J == nc - 1 ? 1.0 : 0.0;
    if ((i & 1) == 0) return J == (i >> 1) ? 1.0 : 0.0;
    return (J == (i >> 1) || J == (i >> 1) + 1) ? 0.5 : 0.0;
}

// rc = P^T tf
template <typename T>
__global__ void k_mg_v_restrict(VDims f, VDims cdim, const T *__restrict__ tf, T *__restrict__ rc,
                                const int *__restrict__ skip)
{
    MG_SKIP;
    const int64_t Vc = (int64_t)cdim.n[0] * cdim.n[1] * cdim.n[2];
    for (int64_t J = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; J < Vc; J += (int64_t)gridDim.x * blockDim.x) {
        const int Jx = (int)(J % cdim.n[0]), Jy = (int)((J / cdim.n[0]) % cdim.n[1]),
                  Jz = (int)(J / ((int64_t)cdim.n[0] * cdim.n[1]));
        // per direction the fine vertices 2J-1, 2J, 2J+1 (in range) and
        // their weights; the last fine vertex, the only other candidate,
        // has weight 0 unless it is one of them (coarse1 puts the last
        // coarse vertex at or beyond it)
        int ix[3], iy[3], iz[3];
        double wx[3], wy[3], wz[3];
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            const int fx = 2 * Jx - 1 + m, fy = 2 * Jy - 1 + m, fz = 2 * Jz - 1 + m;
            const bool okx = fx >= 0 && fx < f.n[0], oky = fy >= 0 && fy < f.n[1], okz = fz >= 0 && fz < f.n[2];
            ix[m] = okx ? fx : 0;
            iy[m] = oky ? fy : 0;
            iz[m] = okz ? fz : 0;
            wx[m] = okx ? w1(fx, Jx, f.n[0], cdim.n[0]) : 0.0;
            wy[m] = oky ? w1(fy, Jy, f.n[1], cdim.n[1]) : 0.0;
            wz[m] = okz ? w1(fz, Jz, f.n[2], cdim.n[2]) : 0.0;
        }
        double acc = 0;
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int b = 0; b < 3; ++b)
#pragma unroll
                for (int a = 0; a < 3; ++a)
                    acc = fma(wx[a] * wy[b] * wz[c],
                              (double)tf[ix[a] + (int64_t)f.n[0] * (iy[b] + (int64_t)f.n[1] * iz[c])], acc);
        rc[J] = (T)acc;
    }
}

// up: x = x0 + P xc (the coarse correction), then the Jacobi sweep
// xout = x + omega dinv (r - A x), in one pass: a thread forms x on the 3 x 3
// vertices of its plane.  A plane has two candidate coarse planes (the second
// weighs in where the plane is odd), and the three vertices of a line have three
// coarse ones; interpolated in FP64, direction by direction.
template <typename T>
__global__ void __launch_bounds__(3 * VS)
    k_mg_v_up(VDims f, VDims cdim, const T *__restrict__ A, const T *__restrict__ dinv, const T *__restrict__ r,
              const T *__restrict__ x0, const T *__restrict__ xc, T *__restrict__ xout, T omega,
              const int *__restrict__ skip)
{
    MG_SKIP;
    __shared__ T part[2][VS];
    const int64_t V = (int64_t)f.n[0] * f.n[1] * f.n[2];
    const int64_t sy = f.n[0], sz = (int64_t)f.n[0] * f.n[1];
    const int dz = (int)threadIdx.y - 1;
    for (int64_t v0 = blockIdx.x * (int64_t)VS; v0 < V; v0 += (int64_t)gridDim.x * VS) {
        const bool ok = v0 + threadIdx.x < V;
        const int64_t v = ok ? v0 + threadIdx.x : V - 1;
        const int pos[3] = { (int)(v % f.n[0]), (int)((v / f.n[0]) % f.n[1]), (int)(v / sz) };
        const int iz = pos[2] + dz;
        const bool inz = iz >= 0 && iz < f.n[2];
        // x0 and the stencil of the plane
        T a[9], xo[9];
#pragma unroll
        for (int q = 0; q < 9; ++q) {
            const int dx = q % 3 - 1, dy = q / 3 - 1;
            const bool in = inz && pos[0] + dx >= 0 && pos[0] + dx < f.n[0] && pos[1] + dy >= 0 && pos[1] + dy < f.n[1];
            a[q] = A[(threadIdx.y * 9 + q) * V + v];
            a[q] = in ? a[q] : T(0);
            xo[q] = x0[in ? v + dx + dy * sy + dz * sz : v];
        }
        // the coarse vertices of the plane and of its lines in x and y
        const int Jz = inz ? iz >> 1 : 0;
        const int jz[2] = { min(Jz, cdim.n[2] - 1), min(Jz + 1, cdim.n[2] - 1) };
        const double wz[2] = { inz && Jz < cdim.n[2] ? w1(iz, Jz, f.n[2], cdim.n[2]) : 0.0,
                               inz && Jz + 1 < cdim.n[2] ? w1(iz, Jz + 1, f.n[2], cdim.n[2]) : 0.0 };
        double w[2][3][3];
        int jc[2][3];
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            const int J0 = ((pos[d] + 1) >> 1) - 1;
#pragma unroll
            for (int J = 0; J < 3; ++J) {
                const bool in = J0 + J >= 0 && J0 + J < cdim.n[d];
                jc[d][J] = in ? J0 + J : 0;
#pragma unroll
                for (int m = 0; m < 3; ++m) {
                    const int i = pos[d] - 1 + m;
                    w[d][m][J] = in && i >= 0 && i < f.n[d] ? w1(i, J0 + J, f.n[d], cdim.n[d]) : 0.0;
                }
            }
        }
        double xp[9] = { 0, 0, 0, 0, 0, 0, 0, 0, 0 };
#pragma unroll
        for (int Jy = 0; Jy < 3; ++Jy) {
            const T *row0 = xc + (int64_t)cdim.n[0] * (jc[1][Jy] + (int64_t)cdim.n[1] * jz[0]);
            const T *row1 = xc + (int64_t)cdim.n[0] * (jc[1][Jy] + (int64_t)cdim.n[1] * jz[1]);
            double c[3], fx[3];
#pragma unroll
            for (int J = 0; J < 3; ++J) c[J] = wz[0] * (double)row0[jc[0][J]] + wz[1] * (double)row1[jc[0][J]];
#pragma unroll
            for (int m = 0; m < 3; ++m) fx[m] = w[0][m][0] * c[0] + w[0][m][1] * c[1] + w[0][m][2] * c[2];
#pragma unroll
            for (int q = 0; q < 9; ++q) xp[q] = fma(w[1][q / 3][Jy], fx[q % 3], xp[q]);
        }
        T acc = 0;
#pragma unroll
        for (int q = 0; q < 9; ++q) {
            xo[q] = (T)((double)xo[q] + xp[q]);
            acc = fma(a[q], xo[q], acc);
        }
        acc = plane_sum(part, acc);
        if (threadIdx.y == 1 && ok) xout[v] = xo[4] + omega * dinv[v] * (r[v] - acc);
    }
}

// x = Ainv r with Ainv row-major: one wavefront per row (four per block),
// the lanes striding its columns (coalesced), then a butterfly sum.  The
// row index is the same on all lanes of a wavefront, so a wavefront past
// the last row leaves as a whole.
template <typename T>
__global__ void __launch_bounds__(256)
    k_mg_dense(int V, const T *__restrict__ Ainv, const T *__restrict__ r, T *__restrict__ x,
               const int *__restrict__ skip)
{
    MG_SKIP;
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= V) return;
    const T *a = Ainv + (int64_t)row * V;
    double acc = 0;
    for (int w = lane; w < V; w += 64) acc = fma((double)a[w], (double)r[w], acc);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (lane == 0) x[row] = (T)acc;
}

// ---- set-up (FP64) -----------------------------------------------------------------------

// the Gauss-weighted element means of a pointwise coefficient [E][K^3]
// (grid-stride: the level kernels' grid is capped)
__global__ void k_mg_cvol_mean(int64_t E, int K, const Tab1D<double> *__restrict__ tab,
                               const double *__restrict__ cvol, double *__restrict__ mean)
{
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < E; e += (int64_t)gridDim.x * blockDim.x) {
        const double *c = cvol + e * K * K * K;
        double s = 0;
        for (int qz = 0; qz < K; ++qz)
            for (int qy = 0; qy < K; ++qy)
                for (int qx = 0; qx < K; ++qx)
                    s += tab->w[qx] * tab->w[qy] * tab->w[qz] * c[qx + K * (qy + K * qz)];
        mean[e] = s;
    }
}

// the conforming level's stencil in closed form: a(phi_W, phi_v) of the DG Q1
// operator `a` on the trilinear hat functions of the (n+1)^3 vertices.  The
// interior face terms of SIPG vanish on continuous functions (no jumps; the
// flux terms against [v] cancel between the two sides), which leaves per
// element the stiffness kappa sum_d (h_t1 h_t2 / h_d) k(a_d, b_d) m(a_t1,
// b_t1) m(a_t2, b_t2) (k = +-1, m = 1/3, 1/6: the 1D linear stiffness and mass
// on [0, 1]), the reaction (c + cvol) at the 2^3 Gauss points, and on the
// domain boundary the Nitsche terms kappa (beta/h_d phi_a phi_b - n_d
// (d_d phi_a phi_b + phi_a d_d phi_b)) over the face.  One thread per vertex
// v and stencil offset s (W = v + d(s)); a, b are the local corners of W and
// v in each element that holds both.
__device__ __forceinline__ double mg_m1(int a, int b) { return a == b ? (1.0 / 3.0) : (1.0 / 6.0); }

__global__ void k_mg_conforming(const DGArgs<double> a, VDims vd, double *__restrict__ A)
{
    const int64_t V = (int64_t)vd.n[0] * vd.n[1] * vd.n[2];
    const Tab1D<double> &tb = *a.tab;
    const double detJ = a.h[0] * a.h[1] * a.h[2];
    for (int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < V * 27; g += (int64_t)gridDim.x * blockDim.x) {
        const int64_t v = g / 27;
        const int so = (int)(g - v * 27);
        const int P[3] = { (int)(v % vd.n[0]), (int)((v / vd.n[0]) % vd.n[1]), (int)(v / ((int64_t)vd.n[0] * vd.n[1])) };
        const int W[3] = { P[0] + so % 3 - 1, P[1] + (so / 3) % 3 - 1, P[2] + so / 9 - 1 };
        double acc = 0;
        if (W[0] >= 0 && W[1] >= 0 && W[2] >= 0 && W[0] < vd.n[0] && W[1] < vd.n[1] && W[2] < vd.n[2]) {
            for (int ez = P[2] - 1; ez <= P[2]; ++ez)
                for (int ey = P[1] - 1; ey <= P[1]; ++ey)
                    for (int ex = P[0] - 1; ex <= P[0]; ++ex) {
                        const int ec[3] = { ex, ey, ez };
                        int ca[3], cb[3];
                        bool in = true;
                        for (int d = 0; d < 3; ++d) {
                            cb[d] = P[d] - ec[d];
                            ca[d] = W[d] - ec[d];
                            in = in && ec[d] >= 0 && ec[d] < a.n[d] && ca[d] >= 0 && ca[d] <= 1;
                        }
                        if (!in) continue;
                        const int64_t e = ex + (int64_t)a.n[0] * (ey + (int64_t)a.n[1] * ez);
                        const double kap = a.kappa_mode == FEM_KAPPA_CELL ? a.kcell[e] : a.kappa_const;
                        for (int d = 0; d < 3; ++d) {
                            const int t1 = (d == 0) ? 1 : 0, t2 = (d == 2) ? 1 : 2;
                            const double mt = mg_m1(ca[t1], cb[t1]) * mg_m1(ca[t2], cb[t2]);
                            const double area = a.h[t1] * a.h[t2];
                            acc += kap * area / a.h[d] * (ca[d] == cb[d] ? 1.0 : -1.0) * mt;
                            for (int sd = 0; sd < 2; ++sd) {
                                if (ec[d] != (sd ? a.n[d] - 1 : 0)) continue;   // boundary faces only
                                const double nrm = sd ? 1.0 : -1.0;
                                const double va = ca[d] == sd ? 1.0 : 0.0, vb = cb[d] == sd ? 1.0 : 0.0;
                                const double da = ca[d] ? 1.0 : -1.0, db = cb[d] ? 1.0 : -1.0;
                                acc += area * mt * kap * (a.beta / a.h[d] * va * vb - nrm / a.h[d] * (da * vb + va * db));
                            }
                        }
                        // (the 2-point rule integrates the products exactly)
                        acc += (a.c + (a.ccell ? a.ccell[e] : 0.0)) * detJ * mg_m1(ca[0], cb[0]) * mg_m1(ca[1], cb[1]) *
                               mg_m1(ca[2], cb[2]);
                        if (!a.cvol) continue;
                        for (int qz = 0; qz < 2; ++qz)
                            for (int qy = 0; qy < 2; ++qy)
                                for (int qx = 0; qx < 2; ++qx) {
                                    const int q[3] = { qx, qy, qz };
                                    double pa = 1, pb = 1;
                                    for (int d = 0; d < 3; ++d) {
                                        const double xq = tb.x[q[d]];
                                        pa *= ca[d] ? xq : 1.0 - xq;
                                        pb *= cb[d] ? xq : 1.0 - xq;
                                    }
                                    acc += tb.w[qx] * tb.w[qy] * tb.w[qz] * detJ * a.cvol[e * 8 + qx + 2 * qy + 4 * qz] *
                                           pa * pb;
                                }
                    }
        }
        A[g] = acc;
    }
}

// The Galerkin product P^T A P of a vertex level, one direction at a time: P is the
// product of three 1D interpolations, so coarsening direction D of the rows and of
// the stencil's columns is a pass of its own,
//   out(V, s) = sum_i P(i, V) sum_t P(i + t, V + s_D) in(i, s with s_D = t),
// i = 2V-1 .. 2V+1 (which holds the last fine vertex when it belongs to V), t = -1 ..
// 1: nine coefficients per entry, loaded together, 0 where a vertex lies outside.
// All three directions in one kernel are up to 343 terms per entry behind branches
// (25^3 and 13^3 vertices: 110 us each, now 11 us in three launches).  One thread per row of the lattice
// c (coarse along D, as `f` along the others) and stencil offset.
template <int D>
__global__ void __launch_bounds__(MGT)
    k_mg_galerkin(VDims f, VDims c, const double *__restrict__ in, double *__restrict__ out)
{
    const int64_t n = (int64_t)c.n[0] * c.n[1] * c.n[2] * 27;
    const int nf = f.n[D], nc = c.n[D];
    constexpr int SD = D == 0 ? 1 : D == 1 ? 3 : 9;
    const int64_t fs = D == 0 ? 1 : D == 1 ? f.n[0] : (int64_t)f.n[0] * f.n[1];
    for (int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < n; g += (int64_t)gridDim.x * blockDim.x) {
        const int64_t v = g / 27;
        const int so = (int)(g - v * 27);
        int p[3] = { (int)(v % c.n[0]), (int)((v / c.n[0]) % c.n[1]), (int)(v / ((int64_t)c.n[0] * c.n[1])) };
        const int V = p[D], W = V + (so / SD) % 3 - 1;
        const int s0 = so - ((so / SD) % 3) * SD;
        p[D] = 0;
        const double *row = in + (p[0] + (int64_t)f.n[0] * (p[1] + (int64_t)f.n[1] * p[2])) * 27 + s0;
        const bool wok = W >= 0 && W < nc;
        double acc = 0;
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            const int i = 2 * V - 1 + m;
            const bool ok = i >= 0 && i < nf && wok;
            const double wv = ok ? w1(i, V, nf, nc) : 0.0;
            const double *a = row + (ok ? i : 0) * fs * 27;
            double r = 0;
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                const int j = i + t - 1;
                r = fma(ok && j >= 0 && j < nf ? w1(j, W, nf, nc) : 0.0, a[t * SD], r);
            }
            acc = fma(wv, r, acc);
        }
        out[g] = acc;
    }
}

// the Jacobi scaling of a vertex level: 1 / max(a_vv, lim sum_w |a_vw|).  By
// Gershgorin the eigenvalues of diag(d)^-1 A are then at most 1 / lim, so a
// sweep damped by omega = 1.9 lim stays convergent.  A diffusion stencil
// (off-diagonal sum -a_vv) keeps its diagonal; a reaction-dominated one (the
// Q1 mass stencil has row sum 3.375 a_vv) is scaled down instead of
// diverging.
__global__ void k_mg_dinv(int64_t V, const double *__restrict__ A, double lim, double *__restrict__ dinv)
{
    for (int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; v < V; v += (int64_t)gridDim.x * blockDim.x) {
        double rs = 0;
        for (int j = 0; j < 27; ++j) rs += fabs(A[v * 27 + j]);
        dinv[v] = 1.0 / fmax(A[v * 27 + 13], lim * rs);
    }
}

// the coarsest level's operator as a dense row-major V x V matrix from its
// 27-point stencil (offset s = sx + 3 sy + 9 sz, 0..2 each, about the vertex)
__global__ void k_mg_dense_fill(VDims d, const double *__restrict__ A, double *__restrict__ M)
{
    const int64_t V = (int64_t)d.n[0] * d.n[1] * d.n[2];
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < V * V; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t v = i / V, w = i - v * V;
        const int dx = (int)(w % d.n[0]) - (int)(v % d.n[0]);
        const int dy = (int)((w / d.n[0]) % d.n[1]) - (int)((v / d.n[0]) % d.n[1]);
        const int dz = (int)(w / ((int64_t)d.n[0] * d.n[1])) - (int)(v / ((int64_t)d.n[0] * d.n[1]));
        const bool in = dx >= -1 && dx <= 1 && dy >= -1 && dy <= 1 && dz >= -1 && dz <= 1;
        M[i] = in ? A[v * 27 + (dx + 1) + 3 * (dy + 1) + 9 * (dz + 1)] : 0.0;
    }
}

// X -> Y: one block step of the in-place Gauss-Jordan inversion of a V x V matrix,
// pivot rows and columns C = c .. c + GJ - 1 (the last step has fewer), with
// P = X[C, C]^-1:
//   Y[C, C] = P,  Y[C, k] = P X[C, k],  Y[r, C] = -X[r, C] P,
//   Y[r, k] = X[r, k] - X[r, C] P X[C, k].
// A launch has to see all of the step before it, so the inversion costs launches:
// 11 block steps for 343 vertices 190 us, 172 steps of two pivots 690 us.  A workgroup makes
// a GJ x GJ tile of Y and inverts the pivot block for itself in LDS, two pivots at a
// time (the chain of a division and an LDS round trip per step is most of a launch:
// one at a time 25 us).  Its pivots are those of the elimination without pivoting (the matrices are
// symmetric positive definite); they are recorded for the host to check.
constexpr int GJ = 32;
__global__ void __launch_bounds__(256)
    k_mg_gj_step(int V, int c, const double *__restrict__ X, double *__restrict__ Y, double *__restrict__ piv)
{
    __shared__ double D[2][GJ][GJ + 1], R[GJ][GJ + 1], L[GJ][GJ + 1];
    const int nb = min(GJ, V - c);
    const int r0 = blockIdx.y * GJ, k0 = blockIdx.x * GJ;
    const int ty = threadIdx.x >> 5, tx = threadIdx.x & 31;   // rows ty, ty + 8, ..., column tx
    constexpr int NR = GJ / 8;
    // the pivot block (1 on the diagonal past its end), the tile's pivot rows
    // and pivot columns (0 past the matrix)
#pragma unroll
    for (int n = 0; n < NR; ++n) {
        const int i = ty + 8 * n;
        D[0][i][tx] = i < nb && tx < nb ? X[(int64_t)(c + i) * V + c + tx] : (i == tx ? 1.0 : 0.0);
        R[i][tx] = i < nb && k0 + tx < V ? X[(int64_t)(c + i) * V + k0 + tx] : 0.0;
        L[i][tx] = r0 + i < V && tx < nb ? X[(int64_t)(r0 + i) * V + c + tx] : 0.0;
    }
    __syncthreads();
    const bool keeper = blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0;
    int h = 0;
    for (int p = 0; p < nb; p += 2, h ^= 1) {
        const double(*A)[GJ + 1] = D[h];
        double(*B)[GJ + 1] = D[h ^ 1];
        const double a = A[p][p], b = A[p][p + 1], g = A[p + 1][p], d = A[p + 1][p + 1];
        const double det = fma(a, d, -b * g), id = 1.0 / det;
        if (keeper) {
            piv[c + p] = a;
            if (p + 1 < nb) piv[c + p + 1] = det / a;
        }
        // rows p and p + 1 of the next matrix
        const bool col = (tx >> 1) == (p >> 1), odd = tx & 1;
        const double u = A[p][tx], v = A[p + 1][tx];
        const double rp = col ? (odd ? -b : d) * id : fma(d, u, -b * v) * id;
        const double rq = col ? (odd ? a : -g) * id : fma(a, v, -g * u) * id;
#pragma unroll
        for (int n = 0; n < NR; ++n) {
            const int i = ty + 8 * n;
            const double y = fma(-A[i][p], rp, fma(-A[i][p + 1], rq, col ? 0.0 : A[i][tx]));
            B[i][tx] = i == p ? rp : i == p + 1 ? rq : y;
        }
        __syncthreads();
    }
    const double(*P)[GJ + 1] = D[h];
    // T = P X[C, k] for the tile's columns (in the free half of D), then the tile
    double(*T)[GJ + 1] = D[h ^ 1];
    const bool pcol = k0 == c, prow = r0 == c;   // tiles and pivot blocks share their edges
    double t[NR] = {};
#pragma unroll 8
    for (int m = 0; m < GJ; ++m) {
        const double x = R[m][tx];
#pragma unroll
        for (int n = 0; n < NR; ++n) t[n] = fma(P[ty + 8 * n][m], x, t[n]);
    }
#pragma unroll
    for (int n = 0; n < NR; ++n) T[ty + 8 * n][tx] = pcol ? P[ty + 8 * n][tx] : t[n];
    __syncthreads();
    double y[NR];
#pragma unroll
    for (int n = 0; n < NR; ++n) {
        const int r = r0 + ty + 8 * n, k = k0 + tx;
        y[n] = prow ? T[ty + 8 * n][tx] : (!pcol && r < V && k < V) ? X[(int64_t)r * V + k] : 0.0;
    }
    if (!prow)
#pragma unroll 8
        for (int m = 0; m < GJ; ++m) {
            const double x = T[m][tx];
#pragma unroll
            for (int n = 0; n < NR; ++n) y[n] = fma(-L[ty + 8 * n][m], x, y[n]);
        }
#pragma unroll
    for (int n = 0; n < NR; ++n) {
        const int r = r0 + ty + 8 * n, k = k0 + tx;
        if (r < V && k < V) Y[(int64_t)r * V + k] = y[n];
    }
}

int coarse1(int nf) { return (nf - 1 + 1) / 2 + 1; }   // ceil((nf - 1) / 2) + 1

// the level's values in precision T
void store_as(int prec, DevBuf &dst, const DevBuf &src64, int64_t n, Context *ctx)
{
    dst.ensure(n * (prec == FEM_F64 ? 8 : 4));
    Vec a, b;
    a.ctx = b.ctx = ctx;
    a.n = b.n = n;
    a.prec = prec;
    b.prec = FEM_F64;
    a.data = dst.p;
    b.data = src64.p;
    a.owner = b.owner = false;
    vec_copy(a, b);
}

}  // namespace

void Multigrid::init(Operator *fine)
{
    op = fine;
    FEM_CHECK(fine->is_dg(), FEM_ERR_UNSUPPORTED, "multigrid: DG operators only");
    const fem_op_desc &d0 = fine->desc;
    FEM_CHECK(d0.b[0] == 0 && d0.b[1] == 0 && d0.b[2] == 0, FEM_ERR_UNSUPPORTED,
              "multigrid: operators without advection (b = 0)");
    FEM_CHECK(!fine->nonlinear(), FEM_ERR_STATE, "multigrid: the operator is nonlinear (build it on the Jacobian)");
    FEM_CHECK(d0.kappa_mode == FEM_KAPPA_CELL || d0.kappa_mode == FEM_KAPPA_CONST, FEM_ERR_UNSUPPORTED,
              "multigrid: cellwise or constant kappa");
    FEM_CHECK(fine->a64.kappa_mode >= 0, FEM_ERR_STATE, "coefficient data not set");
    Context *ctx = fine->ctx;
    desc = d0;
    reaction = fine->cvol64.p != nullptr;
    prec = fine->vec_prec;
    const int lp = prec == FEM_F64 ? FEM_F64 : FEM_F32;
    const int n[3] = { d0.n[0], d0.n[1], d0.n[2] };
    const int64_t E = fine->E;
    if (reaction) {
        cmean.alloc(sizeof(double) * E);
        cmean32.alloc(sizeof(float) * E);
    }
    // a coarse operator: the finest one's description at another order and
    // precision, with buffers for the coefficients update() fills (cellwise
    // kappa; a pointwise reaction as its element means, shared by the levels)
    auto make_op = [&](int order, int precision) {
        std::unique_ptr<Operator> o(new Operator());
        fem_op_desc d = d0;
        d.order = order;
        d.precision = precision;
        o->init(ctx, d);
        if (d0.kappa_mode == FEM_KAPPA_CELL) {
            o->kcell64.alloc(sizeof(double) * E);
            o->kcell32.alloc(sizeof(float) * E);
            o->a64.kcell = o->kcell64.as<double>();
            o->a32.kcell = o->kcell32.as<float>();
            o->a64.kappa_mode = o->a32.kappa_mode = FEM_KAPPA_CELL;
        }
        if (reaction) {
            o->a64.ccell = cmean.as<double>();
            o->a32.ccell = cmean32.as<float>();
        }
        return o;
    };
    const size_t es = lp == FEM_F64 ? 8 : 4;
    // DG levels: p, p/2, ..., 1
    for (int p = d0.order;; p = std::max(1, p / 2)) {
        std::unique_ptr<MGDGLevel> L(new MGDGLevel());
        if (dg.empty()) {
            L->op = fine;
            // BF16 rounds the quadrature values to 2^-8 of their size, which
            // is noise of order 4e-3 * lambda_max |x| in A x: far above the
            // smooth part of a smoothed residual, which is what the coarse
            // levels must see. The smoothers tolerate it; the restricted
            // residual is formed in FP32.
            if (d0.precision == FEM_BF16MFMA) L->resop = make_op(d0.order, FEM_F32);
        } else {
            L->own = make_op(p, lp);
            L->op = L->own.get();
            L->r.alloc(L->op->N * es);
            L->x.alloc(L->op->N * es);
        }
        L->k = p + 1;
        L->t.alloc(L->op->N * es);
        dg.push_back(std::move(L));
        if (p == 1) break;
    }
    corners.alloc(E * 8 * sizeof(double));
    // vertex levels: the conforming one, then every second vertex per
    // direction down to at most MG_DENSE_MAX vertices
    {
        std::unique_ptr<MGVertexLevel> V0(new MGVertexLevel());
        for (int d = 0; d < 3; ++d) V0->nv[d] = n[d] + 1;
        V0->V = (int64_t)V0->nv[0] * V0->nv[1] * V0->nv[2];
        vx.push_back(std::move(V0));
    }
    while (vx.back()->V > MG_DENSE_MAX) {
        const MGVertexLevel &F = *vx.back();
        std::unique_ptr<MGVertexLevel> C(new MGVertexLevel());
        for (int d = 0; d < 3; ++d) C->nv[d] = coarse1(F.nv[d]);
        C->V = (int64_t)C->nv[0] * C->nv[1] * C->nv[2];
        if (C->V == F.V) break;   // nothing left to coarsen
        vx.push_back(std::move(C));
    }
    FEM_CHECK(vx.back()->V <= 4096, FEM_ERR_UNSUPPORTED, "multigrid: coarsest vertex level too large");
    for (auto &L : vx) {
        A64.emplace_back(new DevBuf());
        A64.back()->alloc(L->V * 27 * 8);
        L->x.alloc(L->V * es);
        L->r.alloc(L->V * es);
        L->t.alloc(L->V * es);
        L->x0.alloc(L->V * es);
    }
    d64.alloc(vx[0]->V * 8);
    As64.alloc(vx[0]->V * 27 * 8);   // (also the lattice coarsened in x: no larger, coarse1(n) <= n for n >= 2)
    if (vx.size() > 1) gT.alloc((size_t)vx[1]->nv[0] * vx[1]->nv[1] * vx[0]->nv[2] * 27 * 8);
    const int64_t VC = vx.back()->V;
    gjX.alloc((size_t)VC * VC * 8);
    gjY.alloc((size_t)VC * VC * 8);
    gjp.alloc((size_t)VC * 8);
    update();
}

bool Multigrid::updatable_for(const Operator *o) const
{
    return o == op && (o->cvol64.p != nullptr) == reaction && !o->nonlinear();
}

void Multigrid::update()
{
    Operator *fine = op;
    Context *ctx = fine->ctx;
    hipStream_t s = ctx->stream;
    const int lp = prec == FEM_F64 ? FEM_F64 : FEM_F32;
    const int64_t E = fine->E;
    FEM_CHECK(fine->a64.kappa_mode >= 0, FEM_ERR_STATE, "coefficient data not set");
    FEM_CHECK((fine->cvol64.p != nullptr) == reaction, FEM_ERR_STATE,
              "multigrid: the pointwise reaction was added or removed since the set-up");
    auto round_into = [&](void *lo, const void *hi, int64_t nv) {
        Vec a, b;
        a.ctx = b.ctx = ctx;
        a.n = b.n = nv;
        a.prec = FEM_F32;
        b.prec = FEM_F64;
        a.data = lo;
        b.data = const_cast<void *>(hi);
        a.owner = b.owner = false;
        vec_copy(a, b);
    };
    // coarse coefficients: the cellwise kappa as it is, cvol by its
    // Gauss-weighted element means
    if (reaction) {
        hipLaunchKernelGGL(k_mg_cvol_mean, dim3(mg_grid(E)), dim3(MGT), 0, s, E, fine->k, fine->a64.tab,
                           fine->cvol64.as<double>(), cmean.as<double>());
        FEM_HIP(hipGetLastError());
        round_into(cmean32.p, cmean.p, E);
    }
    auto coefficients = [&](Operator *o) {
        if (desc.kappa_mode == FEM_KAPPA_CELL) {
            FEM_HIP(hipMemcpyAsync(o->kcell64.p, fine->kcell64.p, sizeof(double) * E, hipMemcpyDeviceToDevice, s));
            round_into(o->kcell32.p, o->kcell64.p, E);
        }
    };
    for (auto &L : dg) {
        if (L->own) coefficients(L->own.get());
        if (L->resop) coefficients(L->resop.get());
    }
    // smoother blocks; a varying pointwise reaction enters them by its
    // largest value per element: the damped sweep stays convergent (a block
    // below the true one can make it diverge, and the V-cycle indefinite)
    for (auto &L : dg) {
        if (L->bj.op) L->bj.update();
        else L->bj.init(L->op, FEM_PRE_BLOCK_JACOBI, true);
    }
    // vertex stencils: the conforming level from the Q1 level's FP64
    // coefficient data (every operator precision keeps it), then the
    // Galerkin products
    {
        const MGVertexLevel &V0 = *vx[0];
        VDims dv{ { V0.nv[0], V0.nv[1], V0.nv[2] } };
        hipLaunchKernelGGL(k_mg_conforming, dim3(mg_grid(V0.V * 27)), dim3(MGT), 0, s, dg.back()->op->a64, dv,
                           A64[0]->as<double>());
        FEM_HIP(hipGetLastError());
    }
    for (size_t l = 1; l < vx.size(); ++l) {
        const MGVertexLevel &F = *vx[l - 1], &C = *vx[l];
        VDims df{ { F.nv[0], F.nv[1], F.nv[2] } }, dc{ { C.nv[0], C.nv[1], C.nv[2] } };
        const VDims d1{ { dc.n[0], df.n[1], df.n[2] } }, d2{ { dc.n[0], dc.n[1], df.n[2] } };
        auto pass = [&](auto kernel, const VDims &f, const VDims &c, const DevBuf &in, DevBuf &out) {
            hipLaunchKernelGGL(kernel, dim3(mg_grid((int64_t)c.n[0] * c.n[1] * c.n[2] * 27)), dim3(MGT), 0, s, f, c,
                               in.as<double>(), out.as<double>());
        };
        pass(k_mg_galerkin<0>, df, d1, *A64[l - 1], As64);
        pass(k_mg_galerkin<1>, d1, d2, As64, gT);
        pass(k_mg_galerkin<2>, d2, dc, gT, *A64[l]);
        FEM_HIP(hipGetLastError());
    }
    // level data in the preconditioner's precision; a reaction-free level
    // keeps the plain diagonal (its stencils have row sums of at most twice
    // the diagonal away from the boundary)
    const double lim = (desc.c != 0 || reaction) ? omega_vertex / 1.9 : 0.0;
    for (size_t l = 0; l < vx.size(); ++l) {
        MGVertexLevel &L = *vx[l];
        hipLaunchKernelGGL(k_mg_dinv, dim3(mg_grid(L.V)), dim3(MGT), 0, s, L.V, A64[l]->as<double>(), lim,
                           d64.as<double>());
        hipLaunchKernelGGL(k_mg_by_offset, dim3(mg_grid(L.V * 27)), dim3(MGT), 0, s, L.V, A64[l]->as<double>(),
                           As64.as<double>());
        FEM_HIP(hipGetLastError());
        store_as(lp, L.A, As64, L.V * 27, ctx);
        store_as(lp, L.dinv, d64, L.V, ctx);
    }
    // dense inverse of the coarsest level, stored row-major: Gauss-Jordan on
    // the device (in blocks, no pivoting) for the symmetric
    // positive definite operators of diffusion and non-negative reaction; a
    // non-positive pivot (an indefinite operator) sends the inversion to the
    // host, with partial pivoting
    const MGVertexLevel &LC = *vx.back();
    const int VC = (int)LC.V;
    bool spd = true;
    {
        VDims dc{ { LC.nv[0], LC.nv[1], LC.nv[2] } };
        const unsigned G = mg_grid((int64_t)VC * VC);
        hipLaunchKernelGGL(k_mg_dense_fill, dim3(G), dim3(MGT), 0, s, dc, A64.back()->as<double>(), gjX.as<double>());
        int launches = 0;
        const unsigned T = (unsigned)((VC + GJ - 1) / GJ);
        for (int c = 0; c < VC; c += GJ, ++launches) {
            const DevBuf &src = (launches & 1) ? gjY : gjX;
            DevBuf &dst = (launches & 1) ? gjX : gjY;
            hipLaunchKernelGGL(k_mg_gj_step, dim3(T, T), dim3(256), 0, s, VC, c, src.as<double>(), dst.as<double>(),
                               gjp.as<double>());
        }
        FEM_HIP(hipGetLastError());
        std::vector<double> piv(VC);
        FEM_HIP(hipMemcpyAsync(piv.data(), gjp.p, sizeof(double) * VC, hipMemcpyDeviceToHost, s));
        FEM_HIP(hipStreamSynchronize(s));
        for (int c = 0; c < VC; ++c) spd = spd && piv[c] > 0 && std::isfinite(piv[c]);
        if (spd) store_as(lp, coarse_inv, (launches & 1) ? gjY : gjX, (int64_t)VC * VC, ctx);
    }
    if (!spd) {
        const MGVertexLevel &L = LC;
        const int V = VC;
        std::vector<double> st(L.V * 27);
        FEM_HIP(hipMemcpyAsync(st.data(), A64.back()->p, sizeof(double) * st.size(), hipMemcpyDeviceToHost, s));
        FEM_HIP(hipStreamSynchronize(s));
        std::vector<double> M((size_t)V * V, 0.0), I((size_t)V * V, 0.0);
        for (int v = 0; v < V; ++v) {
            const int x0 = v % L.nv[0], y0 = (v / L.nv[0]) % L.nv[1], z0 = v / (L.nv[0] * L.nv[1]);
            for (int sidx = 0; sidx < 27; ++sidx) {
                const int wx = x0 + sidx % 3 - 1, wy = y0 + (sidx / 3) % 3 - 1, wz = z0 + sidx / 9 - 1;
                if (wx < 0 || wy < 0 || wz < 0 || wx >= L.nv[0] || wy >= L.nv[1] || wz >= L.nv[2]) continue;
                M[(size_t)v * V + wx + L.nv[0] * (wy + L.nv[1] * wz)] = st[(size_t)v * 27 + sidx];
            }
            I[(size_t)v * V + v] = 1.0;
        }
        for (int c = 0; c < V; ++c) {
            int piv = c;
            for (int r = c + 1; r < V; ++r)
                if (std::fabs(M[(size_t)r * V + c]) > std::fabs(M[(size_t)piv * V + c])) piv = r;
            FEM_CHECK(M[(size_t)piv * V + c] != 0.0, FEM_ERR_ARG, "multigrid: singular coarsest operator");
            if (piv != c)
                for (int k = 0; k < V; ++k) {
                    std::swap(M[(size_t)piv * V + k], M[(size_t)c * V + k]);
                    std::swap(I[(size_t)piv * V + k], I[(size_t)c * V + k]);
                }
            const double ip = 1.0 / M[(size_t)c * V + c];
            for (int k = 0; k < V; ++k) {
                M[(size_t)c * V + k] *= ip;
                I[(size_t)c * V + k] *= ip;
            }
            for (int r = 0; r < V; ++r) {
                if (r == c) continue;
                const double f = M[(size_t)r * V + c];
                if (f == 0.0) continue;
                for (int k = 0; k < V; ++k) {
                    M[(size_t)r * V + k] -= f * M[(size_t)c * V + k];
                    I[(size_t)r * V + k] -= f * I[(size_t)c * V + k];
                }
            }
        }
        // row-major: element (row v, column w) at v * V + w
        const std::vector<double> &cm = I;
        DevBuf c64;
        c64.alloc(cm.size() * 8);
        FEM_HIP(hipMemcpy(c64.p, cm.data(), cm.size() * 8, hipMemcpyHostToDevice));
        store_as(lp, coarse_inv, c64, (int64_t)cm.size(), ctx);
    }
    FEM_HIP(hipStreamSynchronize(s));
}

template <typename T>
void Multigrid::cycle_vertex(size_t l, const T *r, T *x, const int *skip)
{
    MGVertexLevel &L = *vx[l];
    hipStream_t s = op->ctx->stream;
    const unsigned G = grid_for(L.V, VS, 16384);
    if (l + 1 == vx.size()) {
        hipLaunchKernelGGL(k_mg_dense<T>, dim3((unsigned)((L.V + 3) / 4)), dim3(256), 0, s, (int)L.V,
                           coarse_inv.as<T>(), r, x, skip);
        return;
    }
    VDims d{ { L.nv[0], L.nv[1], L.nv[2] } };
    T *t = L.t.as<T>(), *x0 = L.x0.as<T>();
    const T *A = L.A.as<T>(), *dv = L.dinv.as<T>();
    const T om = (T)omega_vertex;
    hipLaunchKernelGGL(k_mg_v_down<T>, dim3(G), dim3(VS, 3), 0, s, d, A, dv, r, x0, t, om, skip);
    MGVertexLevel &C = *vx[l + 1];
    VDims dc{ { C.nv[0], C.nv[1], C.nv[2] } };
    hipLaunchKernelGGL(k_mg_v_restrict<T>, dim3(grid_for(C.V, VS, 16384)), dim3(VS), 0, s, d, dc, (const T *)t, C.r.as<T>(), skip);
    cycle_vertex<T>(l + 1, C.r.as<T>(), C.x.as<T>(), skip);
    hipLaunchKernelGGL(k_mg_v_up<T>, dim3(G), dim3(VS, 3), 0, s, d, dc, A, dv, r, (const T *)x0, (const T *)C.x.as<T>(), x,
                       om, skip);
    FEM_HIP(hipGetLastError());
}

// mode 0: x = omega B^-1 r;  mode 1: x += omega B^-1 (r - t), t = A x
template <typename T>
static void mg_bj(const MGDGLevel &L, const T *r, const T *t, T *x, T omega, int mode, const int *skip, hipStream_t s)
{
    dg_block_apply<T>(L.k, L.op->E, L.bj.Q.as<T>(), L.bj.lam.as<T>(), r, mode ? t : nullptr, x, omega, mode != 0, skip, s);
}

// one damped block-Jacobi sweep on a level, out = in + omega B^-1 (r - A in),
// in one pass (FP64 and FP32 operators) or as an apply followed by the
// block-Jacobi kernel (BF16-MFMA operators, whose sweep keeps the BF16 apply;
// then out == in, and t is the scratch for A in)
template <typename T>
static void mg_sweep(const MGDGLevel &L, const T *r, const T *in, T *out, T *t, T omega, const int *skip, hipStream_t s)
{
    const Operator &o = *L.op;
    if (o.desc.precision == FEM_BF16MFMA) {
        L.op->apply_raw(in, t, skip);
        mg_bj<T>(L, r, t, out, omega, 1, skip, s);
        return;
    }
    DGSmooth<T> sm;
    sm.r = r;
    sm.Q = L.bj.Q.as<T>();
    sm.lam = L.bj.lam.as<T>();
    sm.omega = omega;
    sm.xout = out;
    if constexpr (std::is_same<T, double>::value) dg_modal_smooth_f64(o.a64, o.k, in, sm, skip, s);
    else dg_modal_smooth_f32(o.a32, o.k, in, sm, skip, s);
}

template <typename T>
void Multigrid::cycle_dg(size_t l, const T *r, T *x, const int *skip)
{
    MGDGLevel &L = *dg[l];
    hipStream_t s = op->ctx->stream;
    const int *n = op->desc.n;
    const int64_t E = op->E;
    T *t = L.t.as<T>();
    const T om = (T)omega_dg;
    // the fused sweeps write a second buffer (a sweep reads its input's
    // neighbours): cur is the buffer holding the current iterate, and the
    // first sweep is arranged so that the last one ends in x
    const bool fused = L.op->desc.precision != FEM_BF16MFMA;
    T *cur = x;
    auto sweep = [&]() {
        if (!fused) {
            mg_sweep<T>(L, r, cur, cur, t, om, skip, s);
            return;
        }
        T *nxt = cur == x ? t : x;
        mg_sweep<T>(L, r, cur, nxt, t, om, skip, s);
        cur = nxt;
    };
    // the pre-smoothing leaves its result in t when the remaining sweeps
    // (nu - 1 before, nu after) are odd in number, so that they end in x
    if (fused && ((2 * nu_dg - 1) & 1)) cur = t;
    mg_bj<T>(L, r, nullptr, cur, om, 0, skip, s);
    for (int it = 1; it < nu_dg; ++it) sweep();
    // the residual in the form the next level takes
    const Operator &ro = L.resop ? *L.resop : *L.op;
    DGResidual<T> rs;
    rs.r = r;
    auto residual = [&]() {
        if constexpr (std::is_same<T, double>::value) dg_modal_residual_f64(ro.a64, ro.k, cur, rs, skip, s);
        else dg_modal_residual_f32(ro.a32, ro.k, cur, rs, skip, s);
    };
    if (l + 1 < dg.size()) {
        MGDGLevel &C = *dg[l + 1];
        rs.rc = C.r.as<T>();
        rs.kc = C.k;
        residual();
        cycle_dg<T>(l + 1, C.r.as<T>(), C.x.as<T>(), skip);
        hipLaunchKernelGGL(k_mg_prolong_modes<T>, dim3(mg_grid(E * C.k * C.k * C.k)), dim3(MGT), 0, s, E, L.k, C.k,
                           (const T *)C.x.as<T>(), cur, skip);
    } else {
        MGVertexLevel &V0 = *vx[0];
        rs.corners = corners.as<double>();
        residual();
        hipLaunchKernelGGL(k_mg_corners_to_vertex<T>, dim3(mg_grid(V0.V)), dim3(MGT), 0, s, n[0], n[1], n[2],
                           (const double *)corners.as<double>(), V0.r.as<T>(), skip);
        cycle_vertex<T>(0, V0.r.as<T>(), V0.x.as<T>(), skip);
        hipLaunchKernelGGL(k_mg_vertex_to_dg1<T>, dim3(mg_grid(E * 8)), dim3(MGT), 0, s, n[0], n[1], n[2],
                           (const T *)V0.x.as<T>(), cur, skip);
    }
    for (int it = 0; it < nu_dg; ++it) sweep();
    FEM_CHECK(cur == x, FEM_ERR_STATE, "multigrid: the sweeps end outside the output buffer");
    FEM_HIP(hipGetLastError());
}

void Multigrid::smooth_fine(const void *r, const void *t, void *x, const int *skip)
{
    hipStream_t s = op->ctx->stream;
    if (prec == FEM_F64)
        mg_bj<double>(*dg[0], (const double *)r, (const double *)t, (double *)x, (double)omega_dg, 1, skip, s);
    else
        mg_bj<float>(*dg[0], (const float *)r, (const float *)t, (float *)x, (float)omega_dg, 1, skip, s);
    FEM_HIP(hipGetLastError());
}

void Multigrid::apply_raw(const void *r, void *z, const int *skip)
{
    if (prec == FEM_F64) cycle_dg<double>(0, (const double *)r, (double *)z, skip);
    else cycle_dg<float>(0, (const float *)r, (float *)z, skip);
}

}  // namespace femamd
