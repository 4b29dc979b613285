// The element and tile work of the 2D continuous-Q2 kernels (device code).
//
// A workgroup owns TX x TY elements and the nodes (2 ex + i, 2 ey + j), i, j = 0,
// 1, of each; one thread per element of the tile plus a lower halo row and
// column, so every contribution to an owned node is formed inside the workgroup.
// An element leaves the results that other threads own, its right column and top
// row, in LDS; after one barrier each owner adds them in a fixed order (own, left,
// below, below left), so results are deterministic and need no atomics.  The nodes
// of the domain's upper boundary lie outside every 2 x 2 block, but they are
// Dirichlet rows, which take no contributions: the last elements write them.
#pragma once

#include "fem_cg.hpp"

namespace femamd {

// Quadratic interpolation between the nodes 0, 1/2, 1 and the three Gauss points
// (1 -+ sqrt(3/5)) / 2 and 1/2, by even and odd parts: with s = a0 + a2, d = a2 - a0
// the values are 0.3 s + 0.4 a1 -+ (sqrt(0.6) / 2) d and a1, the derivatives
// d -+ 2 sqrt(0.6) (s - 2 a1) and d.
template <typename T>
struct Q2Line {
    static constexpr T E = T(0.38729833462074168852), G = T(1.54919333848296675407), A = T(0.3), B = T(0.4);
    __device__ static __forceinline__ void value(const T (&a)[3], T (&f)[3])
    {
        const T m = fma(A, a[0] + a[2], B * a[1]), e = E * (a[2] - a[0]);
        f[0] = m - e;
        f[1] = a[1];
        f[2] = m + e;
    }
    __device__ static __forceinline__ void deriv(const T (&a)[3], T (&g)[3])
    {
        const T d = a[2] - a[0], h = G * fma(T(-2), a[1], a[0] + a[2]);
        g[0] = d - h;
        g[1] = d;
        g[2] = d + h;
    }
    // a_i = sum_q f_q l_i(x_q) + g_q l_i'(x_q)
    __device__ static __forceinline__ void test(const T (&f)[3], const T (&g)[3], T (&a)[3])
    {
        const T M = f[0] + f[2], H = G * (g[2] - g[0]);
        const T s = fma(A, M, H), d = fma(E, f[2] - f[0], (g[0] + g[2]) + g[1]);
        a[0] = s - d;
        a[1] = fma(T(-2), H, fma(B, M, f[1]));
        a[2] = s + d;
    }
    __device__ static __forceinline__ void test_value(const T (&f)[3], T (&a)[3])
    {
        const T M = f[0] + f[2], s = A * M, d = E * (f[2] - f[0]);
        a[0] = s - d;
        a[1] = fma(B, M, f[1]);
        a[2] = s + d;
    }
    // the Gauss weights 5/18, 4/9, 5/18
    __device__ static __forceinline__ constexpr T w(int q) { return q == 1 ? T(4.0 / 9.0) : T(5.0 / 18.0); }
};

// the element's part of A u: ul and wl are [iy][ix], kap the coefficients at the
// points qx + 3 qy, r(uq, q) the reaction coefficient there (times detJ)
template <typename T, bool RX, typename R>
__device__ __forceinline__ void cg_element(const T (&ul)[3][3], const T (&kap)[9], T sx, T sy, R r, T (&wl)[3][3])
{
    using Q = Q2Line<T>;
    T v[3][3], gx[3][3];   // [qx][iy]
#pragma unroll
    for (int iy = 0; iy < 3; ++iy) {
        T f[3], g[3];
        Q::value(ul[iy], f);
        Q::deriv(ul[iy], g);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            v[q][iy] = f[q];
            gx[q][iy] = g[q];
        }
    }
    T tv[3][3], tg[3][3];   // [iy][qx], to be tested with values and derivatives in x
#pragma unroll
    for (int qx = 0; qx < 3; ++qx) {
        T uq[3], dy[3], dx[3], fx[3], fy[3], fm[3] = { T(0), T(0), T(0) }, a[3];
        Q::deriv(v[qx], dy);
        Q::value(gx[qx], dx);
        if constexpr (RX) Q::value(v[qx], uq);
#pragma unroll
        for (int qy = 0; qy < 3; ++qy) {
            const T W = Q::w(qx) * Q::w(qy), k = W * kap[qx + 3 * qy];
            fx[qy] = k * sx * dx[qy];
            fy[qy] = k * sy * dy[qy];
            if constexpr (RX) fm[qy] = W * r(uq[qy], qx + 3 * qy) * uq[qy];
        }
        Q::test_value(fx, a);
#pragma unroll
        for (int iy = 0; iy < 3; ++iy) tg[iy][qx] = a[iy];
        Q::test(fm, fy, a);
#pragma unroll
        for (int iy = 0; iy < 3; ++iy) tv[iy][qx] = a[iy];
    }
#pragma unroll
    for (int iy = 0; iy < 3; ++iy) Q::test(tv[iy], tg[iy], wl[iy]);
}

// where a workgroup and its threads stand
struct CGTile {
    int tx, ty, ex, ey, NX;
    bool valid, owner;
};

template <int TX, int TY>
__device__ __forceinline__ CGTile cg_tile(const CGInst &P, int bid)
{
    CGTile t;
    const int tile = bid - P.tile_off;
    t.tx = threadIdx.x % (TX + 1);
    t.ty = threadIdx.x / (TX + 1);
    t.ex = (tile % P.tiles_x) * TX - 1 + t.tx;
    t.ey = (tile / P.tiles_x) * TY - 1 + t.ty;
    t.valid = t.ex >= 0 && t.ey >= 0 && t.ex < P.nx && t.ey < P.ny;
    t.owner = t.valid && t.tx > 0 && t.ty > 0;
    t.NX = 2 * P.nx + 1;
    return t;
}

// gathers the element results wl (0 where the element does not exist) and calls
// put(node, boundary, iy, ix, value) for every owned node; iy, ix = the node's place
// in the owner's element.  One barrier, which every thread reaches.
template <int TX, int TY, typename T, typename Put>
__device__ __forceinline__ void cg_gather(const CGInst &P, const CGTile &t, const T (&wl)[3][3],
                                          T (*x)[(TX + 1) * (TY + 1)], Put put)
{
    const int i = threadIdx.x;
    x[0][i] = wl[0][2];
    x[1][i] = wl[1][2];
    x[2][i] = wl[2][2];
    x[3][i] = wl[2][0];
    x[4][i] = wl[2][1];
    __syncthreads();
    if (!t.owner) return;
    const int l = i - 1, b = i - (TX + 1);
    const bool x0 = t.ex == 0, y0 = t.ey == 0;
    const int64_t n0 = (int64_t)(2 * t.ey) * t.NX + 2 * t.ex, n1 = n0 + t.NX, n2 = n1 + t.NX;
    put(n0, x0 || y0, 0, 0, ((wl[0][0] + x[0][l]) + x[3][b]) + x[2][b - 1]);
    put(n0 + 1, y0, 0, 1, wl[0][1] + x[4][b]);
    put(n1, x0, 1, 0, wl[1][0] + x[1][l]);
    put(n1 + 1, false, 1, 1, wl[1][1]);
    const bool xe = t.ex == P.nx - 1, ye = t.ey == P.ny - 1;
    if (xe) {
        put(n0 + 2, true, 0, 2, T(0));
        put(n1 + 2, true, 1, 2, T(0));
    }
    if (ye) {
        put(n2, true, 2, 0, T(0));
        put(n2 + 1, true, 2, 1, T(0));
        if (xe) put(n2 + 2, true, 2, 2, T(0));
    }
}

}  // namespace femamd
