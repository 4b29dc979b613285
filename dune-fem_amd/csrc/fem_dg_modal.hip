// SIPG DG apply for a coefficient that is constant on each element, in the
// modal basis: no quadrature points.
//
// With the orthonormal Legendre basis the mass matrix of every direction is
// the identity, and with kappa constant on the element (and b, c constant)
// every term of the form acts along one direction only: the volume term is
// the 1D stiffness (and advection) matrix along the pencil, and a face term
// couples the pencil to the one pencil behind the face with the same
// tangential modes.  The (p+1)-point Gauss rules of the reference integrate
// all these products exactly (degree at most 2p), so the result is the
// quadrature form's up to rounding, without its basis passes, collocation
// derivatives and tangential contractions.
//
// One 1D line, with v~_m = P_m v_m, P_m = sqrt(2m+1) the basis at xi = 1 and
// L_m = m(m+1), so that phi_m'(1) = L_m P_m and int phi_m' phi_n' =
// 2 P_m P_n L_min(m,n) for m + n even, int phi_m' phi_n = 2 P_m P_n for n < m,
// m + n odd (0 otherwise):
//   r_m = P_m [ c0 +- ... + L_m c1 -+ ... + 2 kappa |K|/h^2 sum_n L_min v~_n
//               - 2 b |F| sum_{n<m} v~_n ]
// with the face fluxes c0 (against the test trace) and c1 (against its
// derivative) of the two ends.
#include <algorithm>
#include <type_traits>

#include "fem_dg.hpp"
#include "fem_dg_bj.hpp"
#include "fem_dg_sync.hpp"

namespace femamd {

namespace {

constexpr double LP[5] = { 1.0, 1.7320508075688772935, 2.2360679774997896964, 2.6457513110645905905, 3.0 };
constexpr double LL[5] = { 0.0, 2.0, 6.0, 12.0, 20.0 };

template <int K>
struct MShape {
    static constexpr int K2 = K * K, K3 = K * K * K;
    static constexpr int NT = 256;                                 // threads of a workgroup
    // elements of a workgroup, each within one wavefront (the exchanges
    // inside an element then need no workgroup barrier)
    static constexpr int EPW = 64 / K2, EPB = NT / 64 * EPW;
    // LDS tensor of an element: (a, b, c) -> 20 a + 5 b + c at K = 4, where the
    // y and z pencils of its 16 lanes then hit 16 different 8-byte banks (the
    // x pencils 13), a K^2 + b K + c otherwise
    static constexpr int SZ = K == 4 ? 80 : (K3 % 2 ? K3 : K3 + 1);
    static constexpr int SQ = 3 * K2 + 3 * K;                      // eigen data of the element block
};

template <int K>
__device__ __forceinline__ int midx(int a, int b, int c)
{
    if constexpr (K == 4) return 20 * a + 5 * b + c;
    else return a * K * K + b * K + c;
}

// traces of a neighbour's pencil n at the shared face: of the lower neighbour
// (UP false) at its xi = 1, of the upper one at its xi = 0, where phi_m(0) =
// (-1)^m phi_m(1), phi_m'(0) = -(-1)^m phi_m'(1)
template <int K, bool UP, typename T>
__device__ __forceinline__ void nbr_trace(const T *n, T &nv, T &nd)
{
    T v = n[0], d = 0;
#pragma unroll
    for (int m = 1; m < K; ++m) {
        const bool neg = UP && (m & 1);
        v = fma(T(neg ? -LP[m] : LP[m]), n[m], v);
        d = fma(T((UP && !(m & 1)) ? -LP[m] * LL[m] : LP[m] * LL[m]), n[m], d);
    }
    nv = v;
    nd = d;
}

// r = line operator on the pencil v; k: kappa here, ks: behind the two faces
// (k where there is no element), w0, w1: |F| / (2 h), on the boundary |F| / h,
// nv, nd: the neighbours' traces (0 on the boundary); up1, ud1 (may be null):
// the own traces at xi = 1.  The order of the additions is one of several as
// good (errors of 1e-15 and 1e-7), but not free: BiCGStab's step counts are chaotic
// in rounding, and test_gpu_solver.py bounds one of them (207 with this order, 234
// with another; 205 to 231 under changes of 1e-15 of the load)
template <int K, int D, typename T>
__device__ __forceinline__ void line(const ModalArgs<T> &a, T k, const T (&ks)[2], T w0, T w1, const T *v,
                                     const T (&nv)[2], const T (&nd)[2], T *r, T *up1 = nullptr, T *ud1 = nullptr)
{
    T t[K];
    t[0] = v[0];
#pragma unroll
    for (int m = 1; m < K; ++m) t[m] = T(LP[m]) * v[m];
    // sums over the even and odd modes: of v~_m without m = 0 (sh[0]), and of
    // L_m v~_m
    T sh[2] = { T(0), t[1] }, sl[2] = { T(0), T(LL[1]) * t[1] };
    if constexpr (K > 2) {
        sh[0] = t[2];
        sl[0] = T(LL[2]) * t[2];
#pragma unroll
        for (int m = 3; m < K; ++m) {
            sh[m & 1] += t[m];
            sl[m & 1] = fma(T(LL[m]), t[m], sl[m & 1]);
        }
    }
    const T e = K > 2 ? t[0] + sh[0] : t[0], o = sh[1];
    const T u1 = e + o, u0 = e - o, d1 = sl[1] + sl[0], d0 = sl[1] - sl[0];
    if (up1) {
        *up1 = u1;
        *ud1 = d1;
    }
    const T j0 = u0 - nv[0], j1 = u1 - nv[1];
    T c00 = fma(a.pen[D] * (k + ks[0]), j0, w0 * fma(k, d0, ks[0] * nd[0]));
    T c01 = fma(a.pen[D] * (k + ks[1]), j1, -w1 * fma(k, d1, ks[1] * nd[1]));
    const T c10 = w0 * k * j0, c11 = -w1 * k * j1;
    const bool adv = a.b[D] != T(0);
    if (adv) {
        c00 = fma(a.bm[D], u0, fma(-a.bp[D], nv[0], c00));
        c01 = fma(a.bp[D], u1, fma(-a.bm[D], nv[1], c01));
    }
    const T ce = c01 + c00, co = c01 - c00, de = c11 - c10, dd = c11 + c10, kv = k * a.kv[D];
    // sum_n L_min(m,n) v~_n over n of m's parity: L_m sh for the lowest mode
    // of its parity (m = 1, 2), sl for the highest (m = K - 2, K - 1)
    r[0] = ce;
#pragma unroll
    for (int m = 1; m < K; ++m) {
        const T c = (m & 1) ? co : ce, d = (m & 1) ? dd : de;
        if (m + 2 >= K) r[m] = fma(kv, sl[m & 1], fma(T(LL[m]), d, c));
        else r[m] = fma(T(LL[m]), fma(kv, sh[m & 1], d), c);
    }
    if (adv) {
#pragma unroll
        for (int m = 1; m < K; ++m) {
            T q = t[m - 1];
#pragma unroll
            for (int n = m - 3; n >= 0; n -= 2) q += t[n];
            r[m] = fma(-a.ad[D], q, r[m]);
        }
    }
#pragma unroll
    for (int m = 1; m < K; ++m) r[m] *= T(LP[m]);
}

// a workgroup's <u, w> from its lanes' parts, in a fixed summation order
template <int NT>
__device__ __forceinline__ void modal_dot(double acc, double *__restrict__ dot)
{
    __shared__ double wsum[NT / 64];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0;
        for (int k = 0; k < NT / 64; ++k) s += wsum[k];
        dot[blockIdx.x] = s;
    }
}

// w = A u; RES: with a reaction per element, and (rs.rc) the residual r - A u on
// the low modes a, b, c < kc in its place, the restriction to the next DG level
// (compiled apart: the apply keeps its 128 registers at Q4).  A workgroup holds a tile of elements in y and z (K x K lanes
// each) and walks along x.  What bounds it is the traffic to memory and the
// loads in flight, so every value is fetched about once per tile:
//   * lane (b, c) loads the x pencils, whose K loads are K^2 contiguous values
//     each; the x neighbours are the pencils of the step before (kept as two
//     traces) and after (loaded two steps ahead);
//   * y and z lines and their neighbours come from the plane's tile in LDS;
//     an edge element's lanes also load the neighbour behind the edge;
//   * the coefficients of the walk are read once, before it.
// FP64 Q4 at 96^3: 1155 us by quadrature, 870 us with every lane loading its
// six neighbour pencils from memory (7 loads of a vector through the vector
// caches), 550 us so (3.2 TB/s of vectors read and written; 2.2 GB moved per
// apply).  Q3 at 64^3: 115, 79, 67 us; Q2 at 96^3: 287, 183, 144 us.
template <int K, typename T, bool RES>
__global__ void __launch_bounds__(MShape<K>::NT)
    k_dg_modal(const ModalArgs<T> a, const ModalTile mt, const T *__restrict__ u, T *__restrict__ w,
               const int *__restrict__ skip, double *__restrict__ dot, const DGResidual<T> rs)
{
    using S = MShape<K>;
    constexpr int K2 = S::K2, K3 = S::K3, EPB = S::EPB, SZ = S::SZ, NT = S::NT;
    if (skip && *skip) return;
    extern __shared__ __align__(16) unsigned char modal_lds[];
    // the plane's u: the tile's elements, the neighbours behind its edges and
    // a slot of zeros; the y and z parts of the result; the coefficients of
    // each slot along the walk, x0 - 1 .. x1
    const int slots = mt.slots;
    T *const U0 = reinterpret_cast<T *>(modal_lds), *const B0 = U0 + (slots + 1) * SZ, *const K0 = B0 + EPB * SZ;
    const int tid = threadIdx.x;
    const int l = tid & 63;
    bool valid = l < S::EPW * K2;
    const int el = valid ? (tid >> 6) * S::EPW + l / K2 : 0;
    const int i = (l % K2) / K, j = l % K2 % K;
    const int nx = a.n[0], ny = a.n[1], nz = a.n[2];
    const int blk = (int)xcd_remap(blockIdx.x, gridDim.x);
    const int cx = (int)udiv((unsigned)blk, mt.dv_plane), rem = blk - cx * (mt.nty * mt.ntz);
    const int btz = (int)udiv((unsigned)rem, mt.dv_nty), bty = rem - btz * mt.nty;
    const int tz = (int)udiv((unsigned)el, mt.dv_ty), ty = el - tz * mt.ty;
    const int ey = bty * mt.ty + ty, ez = btz * mt.tz + tz;
    valid = valid && tz < mt.tz && ey < ny && ez < nz;
    const int x0 = cx * mt.lx, x1 = x0 + mt.lx < nx ? x0 + mt.lx : nx;
    // neighbours in y and z: inside the tile, or behind its edge (loaded by
    // the edge element's lanes into a slot after the tile's); a tile is at
    // least two elements wide where the mesh is, so an element loads at most
    // one per direction; on the domain boundary the slot of zeros stands in
    // for the values and the own slot for the coefficient
    const bool hy0 = ey > 0, hy1 = ey + 1 < ny, hz0 = ez > 0, hz1 = ez + 1 < nz;
    const int sy = ty == 0 ? 0 : 1, sz = tz == 0 ? 0 : 1;
    const bool ldy = valid && (sy ? (ty + 1 == mt.ty && hy1) : hy0);
    const bool ldz = valid && (sz ? (tz + 1 == mt.tz && hz1) : hz0);
    const int sly = mt.ty * mt.tz + 2 * tz + sy, slz = mt.ty * mt.tz + 2 * mt.tz + 2 * ty + sz;
    const int dy0 = ty > 0 ? -1 : sly - el, dy1 = ty + 1 < mt.ty ? 1 : sly - el;
    const int dz0 = tz > 0 ? -mt.ty : slz - el, dz1 = tz + 1 < mt.tz ? mt.ty : slz - el;
    T *const U = U0 + (valid ? el : slots) * SZ, *const B = B0 + el * SZ;
    T *KS = K0 + (valid ? el : 0) * mt.ks + 1;
    const int oy0 = valid ? (hy0 ? dy0 : slots - el) * SZ : 0, oy1 = valid ? (hy1 ? dy1 : slots - el) * SZ : 0;
    const int oz0 = valid ? (hz0 ? dz0 : slots - el) * SZ : 0, oz1 = valid ? (hz1 ? dz1 : slots - el) * SZ : 0;
    const int my0 = valid && hy0 ? dy0 * mt.ks : 0, my1 = valid && hy1 ? dy1 * mt.ks : 0;
    const int mz0 = valid && hz0 ? dz0 * mt.ks : 0, mz1 = valid && hz1 ? dz1 * mt.ks : 0;
    T *const Hy = U0 + sly * SZ, *const Hz = U0 + slz * SZ;
    const int e = x0 + nx * (ey + ny * ez);
    const int lane = i * K + j;
    unsigned ou = (unsigned)((valid ? e : 0) * K3 + lane);   // (below 2^31: modal_check)
    const int gye = sy ? nx : -nx, gze = sz ? nx * ny : -nx * ny;
    const bool kcell = a.kappa_mode == FEM_KAPPA_CELL;

    // v, vn, vm: the own pencils of this step and the next two; qy, qz: the
    // loaded neighbours' pencils of this step
    T v[K], vn[K], vm[K], qy[K], qz[K];
    T nvl = 0, ndl = 0;   // traces of the element before, at its xi = 1
#pragma unroll
    for (int m = 0; m < K; ++m) v[m] = vn[m] = vm[m] = T(0);
    if (valid) {
        const int xn = x0 + 1 < nx ? 1 : 0;
#pragma unroll
        for (int m = 0; m < K; ++m) v[m] = u[(size_t)ou + m * K2];
        if (xn)
#pragma unroll
            for (int m = 0; m < K; ++m) vn[m] = u[(size_t)ou + m * K2 + K3];
        for (int t = lane; t < x1 - x0 + 2; t += K2) {
            int x = x0 - 1 + t;
            x = x < 0 ? 0 : x < nx ? x : nx - 1;
            KS[t - 1] = kcell ? a.kcell[e + x - x0] : a.kappa_const;
        }
    }
    if (ldy) {
        const T *gy = u + (ou + gye * K3);
#pragma unroll
        for (int m = 0; m < K; ++m) qy[m] = gy[m * K2];
        for (int t = lane; t < x1 - x0; t += K2)
            K0[sly * mt.ks + 1 + t] = kcell ? a.kcell[e + gye + t] : a.kappa_const;
    }
    if (ldz) {
        const T *gz = u + (ou + gze * K3);
#pragma unroll
        for (int m = 0; m < K; ++m) qz[m] = gz[m * K2];
        for (int t = lane; t < x1 - x0; t += K2)
            K0[slz * mt.ks + 1 + t] = kcell ? a.kcell[e + gze + t] : a.kappa_const;
    }
    for (int m = tid; m < SZ; m += NT) U0[slots * SZ + m] = T(0);
    if (valid && x0 > 0) {
        T n[K];
#pragma unroll
        for (int m = 0; m < K; ++m) n[m] = u[(size_t)ou + m * K2 - K3];
        nbr_trace<K, false>(n, nvl, ndl);
    }
    auto L = [&](int a_, int b_, int c_) { return midx<K>(a_, b_, c_); };
    const int inner = (hy0 ? 1 : 0) | (hy1 ? 2 : 0) | (hz0 ? 4 : 0) | (hz1 ? 8 : 0);
    double acc = 0;
    // the loads above have landed before the walk.  Left to the compiler, a wait
    // for them can end up inside the loop, behind the loads for the next step
    // that the step is to hide (64^3 Q4 FP64 165 us, then 171 to 199 us)
#pragma unroll
    for (int m = 0; m < K; ++m) asm volatile("" : "+v"(v[m]), "+v"(vn[m]), "+v"(qy[m]), "+v"(qz[m]));
    for (int x = x0; x < x1; ++x) {
        const bool up = x + 1 < nx, more = x + 1 < x1;
        // (opaque: the boundary weights are formed where they are used, not
        // kept in registers through the walk)
        int in = inner;
        asm volatile("" : "+v"(in));
        auto wf = [&](int d, int bit) { return (in & bit) ? a.w[d] : T(2) * a.w[d]; };
        if (valid) {
#pragma unroll
            for (int m = 0; m < K; ++m) U[L(m, i, j)] = v[m];
        }
        if (ldy) {
#pragma unroll
            for (int m = 0; m < K; ++m) Hy[L(m, i, j)] = qy[m];
        }
        if (ldz) {
#pragma unroll
            for (int m = 0; m < K; ++m) Hz[L(m, i, j)] = qz[m];
        }
        if (more) {
            const T *gy = u + (ou + (gye + 1) * K3), *gz = u + (ou + (gze + 1) * K3);
            if (ldy) {
#pragma unroll
                for (int m = 0; m < K; ++m) qy[m] = gy[m * K2];
            }
            if (ldz) {
#pragma unroll
                for (int m = 0; m < K; ++m) qz[m] = gz[m * K2];
            }
            const bool up2 = x + 2 < nx;
            const T *ue = u + ou;
            if (valid) {
#pragma unroll
                for (int m = 0; m < K; ++m) vm[m] = up2 ? ue[m * K2 + 2 * K3] : T(0);
            }
        }
        __syncthreads();
        {
            // y lines: lane (a, c)
            T p[K], n[K], r[K], nv[2], nd[2];
#pragma unroll
            for (int m = 0; m < K; ++m) n[m] = U[L(i, m, j) + oy0];
            nbr_trace<K, false>(n, nv[0], nd[0]);
#pragma unroll
            for (int m = 0; m < K; ++m) n[m] = U[L(i, m, j) + oy1];
            nbr_trace<K, true>(n, nv[1], nd[1]);
            const T ks[2] = { KS[my0], KS[my1] };
#pragma unroll
            for (int m = 0; m < K; ++m) p[m] = U[L(i, m, j)];
            line<K, 1>(a, KS[0], ks, wf(1, 1), wf(1, 2), p, nv, nd, r);
            if (valid)
#pragma unroll
                for (int m = 0; m < K; ++m) B[L(i, m, j)] = r[m];
        }
        {
            // z lines: lane (a, b)
            T p[K], n[K], r[K], nv[2], nd[2];
#pragma unroll
            for (int m = 0; m < K; ++m) n[m] = U[L(i, j, m) + oz0];
            nbr_trace<K, false>(n, nv[0], nd[0]);
#pragma unroll
            for (int m = 0; m < K; ++m) n[m] = U[L(i, j, m) + oz1];
            nbr_trace<K, true>(n, nv[1], nd[1]);
            const T ks[2] = { KS[mz0], KS[mz1] };
#pragma unroll
            for (int m = 0; m < K; ++m) p[m] = U[L(i, j, m)];
            line<K, 2>(a, KS[0], ks, wf(2, 4), wf(2, 8), p, nv, nd, r);
            wave_lds_sync();
            if (valid)
#pragma unroll
                for (int m = 0; m < K; ++m) B[L(i, j, m)] += r[m];
        }
        T rx[K];
        {
            // x lines in registers: lane (b, c); the pencil behind is the
            // next step's own
            T nv[2] = { nvl, T(0) }, nd[2] = { ndl, T(0) };
            nbr_trace<K, true>(vn, nv[1], nd[1]);
            const T ks[2] = { KS[-1], KS[1] };
#pragma unroll
            for (int m = 0; m < K; ++m) v[m] = U[L(m, i, j)];   // (not kept through the other lines)
            line<K, 0>(a, KS[0], ks, x > 0 ? a.w[0] : T(2) * a.w[0], up ? a.w[0] : T(2) * a.w[0], v, nv, nd, rx,
                       &nvl, &ndl);
            if (a.c != T(0))
#pragma unroll
                for (int m = 0; m < K; ++m) rx[m] = fma(a.cv, v[m], rx[m]);
            if constexpr (RES)
                if (a.ccell) {
                    const T cm = a.vol * a.ccell[valid ? e + x - x0 : 0];
#pragma unroll
                    for (int m = 0; m < K; ++m) rx[m] = fma(cm, v[m], rx[m]);
                }
        }
        wave_lds_sync();
        if (valid)
#pragma unroll
            for (int m = 0; m < K; ++m) rx[m] += B[L(m, i, j)];
        if (RES && rs.rc) {
            const int kc = rs.kc;
            if (valid && i < kc && j < kc) {
                const size_t ex = (size_t)(e + x - x0);
                const T *re = rs.r + ex * K3 + lane;
                T *ce = rs.rc + ex * (kc * kc * kc) + i * kc + j;
#pragma unroll
                for (int m = 0; m < K; ++m)
                    if (m < kc) ce[m * kc * kc] = re[m * K2] - rx[m];
            }
        } else {
            if (valid) {
                T *we = w + ou;
#pragma unroll
                for (int m = 0; m < K; ++m) {
                    we[m * K2] = rx[m];
                    acc += (double)v[m] * (double)rx[m];
                }
            }
        }
#pragma unroll
        for (int m = 0; m < K; ++m) {
            v[m] = vn[m];
            vn[m] = vm[m];
        }
        ++KS;
        ou += K3;
        __syncthreads();
    }
    if (dot) modal_dot<NT>(acc, dot);
}

// 1D passes between the modes of a pencil and its Gauss points, by the parity
// of the basis on the symmetric points: B[K-1-q][a] = (-1)^a B[q][a]
template <int K, typename T>
__device__ __forceinline__ void to_points(const Tab1D<T> &tb, const T (&v)[K], T (&out)[K])
{
#pragma unroll
    for (int q = 0; q < (K + 1) / 2; ++q) {
        T ev = 0, od = 0;
#pragma unroll
        for (int a = 0; a < K; ++a) {
            if (a & 1) od = fma(tb.B[q][a], v[a], od);
            else ev = fma(tb.B[q][a], v[a], ev);
        }
        out[q] = ev + od;
        if (q != K - 1 - q) out[K - 1 - q] = ev - od;
    }
}

template <int K, typename T>
__device__ __forceinline__ void from_points(const Tab1D<T> &tb, const T (&v)[K], T (&out)[K])
{
#pragma unroll
    for (int a = 0; a < K; ++a) {
        T s = (K & 1) ? tb.B[K / 2][a] * v[K / 2] : T(0);
#pragma unroll
        for (int q = 0; q < K / 2; ++q) s = fma(tb.B[q][a], (a & 1) ? v[q] - v[K - 1 - q] : v[q] + v[K - 1 - q], s);
        out[a] = s;
    }
}

// The same lines without the walk: a wavefront holds EPW elements of an x-row
// and every lane loads the six neighbour pencils itself.
//   SM: the sweep xout = u + omega B^-1 (r - A u) of a multigrid level, with the
//     element-block inverse in the same pass; otherwise w = A u, the residual on
//     the low modes (rs.rc), or at Q1 the residual's trilinear functionals at
//     the element's corners (rs.corners, see fem_mg.hip).
//   RX: the reaction at the volume points (cvol and the law), by three passes to
//     the Gauss points and back.
// The sweep needs the registers and the LDS of a walk for the element block
// (48^3 Q3 FP64: the V-cycle with a walking sweep 458 us, with this one 415 us),
// at Q1 a step of a walk is too short for its barriers (48^3: FP64 apply
// 8.6 us against 10.4 us, FP32 6.3 us against 7.5 us), and a mesh thin in y and z
// leaves its lanes idle (dg_modal_walks).
template <int K, typename T, bool SM, bool RX>
__global__ void __launch_bounds__(256)
    k_dg_rows(const ModalArgs<T> a, const ModalRows mr, const ModalReaction<T> vr, const T *__restrict__ u,
              T *__restrict__ w, const int *__restrict__ skip, double *__restrict__ dot, const DGSmooth<T> sm, const DGResidual<T> rs)
{
    using S = MShape<K>;
    constexpr int K2 = S::K2, K3 = S::K3, EPW = S::EPW, R = 4, SZ = S::SZ;
    if (skip && *skip) return;
    __shared__ T smem[R * EPW * (SZ + (SM ? S::SQ : 0))];
    const int g = threadIdx.x >> 6, tid = threadIdx.x & 63;
    const bool wr = tid < EPW * K2;
    const int el = wr ? tid / K2 : 0, i = (tid % K2) / K, j = tid % K2 % K, lane = i * K + j;
    const int nx = a.n[0], ny = a.n[1];
    // x-rows in groups of EPW elements, R rows per workgroup, slabs of about
    // 16 rows in y through all z
    const int blk = (int)xcd_remap(blockIdx.x, gridDim.x);
    const int t = (int)udiv((unsigned)blk, mr.dv_slab), rem = blk - t * (mr.nxg * mr.ty * a.n[2]);
    const int ez = (int)udiv((unsigned)rem, mr.dv_zrow), rem2 = rem - ez * (mr.nxg * mr.ty);
    const int yl = (int)udiv((unsigned)rem2, mr.dv_nxg), xu = rem2 - yl * mr.nxg;
    int ex = xu * EPW + el;
    int ey = (t * mr.ty + yl) * R + g;
    // a wavefront (with a dot, whose sum has a barrier, a whole workgroup)
    // past the last row leaves
    if (dot ? ey - g >= ny : ey >= ny) {
        if (dot && threadIdx.x == 0) dot[blockIdx.x] = 0.0;
        return;
    }
    const bool active = wr && ex < nx && ey < ny;
    ex = ex < nx ? ex : nx - 1;
    ey = ey < ny ? ey : ny - 1;
    const int e = ex + nx * (ey + ny * ez);
    const int ec[3] = { ex, ey, ez };
    const int stride[3] = { 1, nx, nx * ny };
    T *const A = smem + (g * EPW + el) * SZ, *const Q = smem + R * EPW * SZ + (g * EPW + el) * S::SQ;
    auto L = [&](int a_, int b_, int c_) { return midx<K>(a_, b_, c_); };
    // the pencil of element en along d through this lane
    auto pencil = [&](int d, int en, T (&n)[K]) {
        const T *un = u + (size_t)en * K3;
#pragma unroll
        for (int m = 0; m < K; ++m)
            n[m] = un[d == 0 ? m * K2 + lane : d == 1 ? i * K2 + m * K + j : i * K2 + j * K + m];
    };
    T v[K], rr[K];   // own x pencil: lane (b, c)
    pencil(0, e, v);
    bool has[3][2];
    const bool kcell = a.kappa_mode == FEM_KAPPA_CELL;
    const T kin = kcell ? a.kcell[e] : a.kappa_const;
    T ks[3][2], nv[3][2], nd[3][2];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            has[d][s] = s ? ec[d] + 1 < a.n[d] : ec[d] > 0;
            const int en = has[d][s] ? e + (s ? stride[d] : -stride[d]) : e;
            ks[d][s] = kcell ? a.kcell[en] : kin;
            T n[K];
            pencil(d, en, n);
            if (s) nbr_trace<K, true>(n, nv[d][s], nd[d][s]);
            else nbr_trace<K, false>(n, nv[d][s], nd[d][s]);
            nv[d][s] = has[d][s] ? nv[d][s] : T(0);
            nd[d][s] = has[d][s] ? nd[d][s] : T(0);
        }
    }
    T cq[K];
    if constexpr (RX)
#pragma unroll
        for (int q = 0; q < K; ++q) cq[q] = vr.cvol ? vr.cvol[(size_t)e * K3 + i + K * j + K2 * q] : T(0);
    if constexpr (SM) {
        const T *re = sm.r + (size_t)e * K3, *Qg = sm.Q + (size_t)e * 3 * K2, *lg = sm.lam + (size_t)e * 3 * K;
#pragma unroll
        for (int m = 0; m < K; ++m) rr[m] = re[m * K2 + lane];
        if (wr) {
#pragma unroll
            for (int k = 0; k < 3; ++k) Q[k * K2 + lane] = Qg[k * K2 + lane];
            for (int k = lane; k < 3 * K; k += K2) Q[3 * K2 + k] = lg[k];
        }
    }
    if (wr)
#pragma unroll
        for (int m = 0; m < K; ++m) A[L(m, i, j)] = v[m];
    auto wf = [&](int d, int s) { return has[d][s] ? a.w[d] : T(2) * a.w[d]; };
    T p[K], q[K], ry[K], rz[K], rx[K];
    wave_lds_sync();
#pragma unroll
    for (int m = 0; m < K; ++m) p[m] = A[L(i, m, j)];   // lane (a, c)
#pragma unroll
    for (int m = 0; m < K; ++m) q[m] = A[L(i, j, m)];   // lane (a, b)
    line<K, 1>(a, kin, ks[1], wf(1, 0), wf(1, 1), p, nv[1], nd[1], ry);
    wave_lds_sync();
    if (wr)
#pragma unroll
        for (int m = 0; m < K; ++m) A[L(i, m, j)] = ry[m];
    line<K, 2>(a, kin, ks[2], wf(2, 0), wf(2, 1), q, nv[2], nd[2], rz);
    wave_lds_sync();
    if (wr)
#pragma unroll
        for (int m = 0; m < K; ++m) A[L(i, j, m)] += rz[m];
    line<K, 0>(a, kin, ks[0], wf(0, 0), wf(0, 1), v, nv[0], nd[0], rx);
    if (a.c != T(0))
#pragma unroll
        for (int m = 0; m < K; ++m) rx[m] = fma(a.cv, v[m], rx[m]);
    if (a.ccell) {
        const T cm = a.vol * a.ccell[e];
#pragma unroll
        for (int m = 0; m < K; ++m) rx[m] = fma(cm, v[m], rx[m]);
    }
    wave_lds_sync();
#pragma unroll
    for (int m = 0; m < K; ++m) rx[m] += A[L(m, i, j)];
    if constexpr (RX) {
        // int (cvol + coef u^pw) u v
        const Tab1D<T> &tb = *vr.tab;
        T f[K], h[K];
        auto put = [&](int d, const T (&x)[K]) {
            if (wr)
#pragma unroll
                for (int m = 0; m < K; ++m) A[d == 0 ? L(m, i, j) : d == 1 ? L(i, m, j) : L(i, j, m)] = x[m];
            wave_lds_sync();
        };
        auto get = [&](int d, T (&x)[K]) {
#pragma unroll
            for (int m = 0; m < K; ++m) x[m] = A[d == 0 ? L(m, i, j) : d == 1 ? L(i, m, j) : L(i, j, m)];
            wave_lds_sync();
        };
        to_points<K>(tb, v, f);
        wave_lds_sync();
        put(0, f);
        get(1, f);
        to_points<K>(tb, f, h);
        put(1, h);
        get(2, f);
        to_points<K>(tb, f, h);
        const T wij = a.vol * tb.w[i] * tb.w[j];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            T c = cq[k];
            if (vr.nl_pow) {
                T pw = vr.nl_coef;
                for (int n = 0; n < vr.nl_pow; ++n) pw *= h[k];
                c += pw;
            }
            f[k] = wij * tb.w[k] * c * h[k];
        }
        from_points<K>(tb, f, h);
        put(2, h);
        get(1, f);
        from_points<K>(tb, f, h);
        put(1, h);
        get(0, f);
        from_points<K>(tb, f, h);
#pragma unroll
        for (int m = 0; m < K; ++m) rx[m] += h[m];
    }
    if constexpr (!SM) {
        if (rs.rc) {
            const int kc = rs.kc;
            if (active && i < kc && j < kc) {
                const T *re = rs.r + (size_t)e * K3 + lane;
                T *ce = rs.rc + (size_t)e * (kc * kc * kc) + i * kc + j;
#pragma unroll
                for (int m = 0; m < K; ++m)
                    if (m < kc) ce[m * kc * kc] = re[m * K2] - rx[m];
            }
            return;
        }
        if constexpr (K == 2)
            if (rs.corners) {
                // the residual's modes in FP64, then this lane's two corners
                // (0, i, j) and (1, i, j)
                __shared__ double cs[R * EPW * 8];
                double *C = cs + (g * EPW + el) * 8;
                const T *re = rs.r + (size_t)e * K3 + lane;
#pragma unroll
                for (int m = 0; m < 2; ++m) C[m * 4 + lane] = (double)re[m * K2] - (double)rx[m];
                wave_lds_sync();
                const double s1 = 0.28867513459481287;   // 1 / (2 sqrt 3)
                const double ti = i ? s1 : -s1, tj = j ? s1 : -s1;
                double x[2];
#pragma unroll
                for (int m = 0; m < 2; ++m)
                    x[m] = 0.5 * (0.5 * C[m * 4] + tj * C[m * 4 + 1]) + ti * (0.5 * C[m * 4 + 2] + tj * C[m * 4 + 3]);
                if (active) {
                    double *ce = rs.corners + (size_t)e * 8 + 2 * i + 4 * j;
                    ce[0] = 0.5 * x[0] - s1 * x[1];
                    ce[1] = 0.5 * x[0] + s1 * x[1];
                }
                return;
            }
        double acc = 0;
        if (active) {
            T *we = w + (size_t)e * K3 + lane;
#pragma unroll
            for (int m = 0; m < K; ++m) {
                we[m * K2] = rx[m];
                acc += (double)v[m] * (double)rx[m];
            }
        }
        if (dot) modal_dot<256>(acc, dot);
        return;
    }
#pragma unroll
    for (int m = 0; m < K; ++m) rx[m] = rr[m] - rx[m];
    wave_lds_sync();
    bj_transform_x<K, T>([&](int a_, int b_, int c_) -> T & { return A[L(a_, b_, c_)]; }, Q, i, j, wr, rx);
    if (active) {
        T *xe = sm.xout + (size_t)e * K3 + lane;
#pragma unroll
        for (int m = 0; m < K; ++m) xe[m * K2] = fma(sm.omega, rx[m], v[m]);
    }
}

// y = (ADD ? y : 0) + omega B^-1 (x - t), t may be null; four wavefronts of
// EPW elements each.  dot (may be null): the workgroup's <x, y> and <x, x>.
// Reads and writes the vectors once and the eigen data (3 K^2 + 3 K values per
// element) once, which is what bounds it.
template <int K, typename T, bool ADD, bool DOT>
__global__ void __launch_bounds__(256)
    k_dg_block(int64_t E, const T *__restrict__ Qg, const T *__restrict__ lg, const T *__restrict__ x,
               const T *__restrict__ t, T *__restrict__ y, T omega, const int *__restrict__ skip,
               double *__restrict__ dot)
{
    using S = MShape<K>;
    constexpr int K2 = S::K2, K3 = S::K3, EPW = S::EPW, R = 4, SZ = S::SZ;
    if (skip && *skip) return;
    __shared__ T smem[R * EPW * (SZ + S::SQ)];
    const int g = threadIdx.x >> 6, tid = threadIdx.x & 63;
    const bool wr = tid < EPW * K2;
    const int el = wr ? tid / K2 : 0, i = (tid % K2) / K, j = tid % K2 % K, lane = i * K + j;
    const int64_t e_raw = ((int64_t)blockIdx.x * R + g) * EPW + el;
    const bool active = wr && e_raw < E;
    const int64_t e = e_raw < E ? e_raw : E - 1;
    T *const A = smem + (g * EPW + el) * SZ, *const Q = smem + R * EPW * SZ + (g * EPW + el) * S::SQ;
    const T *xe = x + e * K3 + lane;
    T v[K], xv[K];
#pragma unroll
    for (int m = 0; m < K; ++m) xv[m] = v[m] = xe[m * K2];
    if constexpr (ADD) {
        const T *te = t + e * K3 + lane;
#pragma unroll
        for (int m = 0; m < K; ++m) v[m] -= te[m * K2];
    }
    if (wr) {
        const T *Qe = Qg + e * 3 * K2, *le = lg + e * 3 * K;
#pragma unroll
        for (int k = 0; k < 3; ++k) Q[k * K2 + lane] = Qe[k * K2 + lane];
        for (int k = lane; k < 3 * K; k += K2) Q[3 * K2 + k] = le[k];
    }
    wave_lds_sync();
    bj_transform_x<K, T>([&](int a_, int b_, int c_) -> T & { return A[midx<K>(a_, b_, c_)]; }, Q, i, j, wr, v);
    double a1 = 0, a2 = 0;
    if (active) {
        T *ye = y + e * K3 + lane;
#pragma unroll
        for (int m = 0; m < K; ++m) {
            const T r = ADD ? fma(omega, v[m], ye[m * K2]) : omega * v[m];
            ye[m * K2] = r;
            if constexpr (DOT) {
                a1 += (double)xv[m] * (double)r;
                a2 += (double)xv[m] * (double)xv[m];
            }
        }
    }
    if constexpr (DOT) {
        modal_dot<256>(a1, dot);
        __syncthreads();
        modal_dot<256>(a2, dot + gridDim.x);
    }
}

template <typename T>
ModalArgs<T> modal_args(const DGPlan<T> &p)
{
    ModalArgs<T> a = p.modal;
    a.kappa_mode = p.kappa_mode;
    a.kappa_const = p.kappa_const;
    a.kcell = p.kcell;
    a.ccell = p.ccell;
    return a;
}

template <int K, typename T, bool SM>
void launch_rows(const DGPlan<T> &p, const T *u, T *w, const DGSmooth<T> &sm, const DGResidual<T> &rs, const int *skip,
                 hipStream_t s, double *dot)
{
    const ModalReaction<T> vr{ p.cvol, p.nl_coef, p.nl_pow, p.tab };
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)p.rows.blocks), dim3(256), 0, s, modal_args(p), p.rows, vr, u, w, skip,
                           dot, sm, rs);
    };
    if (p.cvol || p.nl_pow) go(k_dg_rows<K, T, SM, true>);
    else go(k_dg_rows<K, T, SM, false>);
}

template <int K, typename T>
void launch_apply(const DGPlan<T> &p, const T *u, T *w, const DGResidual<T> &rs, const int *skip, hipStream_t s,
                  double *dot)
{
    if (!p.walks || p.cvol || p.nl_pow) {
        launch_rows<K, T, false>(p, u, w, DGSmooth<T>{}, rs, skip, s, dot);
    } else if constexpr (K > 2) {
        using S = MShape<K>;
        const ModalTile &t = p.tile;
        const size_t lds = sizeof(T) * ((size_t)(t.slots + 1 + S::EPB) * S::SZ + (size_t)t.slots * t.ks);
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3((unsigned)t.blocks), dim3(S::NT), lds, s, modal_args(p), t, u, w, skip, dot,
                               rs);
        };
        if (rs.rc || p.ccell) go(k_dg_modal<K, T, true>);
        else go(k_dg_modal<K, T, false>);
    }
}

template <int K, typename T>
void launch_sweep(const DGPlan<T> &p, const T *u, const DGSmooth<T> &sm, const int *skip, hipStream_t s)
{
    launch_rows<K, T, true>(p, u, nullptr, sm, DGResidual<T>{}, skip, s, nullptr);
}

#define MODAL_SWITCH(CALL)                                                             \
    switch (k) {                                                                       \
    case 2: CALL(2); break;                                                            \
    case 3: CALL(3); break;                                                            \
    case 4: CALL(4); break;                                                            \
    case 5: CALL(5); break;                                                            \
    default: throw Error(FEM_ERR_UNSUPPORTED, "DG: order must be 1..4");               \
    }                                                                                  \
    FEM_HIP(hipGetLastError())

template <typename T>
void modal_check(const DGPlan<T> &a, int k)
{
    FEM_CHECK((int64_t)a.n[0] * a.n[1] * a.n[2] * k * k * k < (int64_t)1 << 31, FEM_ERR_UNSUPPORTED,
              "DG apply: more than 2^31 DoFs");
}

template <typename T>
void modal_apply(const DGPlan<T> &a, int k, const T *u, T *w, const DGResidual<T> &rs, const int *skip, hipStream_t s,
                 double *dot)
{
    modal_check(a, k);
    FEM_CHECK(!rs.corners || k == 2, FEM_ERR_ARG, "corner functionals: Q1 only");
#define CALL(KK) launch_apply<KK, T>(a, u, w, rs, skip, s, dot)
    MODAL_SWITCH(CALL);
#undef CALL
}

template <typename T>
void modal_smooth(const DGPlan<T> &a, int k, const T *u, const DGSmooth<T> &sm, const int *skip, hipStream_t s)
{
    modal_check(a, k);
    FEM_CHECK(dg_is_modal(a), FEM_ERR_UNSUPPORTED, "smoothing sweep: cellwise or constant kappa");
    FEM_CHECK(sm.r && sm.Q && sm.lam && sm.xout && sm.xout != u, FEM_ERR_ARG,
              "smoothing sweep: r, eigen data and an output other than the input");
#define CALL(KK) launch_sweep<KK, T>(a, u, sm, skip, s)
    MODAL_SWITCH(CALL);
#undef CALL
}

template <int K, typename T>
void launch_block(int64_t E, const T *Q, const T *lam, const T *x, const T *t, T *y, T omega, bool add,
                  const int *skip, hipStream_t s, double *dot)
{
    const unsigned nb = (unsigned)dg_bj_blocks(K, E);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(nb), dim3(256), 0, s, E, Q, lam, x, t, y, omega, skip, dot);
    };
    if (add) go(k_dg_block<K, T, true, false>);
    else if (dot) go(k_dg_block<K, T, false, true>);
    else go(k_dg_block<K, T, false, false>);
}

}  // namespace

ModalTile dg_modal_tile(int k, const int *n)
{
    FEM_CHECK(k >= 2 && k <= 5, FEM_ERR_UNSUPPORTED, "DG: order must be 1..4");
    ModalTile t;
    const int epb = 4 * (64 / (k * k));
    // the tile with the fewest lanes without an element and the shortest edge
    // (an edge element costs a second load of it); at least two elements in
    // each direction where the mesh has them (see k_dg_modal)
    double best = 0;
    for (int ty = n[1] > 1 ? 2 : 1; ty <= n[1] && ty <= epb; ++ty) {
        const int tz = std::min(epb / ty, n[2]);
        if (tz < std::min(2, n[2])) break;
        const int nty = (n[1] + ty - 1) / ty, ntz = (n[2] + tz - 1) / tz;
        const double cost = (double)nty * ntz * (epb + 0.5 * (ty + tz));
        if (best == 0 || cost < best) {
            best = cost;
            t.ty = ty;
            t.tz = tz;
            t.nty = nty;
            t.ntz = ntz;
        }
    }
    t.slots = t.ty * t.tz + 2 * (t.ty + t.tz);
    // walks of up to 16 steps, as long as 2048 of them are left to run (a
    // chip holds 768 to 1536 at a time): walks of 1, 2, 4, 8 steps give 800,
    // 687, 629, 600 us at 96^3 Q4, and 6.6, 7.3, 9.1, 14.8 us at 24^3 Q2
    const int64_t tiles = (int64_t)t.nty * t.ntz;
    const int most = (int)std::min<int64_t>(16, (tiles * n[0] + 2047) / 2048);
    t.ncx = (n[0] + most - 1) / most;
    t.lx = (n[0] + t.ncx - 1) / t.ncx;
    t.ncx = (n[0] + t.lx - 1) / t.lx;
    t.ks = (t.lx + 2) | 1;
    t.blocks = tiles * t.ncx;
    t.dv_ty = make_udiv((unsigned)t.ty);
    t.dv_nty = make_udiv((unsigned)t.nty);
    t.dv_plane = make_udiv((unsigned)tiles);
    return t;
}

// Q1 steps are too short for a walk (see k_dg_rows).  Otherwise the walk, if at
// least half of a tile's elements exist: on a mesh thin in y and z a workgroup
// walks along x with few lanes at work, and nothing is left to share through
// LDS.  Q3 FP64, 20000 x 1 x 1 elements (1/16 of a tile): 46 us walking, 10.6 us by
// rows; 60000 x 2 x 2 (1/4): 135 and 75 us; 60000 x 3 x 3 (9/16): 190 and 230 us.
// At Q2 the same meshes have 1/28, 1/7 and 9/28 of a tile: 31.7 and 6.7, 97 and 42, 113
// and 80 us; Q4 1/8, 1/2 and 9/16: 58 and 20, 221 and 243, 528 and 559 us.  Idle
// lanes cost nothing while all workgroups run at once (768 do at three per CU):
// 700 x 6 x 1 Q3 5.0 and 5.2 us, 1600 x 3 x 3 Q2 7.7 and 5.9 us.
bool dg_modal_walks(int k, const int *n, const ModalTile &t)
{
    const int64_t epb = 4 * (64 / (k * k));
    return k > 2 && (2 * (int64_t)n[1] * n[2] >= (int64_t)t.nty * t.ntz * epb || t.blocks <= 768);
}

ModalRows dg_modal_rows(int k, const int *n)
{
    ModalRows r;
    const int epw = 64 / (k * k), yb = (n[1] + 3) / 4;
    r.nxg = (n[0] + epw - 1) / epw;
    r.ty = (yb + (yb + 3) / 4 - 1) / ((yb + 3) / 4);
    r.blocks = (int64_t)r.nxg * r.ty * ((yb + r.ty - 1) / r.ty) * n[2];
    r.dv_slab = make_udiv((unsigned)(r.nxg * r.ty * n[2]));
    r.dv_zrow = make_udiv((unsigned)(r.nxg * r.ty));
    r.dv_nxg = make_udiv((unsigned)r.nxg);
    return r;
}

int64_t dg_modal_blocks(int k, const int *n, bool reaction)
{
    const ModalTile t = dg_modal_tile(k, n);
    return reaction || !dg_modal_walks(k, n, t) ? dg_modal_rows(k, n).blocks : t.blocks;
}

int64_t dg_bj_blocks(int k, int64_t E)
{
    FEM_CHECK(k >= 2 && k <= 5, FEM_ERR_UNSUPPORTED, "DG: order must be 1..4");
    const int epb = 4 * (64 / (k * k));
    return (E + epb - 1) / epb;
}

template <typename T>
void dg_block_apply(int k, int64_t E, const T *Q, const T *lam, const T *x, const T *t, T *y, T omega, bool add,
                    const int *skip, hipStream_t s, double *dot)
{
#define CALL(KK) launch_block<KK, T>(E, Q, lam, x, t, y, omega, add, skip, s, dot)
    MODAL_SWITCH(CALL);
#undef CALL
}
template void dg_block_apply<double>(int, int64_t, const double *, const double *, const double *, const double *,
                                     double *, double, bool, const int *, hipStream_t, double *);
template void dg_block_apply<float>(int, int64_t, const float *, const float *, const float *, const float *, float *,
                                    float, bool, const int *, hipStream_t, double *);

void dg_modal_apply_f64(const DGPlan<double> &a, int k, const double *u, double *w, const int *skip, hipStream_t s,
                        double *dot)
{
    modal_apply<double>(a, k, u, w, DGResidual<double>{}, skip, s, dot);
}
void dg_modal_apply_f32(const DGPlan<float> &a, int k, const float *u, float *w, const int *skip, hipStream_t s,
                        double *dot)
{
    modal_apply<float>(a, k, u, w, DGResidual<float>{}, skip, s, dot);
}
void dg_modal_residual_f64(const DGPlan<double> &a, int k, const double *u, const DGResidual<double> &rs,
                           const int *skip, hipStream_t s)
{
    modal_apply<double>(a, k, u, nullptr, rs, skip, s, nullptr);
}
void dg_modal_residual_f32(const DGPlan<float> &a, int k, const float *u, const DGResidual<float> &rs, const int *skip,
                           hipStream_t s)
{
    modal_apply<float>(a, k, u, nullptr, rs, skip, s, nullptr);
}
void dg_modal_smooth_f64(const DGPlan<double> &a, int k, const double *u, const DGSmooth<double> &sm, const int *skip,
                         hipStream_t s)
{
    modal_smooth<double>(a, k, u, sm, skip, s);
}
void dg_modal_smooth_f32(const DGPlan<float> &a, int k, const float *u, const DGSmooth<float> &sm, const int *skip,
                         hipStream_t s)
{
    modal_smooth<float>(a, k, u, sm, skip, s);
}

}  // namespace femamd
