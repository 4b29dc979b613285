// Exact element block-Jacobi transform of the SIPG operator with cellwise
// kappa and b = 0: the element block is a Kronecker sum of 1D matrices, so
//   y_e = (Qx (x) Qy (x) Qz) diag(1 / (lx + ly + lz)) (Qx (x) Qy (x) Qz)^T x_e
// with the per-element eigenvectors Qe [3][K][K] (Q_d[r][c] = Qe[d*K2 + r*K + c],
// columns are eigenvectors) and eigenvalues le [3][K], read from global
// memory (Qg, lg) into the element's LDS slice Qs [3K^2 + 3K].  One element is
// handled by K*K lanes (i, j); lane (i, j) passes its z pencil x[i][j][0..K)
// in v and receives y[i][j][0..K).  A is the element's K^3 LDS scratch; each
// phase reads and rewrites the pencils of one direction, which partition the
// tensor, so only the direction changes need a barrier.  The transform
// synchronises the group of G lanes that holds the element (one wavefront, or
// the workgroup for G > 64): every lane of it must call it.  Lanes without an
// element of their own (wr false) shadow another's and write nothing: in a
// group of several wavefronts a shadow's write could come between that
// element's reads and writes of the same phase.
#pragma once

#include "fem_dg_sync.hpp"

namespace femamd {

// lanes of one workgroup of the block-Jacobi kernels: EPB elements of K*K lanes
template <int K>
struct BJShape {
    static constexpr int K2 = K * K, K3 = K2 * K, EPB = 64 / K2, THREADS = EPB * K2;
};

// the transform with the eigen data already in Qs (and synchronised), for
// lanes that pass and receive the x pencil y[0..K)[i][j]; A(a, b, c) gives
// the address of a tensor entry in the element's LDS scratch
template <int K, typename T, int G, typename A3>
__device__ __forceinline__ void bj_transform_x(A3 A, const T *Qs, int i, int j, bool wr, T (&v)[K])
{
    constexpr int K2 = K * K;
    const T *Qe = Qs, *le = Qs + 3 * K2;
    T tmp[K];
    // tmp = Q_d^T v (fwd) or Q_d v
    auto mul = [&](int d, bool fwd) {
#pragma unroll
        for (int r = 0; r < K; ++r) {
            T s = 0;
#pragma unroll
            for (int c = 0; c < K; ++c) s = fma(Qe[d * K2 + (fwd ? c * K + r : r * K + c)], v[c], s);
            tmp[r] = s;
        }
    };
    mul(0, true);
    if (wr)
#pragma unroll
        for (int r = 0; r < K; ++r) A(r, i, j) = tmp[r];
    lds_sync<G>();
    // y: lane (i=a', j=c)
#pragma unroll
    for (int b = 0; b < K; ++b) v[b] = A(i, b, j);
    mul(1, true);
    if (wr)
#pragma unroll
        for (int r = 0; r < K; ++r) A(i, r, j) = tmp[r];
    lds_sync<G>();
    // z, scale, back: lane (i=a', j=b')
#pragma unroll
    for (int c = 0; c < K; ++c) v[c] = A(i, j, c);
    mul(2, true);
    const T lij = le[i] + le[K + j];
#pragma unroll
    for (int r = 0; r < K; ++r) v[r] = tmp[r] / (lij + le[2 * K + r]);
    mul(2, false);
    if (wr)
#pragma unroll
        for (int r = 0; r < K; ++r) A(i, j, r) = tmp[r];
    lds_sync<G>();
#pragma unroll
    for (int b = 0; b < K; ++b) v[b] = A(i, b, j);
    mul(1, false);
    if (wr)
#pragma unroll
        for (int r = 0; r < K; ++r) A(i, r, j) = tmp[r];
    lds_sync<G>();
#pragma unroll
    for (int a = 0; a < K; ++a) v[a] = A(a, i, j);
    mul(0, false);
#pragma unroll
    for (int r = 0; r < K; ++r) v[r] = tmp[r];
}

template <int K, typename T, int G = 64>
__device__ __forceinline__ void bj_element(const T *__restrict__ Qg, const T *__restrict__ lg, T *A, T *Qs, int i,
                                           int j, bool wr, T (&v)[K])
{
    constexpr int K2 = K * K;
    // every lane of the element needs all of Qe and le: stage them in LDS once
    // (the element's K*K lanes copy 3K^2 + 3K values) instead of each lane
    // loading them from memory in every pass
    const int t = i * K + j;
    if (wr) {
        for (int k = t; k < 3 * K2; k += K2) Qs[k] = Qg[k];
        for (int k = t; k < 3 * K; k += K2) Qs[3 * K2 + k] = lg[k];
    }
    lds_sync<G>();
    const T *Qe = Qs, *le = Qs + 3 * K2;
    T tmp[K];
    // Q_z^T along c: lane (i=a, j=b)
#pragma unroll
    for (int r = 0; r < K; ++r) {
        T s = 0;
#pragma unroll
        for (int c = 0; c < K; ++c) s = fma(Qe[2 * K2 + c * K + r], v[c], s);
        tmp[r] = s;
    }
    if (wr)
#pragma unroll
        for (int r = 0; r < K; ++r) A[i * K2 + j * K + r] = tmp[r];
    lds_sync<G>();
    // Q_y^T along b: lane (i=a, j=c')
#pragma unroll
    for (int b = 0; b < K; ++b) v[b] = A[i * K2 + b * K + j];
#pragma unroll
    for (int r = 0; r < K; ++r) {
        T s = 0;
#pragma unroll
        for (int b = 0; b < K; ++b) s = fma(Qe[1 * K2 + b * K + r], v[b], s);
        tmp[r] = s;
    }
    if (wr)
#pragma unroll
        for (int r = 0; r < K; ++r) A[i * K2 + r * K + j] = tmp[r];
    lds_sync<G>();
    // Q_x^T along a, scale, Q_x: lane (i=b', j=c')
#pragma unroll
    for (int b = 0; b < K; ++b) v[b] = A[b * K2 + i * K + j];
#pragma unroll
    for (int r = 0; r < K; ++r) {
        T s = 0;
#pragma unroll
        for (int b = 0; b < K; ++b) s = fma(Qe[0 * K2 + b * K + r], v[b], s);
        tmp[r] = s / (le[0 * K + r] + le[1 * K + i] + le[2 * K + j]);
    }
#pragma unroll
    for (int r = 0; r < K; ++r) {
        T s = 0;
#pragma unroll
        for (int b = 0; b < K; ++b) s = fma(Qe[0 * K2 + r * K + b], tmp[b], s);
        v[r] = s;
    }
    if (wr)
#pragma unroll
        for (int r = 0; r < K; ++r) A[r * K2 + i * K + j] = v[r];
    lds_sync<G>();
    // Q_y along b: lane (i=a, j=c')
#pragma unroll
    for (int b = 0; b < K; ++b) v[b] = A[i * K2 + b * K + j];
#pragma unroll
    for (int r = 0; r < K; ++r) {
        T s = 0;
#pragma unroll
        for (int b = 0; b < K; ++b) s = fma(Qe[1 * K2 + r * K + b], v[b], s);
        tmp[r] = s;
    }
    if (wr)
#pragma unroll
        for (int r = 0; r < K; ++r) A[i * K2 + r * K + j] = tmp[r];
    lds_sync<G>();
    // Q_z along c: lane (i=a, j=b)
#pragma unroll
    for (int c = 0; c < K; ++c) v[c] = A[i * K2 + j * K + c];
    lds_sync<G>();   // A is free again for the caller's next element
#pragma unroll
    for (int r = 0; r < K; ++r) {
        T s = 0;
#pragma unroll
        for (int c = 0; c < K; ++c) s = fma(Qe[2 * K2 + r * K + c], v[c], s);
        tmp[r] = s;
    }
#pragma unroll
    for (int r = 0; r < K; ++r) v[r] = tmp[r];
}

}  // namespace femamd
