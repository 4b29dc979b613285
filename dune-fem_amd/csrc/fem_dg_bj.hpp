// Exact element block-Jacobi transform of the SIPG operator with cellwise
// kappa and b = 0: the element block is a Kronecker sum of 1D matrices, so
//   y_e = (Qx (x) Qy (x) Qz) diag(1 / (lx + ly + lz)) (Qx (x) Qy (x) Qz)^T x_e
// with the per-element eigenvectors Qe [3][K][K] (Q_d[r][c] = Qe[d*K2 + r*K + c],
// columns are eigenvectors) and eigenvalues le [3][K].  One element is handled
// by K*K lanes (i, j).  The phases read and rewrite the pencils of one
// direction, which partition the tensor, so only the direction changes need a
// barrier.  An element lies within one wavefront, every lane of which must call
// the transform.  Lanes without an element of their own (wr false) shadow
// another's and write nothing.
#pragma once

#include "fem_dg_sync.hpp"

namespace femamd {

// the transform with the eigen data in LDS (Qs = Qe, le, synchronised), for
// lanes that pass and receive the x pencil y[0..K)[i][j]; A(a, b, c) gives
// the address of a tensor entry in the element's LDS scratch
template <int K, typename T, typename A3>
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
    wave_lds_sync();
    // y: lane (i=a', j=c)
#pragma unroll
    for (int b = 0; b < K; ++b) v[b] = A(i, b, j);
    mul(1, true);
    if (wr)
#pragma unroll
        for (int r = 0; r < K; ++r) A(i, r, j) = tmp[r];
    wave_lds_sync();
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
    wave_lds_sync();
#pragma unroll
    for (int b = 0; b < K; ++b) v[b] = A(i, b, j);
    mul(1, false);
    if (wr)
#pragma unroll
        for (int r = 0; r < K; ++r) A(i, r, j) = tmp[r];
    wave_lds_sync();
#pragma unroll
    for (int a = 0; a < K; ++a) v[a] = A(a, i, j);
    mul(0, false);
#pragma unroll
    for (int r = 0; r < K; ++r) v[r] = tmp[r];
}

}  // namespace femamd
