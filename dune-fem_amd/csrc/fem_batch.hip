// Batched solves of many independent continuous-Q2 problems of different
// sizes in one set of launches.
//
// No reference counterpart: the reference solves one problem per
// FemScheme::solve call (dune/fem/schemes/femscheme.hh:195-253).  Each
// instance here follows the same CG recurrence as the single-instance solver
// (LinearSolver::cg, dune/fem/solver/linear/cg.hh:19-117, Jacobi
// preconditioned) with its own scalars, inside an FP64 iterative-refinement
// loop; instances that have converged are masked out of every launch.
//
// Layout: all instances' DoFs are concatenated (dof_off), their elements too
// (elem_off, coefficient arrays [E][9]).  Reductions are segmented: every
// workgroup belongs to one instance and writes its partial, and the workgroups of
// the kernel that needs the sum add that instance's partials in a fixed order.
// One inner CG step is two launches; a few steps are captured in a HIP graph.  Most
// batches are a few hundred workgroups per kernel, so a step costs what its chain of
// launches and dependent loads costs: 24 instances of 32 to 128 elements a side
// (616k DoFs) 32 us in four launches whose sums the last workgroup of an instance
// finished behind atomics, now 16.7 us (apply 8.3, update 6.1).
#include <algorithm>
#include <chrono>
#include <cmath>

#include "fem_batch.hpp"
#include "fem_blas.hpp"
#include "fem_cg_tile.hpp"

namespace femamd {

constexpr int SEG_THREADS = 256;
constexpr int SEG_ITEMS = 4;     // DoFs in flight per thread
constexpr int SEG_CHUNK = SEG_THREADS * SEG_ITEMS;
// segments of an instance at most: each workgroup of its apply sums their partials,
// as each segment sums those of the instance's tiles, in L2 (one instance of 1024^2
// elements 58 us a step, 2048^2 282 us, 4096^2 1128 us: 14 to 17 ns per 1000 DoFs)
constexpr int SEG_MOST = 1024;
constexpr int GRAPH_STEPS = 8;   // steps per captured graph (even: q has two buffers)

struct SegTab {
    const int *inst;       // [nseg] instance of each segment
    const int64_t *lo;     // [nseg] first DoF
    const int64_t *hi;     // [nseg] one past the last DoF
    const int *first;      // [count + 1] first segment of each instance
    double *parts;         // [2][nseg]
};

// per-instance scalars (device arrays).  No kernel reads what one of its own
// workgroups writes: res (<p, s>) and done are set by the apply and read by the
// update that follows; prev (that of the step before), it and idle (done, as the
// applies after it see it) are set by the update and read by the apply.
struct BState {
    double *res, *prev, *tol, *rn, *bn2, *scale, *eps2;
    int *it, *done, *idle, *conv, *maxit;
};

// the sums of the instance's partials a[lo .. hi) and b[lo .. hi), in every thread,
// for every workgroup of NT threads alike; two barriers
template <int NT, int NQ>
__device__ __forceinline__ void seg_sum(const double *__restrict__ a, const double *__restrict__ b, int lo, int hi,
                                        double *lds, double (&sum)[NQ])
{
    double v[NQ] = {};
#pragma unroll 4
    for (int k = lo + (int)threadIdx.x; k < hi; k += NT) {
        v[0] += a[k];
        if constexpr (NQ > 1) v[1] += b[k];
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) v[q] += __shfl_xor(v[q], off, 64);
        if ((threadIdx.x & 63) == 0) lds[q * (NT / 64) + (threadIdx.x >> 6)] = v[q];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        sum[q] = 0;
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) sum[q] += lds[q * (NT / 64) + w];
    }
    __syncthreads();
}

// the workgroup's sums of v, to parts[q * stride]
template <int NT, int NQ>
__device__ __forceinline__ void seg_part(double (&v)[NQ], double *lds, double *parts, int stride)
{
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) v[q] += __shfl_xor(v[q], off, 64);
        if ((threadIdx.x & 63) == 0) lds[q * (NT / 64) + (threadIdx.x >> 6)] = v[q];
    }
    __syncthreads();
    if (threadIdx.x < NQ) {
        double s = 0;
        for (int w = 0; w < NT / 64; ++w) s += lds[threadIdx.x * (NT / 64) + w];
        parts[(size_t)threadIdx.x * stride] = s;
    }
}

// f(i, k): the loads of DoF i into slot k; g(i, k): its update
template <typename F, typename G>
__device__ __forceinline__ void seg_loop(int64_t lo, int64_t hi, F f, G g)
{
    for (int64_t i0 = lo; i0 < hi; i0 += SEG_CHUNK) {
#pragma unroll
        for (int k = 0; k < SEG_ITEMS; ++k) {
            const int64_t i = i0 + threadIdx.x + (int64_t)k * SEG_THREADS;
            f(i < hi ? i : lo, k);
        }
#pragma unroll
        for (int k = 0; k < SEG_ITEMS; ++k) {
            const int64_t i = i0 + threadIdx.x + (int64_t)k * SEG_THREADS;
            if (i < hi) g(i, k);
        }
    }
}

// start of an inner solve: p = scale r (FP32), s = dinv p, x = 0; partials of
// <p, s>, <p, p>
__global__ void __launch_bounds__(SEG_THREADS)
    k_bcg_init(SegTab S, BState B, const double *__restrict__ r, const float *__restrict__ dinv, float *__restrict__ x,
               float *__restrict__ p, float *__restrict__ s, double eps, int maxit)
{
    __shared__ double lds[2 * SEG_THREADS / 64];
    const int inst = S.inst[blockIdx.x];
    const bool skip = B.conv[inst] != 0;
    if (threadIdx.x == 0) {
        if (blockIdx.x == 0) {
            *B.eps2 = eps * eps;   // relative reduction of the true residual
            *B.maxit = maxit;
        }
        if (S.first[inst] == (int)blockIdx.x) {
            B.done[inst] = B.idle[inst] = skip;
            B.it[inst] = 0;
        }
    }
    if (skip) return;   // uniform over the block
    const double a = B.scale[inst];
    double v[2] = {};
    double vr[SEG_ITEMS];
    float vd[SEG_ITEMS];
    seg_loop(S.lo[blockIdx.x], S.hi[blockIdx.x],
             [&](int64_t i, int k) {
                 vr[k] = r[i];
                 vd[k] = dinv[i];
             },
             [&](int64_t i, int k) {
                 const float b = (float)(vr[k] * a), sv = vd[k] * b;
                 x[i] = 0.f;
                 p[i] = b;
                 s[i] = sv;
                 v[0] += (double)b * (double)sv;
                 v[1] += (double)b * (double)b;
             });
    seg_part<SEG_THREADS, 2>(v, lds, S.parts + blockIdx.x, gridDim.x);
}

// first half of a step: the end of the last one (<p, s>, <p, p>, whether the
// instance is done, beta), q = s + beta q on the way into the apply, h = A q and the
// partials of <q, h>.  The nodes of an element are combined as they are read, by up
// to four elements, so the new q goes to a second buffer.
template <int TX, int TY>
__global__ void __launch_bounds__((TX + 1) * (TY + 1))
    k_bcg_apply(SegTab S, BState B, const CGInst *__restrict__ insts, const int *__restrict__ tile_inst,
                const float *__restrict__ kvol, const float *__restrict__ s, const float *__restrict__ q,
                float *__restrict__ qn, float *__restrict__ h, double *__restrict__ dot, int nseg)
{
    constexpr int NT = (TX + 1) * (TY + 1);
    __shared__ float xch[5][NT];
    __shared__ double lds[2 * ((NT + 63) / 64)];
    const int bid = (int)xcd_remap(blockIdx.x, gridDim.x);
    const int ii = tile_inst[bid];
    if (B.idle[ii]) return;
    const CGInst P = insts[ii];
    const CGTile t = cg_tile<TX, TY>(P, bid);
    const int it = B.it[ii];
    float ul[3][3] = {}, uo[3][3] = {}, wl[3][3] = {}, kap[9] = {};
    const int64_t e = P.elem_off + (int64_t)t.ey * P.nx + t.ex;
    if (t.valid) {
        const float *se = s + P.dof_off, *qe = q + P.dof_off;
#pragma unroll
        for (int iy = 0; iy < 3; ++iy)
#pragma unroll
            for (int ix = 0; ix < 3; ++ix) {
                const int64_t n = (int64_t)(2 * t.ey + iy) * t.NX + 2 * t.ex + ix;
                ul[iy][ix] = se[n];
                if (it) uo[iy][ix] = qe[n];
            }
#pragma unroll
        for (int k = 0; k < 9; ++k) kap[k] = kvol[e * 9 + k];
    }
    double r[2];
    seg_sum<NT, 2>(S.parts, S.parts + nseg, S.first[ii], S.first[ii + 1], lds, r);
    const double tol = it ? B.tol[ii] : *B.eps2 * r[1];
    const bool done = !(r[1] > tol) || it >= *B.maxit;
    const double beta = it ? r[0] / B.prev[ii] : 0.0;
    if (bid == P.tile_off && threadIdx.x == 0) {
        B.res[ii] = r[0];
        B.done[ii] = done;
        if (!it) B.tol[ii] = tol;
    }
    if (done) return;
    if (it)
#pragma unroll
        for (int iy = 0; iy < 3; ++iy)
#pragma unroll
            for (int ix = 0; ix < 3; ++ix) ul[iy][ix] = (float)(beta * (double)uo[iy][ix] + (double)ul[iy][ix]);
    if (t.valid) {
        const float c = (float)P.c * (float)P.detJ;
        cg_element<float, true>(ul, kap, (float)P.sx, (float)P.sy, [&](float, int) { return c; }, wl);
    }
    float *he = h + P.dof_off, *qo = qn + P.dof_off;
    double d[1] = {};
    cg_gather<TX, TY, float>(P, t, wl, xch, [&](int64_t node, bool bnd, int iy, int ix, float v) {
        if (bnd) v = ul[iy][ix];
        he[node] = v;
        qo[node] = ul[iy][ix];
        d[0] += (double)ul[iy][ix] * (double)v;
    });
    seg_part<NT, 1>(d, lds, dot + bid, 0);
}

// second half: alpha = <p, s> / <q, h>, x += alpha q, p -= alpha h, s = dinv p, and
// the partials of <p, s>, <p, p>
__global__ void __launch_bounds__(SEG_THREADS)
    k_bcg_update(SegTab S, BState B, const int *__restrict__ tile_first, const double *__restrict__ dot,
                 const float *__restrict__ dinv, const float *__restrict__ q, const float *__restrict__ h,
                 float *__restrict__ x, float *__restrict__ p, float *__restrict__ s)
{
    __shared__ double lds[2 * SEG_THREADS / 64];
    const int inst = S.inst[blockIdx.x];
    if (B.done[inst]) {
        if (S.first[inst] == (int)blockIdx.x && threadIdx.x == 0) B.idle[inst] = 1;
        return;
    }
    float vp[SEG_ITEMS], vh[SEG_ITEMS], vd[SEG_ITEMS], vx[SEG_ITEMS], vq[SEG_ITEMS];
    const int64_t lo = S.lo[blockIdx.x], hi = S.hi[blockIdx.x];
    double qh[1], v[2] = {};
    seg_sum<SEG_THREADS, 1>(dot, nullptr, tile_first[inst], tile_first[inst + 1], lds, qh);
    const double res = B.res[inst], alpha = res / qh[0];
    if (S.first[inst] == (int)blockIdx.x && threadIdx.x == 0) {
        B.prev[inst] = res;
        B.it[inst] += 1;
    }
    seg_loop(lo, hi,
             [&](int64_t i, int k) {
                 vp[k] = p[i];
                 vh[k] = h[i];
                 vd[k] = dinv[i];
                 vx[k] = x[i];
                 vq[k] = q[i];
             },
             [&](int64_t i, int k) {
                 x[i] = (float)((double)vx[k] + alpha * (double)vq[k]);
                 const float pn = (float)((double)vp[k] - alpha * (double)vh[k]), sv = vd[k] * pn;
                 p[i] = pn;
                 s[i] = sv;
                 v[0] += (double)pn * (double)sv;
                 v[1] += (double)pn * (double)pn;
             });
    seg_part<SEG_THREADS, 2>(v, lds, S.parts + blockIdx.x, gridDim.x);
}

// the sum of part[lo .. hi) by one wavefront
__device__ __forceinline__ double wave_parts(const double *part, int lo, int hi)
{
    double v = 0;
    for (int k = lo + (int)(threadIdx.x & 63); k < hi; k += 64) v += part[k];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// the instances still at work, a wavefront per instance: RES64 = false, after a
// step (the test of the next apply); true, after the residual (rn, bn2, conv, scale)
template <bool RES64>
__global__ void __launch_bounds__(1024) k_batch_look(SegTab S, BState B, int count, int nseg, double eps, int *out)
{
    __shared__ int active;
    if (threadIdx.x == 0) active = 0;
    __syncthreads();
    for (int i = threadIdx.x >> 6; i < count; i += 1024 / 64) {
        const double a = wave_parts(S.parts, S.first[i], S.first[i + 1]),
                     b = wave_parts(S.parts + nseg, S.first[i], S.first[i + 1]);
        if ((threadIdx.x & 63) != 0) continue;
        if (RES64) {
            if (!B.conv[i]) {
                const double rn = sqrt(a);
                B.rn[i] = rn;
                B.bn2[i] = b;
                B.conv[i] = rn <= eps * sqrt(b);
                B.scale[i] = rn > 0 ? 1.0 / rn : 1.0;
            }
            if (!B.conv[i]) atomicAdd(&active, 1);
        } else if (!B.done[i]) {
            if (!(b > B.tol[i]) || B.it[i] >= *B.maxit) B.done[i] = B.idle[i] = 1;
            else atomicAdd(&active, 1);
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) *out = active;
}

// r = b - h (FP64) and the partials of <r, r>, <b, b>
__global__ void __launch_bounds__(SEG_THREADS)
    k_seg_res64(SegTab S, BState B, const double *__restrict__ b, const double *__restrict__ h, double *__restrict__ r)
{
    __shared__ double lds[2 * SEG_THREADS / 64];
    if (B.conv[S.inst[blockIdx.x]]) return;
    double vb[SEG_ITEMS], vh[SEG_ITEMS], v[2] = {};
    seg_loop(S.lo[blockIdx.x], S.hi[blockIdx.x],
             [&](int64_t i, int k) {
                 vb[k] = b[i];
                 vh[k] = h[i];
             },
             [&](int64_t i, int k) {
                 const double d = vb[k] - vh[k];
                 r[i] = d;
                 v[0] += d * d;
                 v[1] += vb[k] * vb[k];
             });
    seg_part<SEG_THREADS, 2>(v, lds, S.parts + blockIdx.x, gridDim.x);
}

__global__ void __launch_bounds__(SEG_THREADS)
    k_seg_upd64(SegTab S, BState B, double *__restrict__ x, const float *__restrict__ d)
{
    const int inst = S.inst[blockIdx.x];
    if (B.conv[inst]) return;
    const double a = 1.0 / B.scale[inst];
    for (int64_t i = S.lo[blockIdx.x] + threadIdx.x; i < S.hi[blockIdx.x]; i += SEG_THREADS)
        x[i] += a * (double)d[i];
}

template <typename T>
__global__ void k_jacobi_inv_b(const double *__restrict__ d, T *__restrict__ dinv, int64_t n)
{
    const double eps = 16.0 * 2.220446049250313e-16;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        dinv[i] = (T)(fabs(d[i]) < eps ? 1.0 : 1.0 / d[i]);
}

// ---------------------------------------------------------------------------------
void Batch::init(Context *c, int n, const int *nx_, const int *ny_, double c_)
{
    ctx = c;
    count = n;
    creac = c_;
    FEM_CHECK(n >= 1, FEM_ERR_ARG, "batch: at least one instance");
    nx.assign(nx_, nx_ + n);
    ny.assign(ny_, ny_ + n);
    dof_off.assign(n + 1, 0);
    elem_off.assign(n + 1, 0);
    for (int i = 0; i < n; ++i) {
        FEM_CHECK(nx[i] > 0 && ny[i] > 0, FEM_ERR_ARG, "batch: mesh size");
        dof_off[i + 1] = dof_off[i] + (int64_t)(2 * nx[i] + 1) * (2 * ny[i] + 1);
        elem_off[i + 1] = elem_off[i] + (int64_t)nx[i] * ny[i];
    }
    N = dof_off[n];
    E = elem_off[n];
    for (int sh = 0; sh < CG_NSHAPES; ++sh) {
        std::vector<CGInst> v(n);
        std::vector<int> of;
        for (int i = 0; i < n; ++i) {
            CGInst &I = v[i];
            I = cg_inst(nx[i], ny[i], sh, creac, 1.0);
            I.dof_off = dof_off[i];
            I.elem_off = elem_off[i];
            I.tile_off = (int)of.size();
            of.insert(of.end(), I.ntiles, i);
        }
        std::vector<int> tf(n + 1);
        for (int i = 0; i < n; ++i) tf[i] = v[i].tile_off;
        tf[n] = (int)of.size();
        tile_first[sh].alloc(sizeof(int) * (n + 1));
        FEM_HIP(hipMemcpy(tile_first[sh].p, tf.data(), sizeof(int) * (n + 1), hipMemcpyHostToDevice));
        tile_inst[sh].alloc(sizeof(int) * of.size());
        FEM_HIP(hipMemcpy(tile_inst[sh].p, of.data(), sizeof(int) * of.size(), hipMemcpyHostToDevice));
        tiles[sh] = (int)of.size();
        inst_dev[sh].alloc(sizeof(CGInst) * n);
        FEM_HIP(hipMemcpy(inst_dev[sh].p, v.data(), sizeof(CGInst) * n, hipMemcpyHostToDevice));
    }
    CGTab t = make_cg_tab();
    tab.alloc(sizeof(t));
    FEM_HIP(hipMemcpy(tab.p, &t, sizeof(t), hipMemcpyHostToDevice));
    // segment table
    std::vector<int> sinst, first(n + 1, 0);
    std::vector<int64_t> slo, shi;
    for (int i = 0; i < n; ++i) {
        first[i] = (int)sinst.size();
        const int64_t nd = dof_off[i + 1] - dof_off[i], most = (int64_t)SEG_MOST * SEG_CHUNK;
        const int64_t len = SEG_CHUNK * ((nd + most - 1) / most);
        for (int64_t a = dof_off[i]; a < dof_off[i + 1]; a += len) {
            sinst.push_back(i);
            slo.push_back(a);
            shi.push_back(std::min<int64_t>(a + len, dof_off[i + 1]));
        }
    }
    first[n] = (int)sinst.size();
    nseg = (int)sinst.size();
    seg_inst.alloc(sizeof(int) * nseg);
    seg_lo.alloc(sizeof(int64_t) * nseg);
    seg_hi.alloc(sizeof(int64_t) * nseg);
    seg_first.alloc(sizeof(int) * (n + 1));
    seg_parts.alloc(sizeof(double) * 2 * nseg);
    FEM_HIP(hipMemcpy(seg_inst.p, sinst.data(), sizeof(int) * nseg, hipMemcpyHostToDevice));
    FEM_HIP(hipMemcpy(seg_lo.p, slo.data(), sizeof(int64_t) * nseg, hipMemcpyHostToDevice));
    FEM_HIP(hipMemcpy(seg_hi.p, shi.data(), sizeof(int64_t) * nseg, hipMemcpyHostToDevice));
    FEM_HIP(hipMemcpy(seg_first.p, first.data(), sizeof(int) * (n + 1), hipMemcpyHostToDevice));
    // per-instance state
    sdbl.alloc(sizeof(double) * (6 * n + 1));
    sint.alloc(sizeof(int) * (4 * n + 1));
    FEM_HIP(hipMemset(sdbl.p, 0, sdbl.bytes));
    FEM_HIP(hipMemset(sint.p, 0, sint.bytes));
    active.alloc(sizeof(int));
    FEM_HIP(hipHostMalloc((void **)&hactive, sizeof(int), hipHostMallocDefault));
}

void Batch::drop_graph()
{
    if (graph_exec) (void)hipGraphExecDestroy(graph_exec);
    if (graph) (void)hipGraphDestroy(graph);
    graph_exec = nullptr;
    graph = nullptr;
}

Batch::~Batch()
{
    drop_graph();
    if (hactive) (void)hipHostFree(hactive);
}

void Batch::set_kappa_qp(const double *kv)
{
    FEM_CHECK(kv, FEM_ERR_ARG, "null kappa");
    // the coefficient and Jacobi buffers keep their addresses after the first
    // call (the captured graph reads kvol32 and dinv32); a first allocation
    // drops any graph
    if (!kvol64.p) {
        drop_graph();
        kvol64.alloc(sizeof(double) * E * 9);
        kvol32.alloc(sizeof(float) * E * 9);
        dinv64.alloc(sizeof(double) * N);
        dinv32.alloc(sizeof(float) * N);
    }
    FEM_HIP(hipMemcpy(kvol64.p, kv, sizeof(double) * E * 9, hipMemcpyHostToDevice));
    std::vector<float> f(E * 9);
    for (int64_t i = 0; i < E * 9; ++i) f[i] = (float)kv[i];
    FEM_HIP(hipMemcpy(kvol32.p, f.data(), sizeof(float) * E * 9, hipMemcpyHostToDevice));
    // Jacobi diagonal (FP64 and FP32 inverses)
    DevBuf d;
    d.alloc(sizeof(double) * N);
    cg_launch_shape<double>(0, CG_MODE_DIAG, inst_dev[0].as<CGInst>(), tile_inst[0].as<int>(), tiles[0], tab.as<CGTab>(),
                            kvol64.as<double>(), nullptr, d.as<double>(), nullptr, nullptr, ctx->stream,
                            CGReaction<double>(), true);
    hipLaunchKernelGGL(k_jacobi_inv_b<double>, dim3(grid_for(N, 256, 8192)), dim3(256), 0, ctx->stream, d.as<double>(), dinv64.as<double>(), N);
    hipLaunchKernelGGL(k_jacobi_inv_b<float>, dim3(grid_for(N, 256, 8192)), dim3(256), 0, ctx->stream, d.as<double>(), dinv32.as<float>(), N);
    FEM_HIP(hipGetLastError());
    FEM_HIP(hipStreamSynchronize(ctx->stream));
}

void Batch::apply_raw(int prec, const void *u, void *w, const int *inst_done) const
{
    FEM_CHECK(kvol64.p, FEM_ERR_STATE, "batch: coefficient data not set");
    if (prec == FEM_F64)
        cg_launch_shape<double>(shape, CG_MODE_APPLY, inst_dev[shape].as<CGInst>(), tile_inst[shape].as<int>(),
                                tiles[shape], tab.as<CGTab>(), kvol64.as<double>(), (const double *)u, (double *)w,
                                nullptr, inst_done, ctx->stream, CGReaction<double>(), creac != 0);
    else
        cg_launch_shape<float>(shape, CG_MODE_APPLY, inst_dev[shape].as<CGInst>(), tile_inst[shape].as<int>(),
                               tiles[shape], tab.as<CGTab>(), kvol32.as<float>(), (const float *)u, (float *)w, nullptr,
                               inst_done, ctx->stream, CGReaction<float>(), creac != 0);
}

void Batch::rhs(const double *fq, Vec &F) const
{
    FEM_CHECK(F.n == N && F.prec == FEM_F64, FEM_ERR_ARG, "batch rhs: FP64 vector of the batch size");
    DevBuf f;
    f.alloc(sizeof(double) * E * 9);
    FEM_HIP(hipMemcpy(f.p, fq, sizeof(double) * E * 9, hipMemcpyHostToDevice));
    cg_launch_shape<double>(0, CG_MODE_RHS, inst_dev[0].as<CGInst>(), tile_inst[0].as<int>(), tiles[0], tab.as<CGTab>(),
                            f.as<double>(), nullptr, (double *)F.data, nullptr, nullptr, ctx->stream,
                            CGReaction<double>(), false);
    FEM_HIP(hipStreamSynchronize(ctx->stream));
}

int Batch::autotune(int reps)
{
    // time the FP32 apply of the whole batch for every tile shape; keep the fastest.
    // The apply alone stands for the solve's step (apply and update with the sums):
    // over eleven batches of 1 to 4096 instances it found the step's best shape seven
    // times and one within 2.6 % of it four times
    DevBuf u, w;
    u.alloc(sizeof(float) * N);
    w.alloc(sizeof(float) * N);
    FEM_HIP(hipMemset(u.p, 0, u.bytes));
    float best = 1e30f;
    int bestsh = 0;
    for (int sh = 0; sh < CG_NSHAPES; ++sh) {
        shape = sh;
        apply_raw(FEM_F32, u.p, w.p, nullptr);
        FEM_HIP(hipEventRecord(ctx->ev0, ctx->stream));
        for (int r = 0; r < reps; ++r) apply_raw(FEM_F32, u.p, w.p, nullptr);
        FEM_HIP(hipEventRecord(ctx->ev1, ctx->stream));
        FEM_HIP(hipEventSynchronize(ctx->ev1));
        float ms;
        FEM_HIP(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
        tune_ms[sh] = ms / reps;
        if (ms < best) { best = ms; bestsh = sh; }
    }
    shape = bestsh;
    drop_graph();
    return bestsh;
}

void Batch::solve(const Vec &b, Vec &x, double tol, double inner_tol, int inner_maxit, int max_outer, int use_graph,
                  fem_batch_info &info)
{
    FEM_CHECK(b.n == N && x.n == N && b.prec == FEM_F64 && x.prec == FEM_F64, FEM_ERR_ARG,
              "batch solve: FP64 vectors of the batch size");
    FEM_CHECK(dinv32.p, FEM_ERR_STATE, "batch: coefficient data not set");
    hipStream_t st = ctx->stream;
    std::memset(&info, 0, sizeof(info));
    auto t0 = std::chrono::steady_clock::now();
    // work vectors: allocated on the first solve only (N is fixed for a
    // batch), so the pointers captured in the HIP graph stay valid
    if (!h64.p) {
        drop_graph();
        h64.alloc(sizeof(double) * N);
        r64.alloc(sizeof(double) * N);
        for (DevBuf *v : { &d32, &p32, &q32[0], &q32[1], &s32, &h32 }) v->alloc(sizeof(float) * N);
        dot_parts.alloc(sizeof(double) * *std::max_element(tiles, tiles + CG_NSHAPES));
    }
    const int n = count;
    double *D = sdbl.as<double>();
    int *I = sint.as<int>();
    BState B{ D, D + n, D + 2 * n, D + 3 * n, D + 4 * n, D + 5 * n, D + 6 * n, I, I + n, I + 2 * n, I + 3 * n, I + 4 * n };
    SegTab S{ seg_inst.as<int>(), seg_lo.as<int64_t>(), seg_hi.as<int64_t>(), seg_first.as<int>(),
              seg_parts.as<double>() };
    float *d = d32.as<float>(), *p = p32.as<float>(), *s = s32.as<float>(), *h = h32.as<float>();
    const float *dv = dinv32.as<float>();
    auto step = [&](hipStream_t ss, int k) {
        const float *q = q32[k & 1].as<float>();
        float *qn = q32[(k + 1) & 1].as<float>();
        const auto apply = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(tiles[shape]),
                               dim3((CG_SHAPES[shape][0] + 1) * (CG_SHAPES[shape][1] + 1)), 0, ss, S, B,
                               inst_dev[shape].as<CGInst>(), tile_inst[shape].as<int>(), kvol32.as<float>(), s, q, qn, h,
                               dot_parts.as<double>(), nseg);
        };
        switch (shape) {
        case 0: apply(k_bcg_apply<15, 15>); break;
        case 1: apply(k_bcg_apply<7, 7>); break;
        case 2: apply(k_bcg_apply<15, 7>); break;
        case 3: apply(k_bcg_apply<31, 7>); break;
        default: apply(k_bcg_apply<7, 31>); break;
        }
        hipLaunchKernelGGL(k_bcg_update, dim3(nseg), dim3(SEG_THREADS), 0, ss, S, B, tile_first[shape].as<int>(),
                           dot_parts.as<double>(), dv, qn, h, d, p, s);
        FEM_HIP(hipGetLastError());
    };
    if (use_graph && !graph_exec) {
        FEM_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
        for (int k = 0; k < GRAPH_STEPS; ++k) step(st, k);
        FEM_HIP(hipStreamEndCapture(st, &graph));
        FEM_HIP(hipGraphInstantiate(&graph_exec, graph, nullptr, nullptr, 0));
    }
    FEM_HIP(hipMemsetAsync(B.conv, 0, sizeof(int) * n, st));   // not captured
    // the number of instances still at work
    auto look = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(1), dim3(1024), 0, st, S, B, n, nseg, tol, active.as<int>());
        FEM_HIP(hipGetLastError());
        FEM_HIP(hipMemcpyAsync(hactive, active.p, sizeof(int), hipMemcpyDeviceToHost, st));
        FEM_HIP(hipStreamSynchronize(st));
        return *hactive;
    };
    int outer = 0, total_inner = 0;
    std::vector<int> its(n, 0);
    while (true) {
        // FP64 true residual per instance (those that have converged are skipped)
        apply_raw(FEM_F64, x.data, h64.p, B.conv);
        hipLaunchKernelGGL(k_seg_res64, dim3(nseg), dim3(SEG_THREADS), 0, st, S, B, (const double *)b.data,
                           h64.as<double>(), r64.as<double>());
        if (look(k_batch_look<true>) == 0 || outer >= max_outer) break;
        hipLaunchKernelGGL(k_bcg_init, dim3(nseg), dim3(SEG_THREADS), 0, st, S, B, r64.as<double>(), dv, d, p, s, inner_tol,
                           inner_maxit);
        int chunk = 8, done_steps = 0;   // multiples of GRAPH_STEPS
        while (true) {
            for (int c = 0; c < chunk; c += use_graph ? GRAPH_STEPS : 1) {
                if (use_graph) FEM_HIP(hipGraphLaunch(graph_exec, st));
                else step(st, c);
            }
            done_steps += chunk;
            if (look(k_batch_look<false>) == 0 || done_steps >= inner_maxit) break;
            if (chunk < 64) chunk *= 2;
        }
        std::vector<int> it(n);
        FEM_HIP(hipMemcpy(it.data(), B.it, sizeof(int) * n, hipMemcpyDeviceToHost));
        int mx = 0;
        for (int i = 0; i < n; ++i) {
            its[i] += it[i];
            mx = std::max(mx, it[i]);
            total_inner += it[i];
        }
        info.max_inner_iterations += mx;
        hipLaunchKernelGGL(k_seg_upd64, dim3(nseg), dim3(SEG_THREADS), 0, st, S, B, (double *)x.data, d);
        FEM_HIP(hipGetLastError());
        ++outer;
    }
    FEM_HIP(hipStreamSynchronize(st));
    auto t1 = std::chrono::steady_clock::now();
    std::vector<int> conv(n);
    std::vector<double> rn(n), bn2(n);
    FEM_HIP(hipMemcpy(conv.data(), B.conv, sizeof(int) * n, hipMemcpyDeviceToHost));
    FEM_HIP(hipMemcpy(rn.data(), B.rn, sizeof(double) * n, hipMemcpyDeviceToHost));
    FEM_HIP(hipMemcpy(bn2.data(), B.bn2, sizeof(double) * n, hipMemcpyDeviceToHost));
    info.count = n;
    info.converged = 0;
    info.max_true_rel_residual = 0;
    last_iters = its;
    last_relres.assign(n, 0.0);
    for (int i = 0; i < n; ++i) {
        info.converged += conv[i] ? 1 : 0;
        const double rel = bn2[i] > 0 ? rn[i] / std::sqrt(bn2[i]) : rn[i];
        last_relres[i] = rel;
        info.max_true_rel_residual = std::max(info.max_true_rel_residual, rel);
    }
    info.outer_iterations = outer;
    info.total_inner_iterations = total_inner;
    info.time_s = std::chrono::duration<double>(t1 - t0).count();
    info.tile_x = CG_SHAPES[shape][0];
    info.tile_y = CG_SHAPES[shape][1];
}

}  // namespace femamd
