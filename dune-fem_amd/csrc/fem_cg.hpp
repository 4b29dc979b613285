// Continuous Lagrange Q2 operator on structured quad meshes of [0,1]^2,
// single instance or a batch of independent instances in one launch.
#pragma once

#include "fem_common.hpp"

namespace femamd {

// one problem instance of a batch
struct CGInst {
    int nx, ny;
    int64_t dof_off;    // offset of its DoFs in the batched vectors
    int64_t elem_off;   // offset of its elements (kappa / f arrays: elem_off * 9)
    int tiles_x;        // tiles per row
    int tile_off;       // first workgroup of this instance
    int ntiles;
    double c;           // reaction coefficient
    double kappa_const; // used when kvol == nullptr
    double sx, sy;      // hy / hx and hx / hy
    double detJ;        // hx hy
};

// tile shapes available to the autotuner (owned elements per tile)
constexpr int CG_NSHAPES = 5;
constexpr int CG_SHAPES[CG_NSHAPES][2] = { { 15, 15 }, { 7, 7 }, { 15, 7 }, { 31, 7 }, { 7, 31 } };
// the shape of a single instance's operator: FP64, pointwise kappa, back to back on the
// same vectors, 517 x 386 elements 7.1 us (7 x 7: 8.3, 15 x 7: 7.4, 31 x 7: 7.4), 1024^2
// 27.7 us (32.4, 27.7, 26.5): 31 x 7 is ahead by 4 % where the chip is full many times
// over, behind by as much at a single set of workgroups
constexpr int CG_SINGLE = 0;

// an instance of nx x ny elements in tiles of the given shape
inline CGInst cg_inst(int nx, int ny, int shape, double c, double kappa_const)
{
    CGInst I{};
    I.nx = nx;
    I.ny = ny;
    I.tiles_x = (nx + CG_SHAPES[shape][0] - 1) / CG_SHAPES[shape][0];
    I.ntiles = I.tiles_x * ((ny + CG_SHAPES[shape][1] - 1) / CG_SHAPES[shape][1]);
    I.c = c;
    I.kappa_const = kappa_const;
    I.sx = (double)nx / ny;
    I.sy = (double)ny / nx;
    I.detJ = 1.0 / ((double)nx * ny);
    return I;
}

struct CGTab {
    double L[3][3];   // Q2 basis i at Gauss point q: L[q][i]
    double Ld[3][3];  // derivative
    double w[3];
};

enum { CG_MODE_APPLY = 0, CG_MODE_DIAG = 1, CG_MODE_RHS = 2, CG_MODE_RHS_ADD = 3 };

// the reaction beyond the constant c of a single instance: a pointwise
// coefficient at the volume quadrature points [E][9] (qx + 3 qy) and the
// nonlinear law coef u^pw, both multiplying u v
template <typename T>
struct CGReaction {
    const T *cvol = nullptr;
    T coef = 0;
    int pw = 0;
};

// mode APPLY  : out = A in (Dirichlet rows: out = in)
// mode DIAG   : out = diag(A) (Dirichlet rows: 1), `in` unused
// mode RHS    : out = F from f at quadrature points (kvol slot carries f), Dirichlet rows 0
// mode RHS_ADD: out += F on the interior rows (Dirichlet rows unchanged)
// in tiles of CG_SHAPES[shape]; tile_inst: the instance of each tile, inst the table on
// the device (null: a single instance, inst on the host); instances with inst_done[i] != 0 (may be null) are skipped; `c`: some
// instance has a reaction c; `dot` (APPLY, may be null): the workgroups' FP64
// partials of <in, out>, one per tile
template <typename T>
void cg_launch_shape(int shape, int mode, const CGInst *inst, const int *tile_inst, int total_tiles, const CGTab *d_tab,
                     const T *kvol, const T *in, T *out, const int *skip, const int *inst_done, hipStream_t s,
                     const CGReaction<T> &rx, bool c, double *dot = nullptr);
// out[e*9 + qx + 3 qy] = base + coef u(x_q)^pw (base may be null) for a
// single instance of nx x ny elements
template <typename T>
void cg_eval_qp(int nx, int ny, const CGTab *d_tab, const T *u, const T *base, T coef, int pw, T *out, hipStream_t s);

CGTab make_cg_tab();

}  // namespace femamd
