// Launches of the operator's stencils and of the sparse product.
#pragma once
#include "krylov_dev.hpp"
#include "tile_rule.hpp"

namespace mfd {

// the tile shape of a stencil launch over nrhs right-hand sides (mode: A or P;
// cocg: COCG's fused P)
struct Tile {
    int ty, kz, xr;   // rows, planes, order (bit 0: XCD runs, bit 1: 32-wide); ty = 0: the direct kernel
};
Tile stencil_tile(const mfd_op *op, bool fp64, int64_t nrhs, int mode, bool cocg = false);

// a 2D model's window on one plane of cells that k_apply_plane serves
static inline bool plane_ok(const mfd_op *op, bool fp64) {
    const DGrid<double> &g = op->G.d64;
    return op->win && g.N[2] == 1 && g.bloch[2] && g.ph[2].re == 1.0 && g.ph[2].im == 0.0 && op->ee_all &&
           ((g.c0 == 0 && g.nc == 2) || (g.c0 == 2 && g.nc == 1)) && op->tile_set[fp64 ? 0 : 1] != 1;
}

// launch one operator apply; returns the number of partial sums per RHS its
// reduction wrote (finish = false leaves them to the next kernel)
template <typename R, int MODE, int EPI>
int launch_apply(mfd_op *op, const cx<R> *x, cx<R> *y, const c64 *b, int64_t nrhs, double *part, Scal *scal, double *rn,
                 const int *mask = nullptr, hipEvent_t after_main = nullptr, bool finish = true);
// finish kernel of a stencil epilogue with a reduction (nb partials per RHS)
template <int EPI>
void launch_finish(hipStream_t s, int nb, int64_t nrhs, double *part, Scal *scal, double *rn, const int *mask);
// COCG's fused stencil: p = r + β p_old formed while staging (stored in pn),
// the deferred it += α_prev p_old, t = P p and the pᵀt partials
template <typename R>
void launch_cocg_stencil(mfd_op *op, dim3 grid, int ty, int kz, int nch, int xr, const cx<R> *po, cx<R> *t,
                         const cx<R> *rr, cx<R> *pn, cx<R> *xi);

}  // namespace mfd
