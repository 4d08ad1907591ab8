// Stencil kernels and their launches, included by the stencil_*.hip sources,
// which instantiate them (one source per vector precision and mode, so that
// they compile side by side).
#include "stencil.hpp"

namespace mfd {

// after the stencil with EPI_DOT: σ = qᵀPq, α = ρ/σ (one block per RHS)
static __global__ __launch_bounds__(BS) void k_fin_dot(const double *part, int nb, Scal *scal) {
    const int rhs = blockIdx.x;
    Scal &S = scal[rhs];
    if (S.done) return;
    double tot[2];
    sum_partials<2>(part + (size_t)rhs * NPART * 4, nb, tot);
    if (threadIdx.x != 0) return;
    if (S.conv) { S.done = 1; return; }
    S.sig_re = tot[0];
    S.sig_im = tot[1];
    if (tot[0] == 0.0 && tot[1] == 0.0) {   // breakdown: no step (the stencil already applied the pending update)
        S.breakdown = 1;
        S.conv = 1;
        S.alpha_re = S.alpha_im = 0;
        S.apend_re = S.apend_im = 0;
        return;
    }
    c64 a = cdiv(mk<double>(S.rho_re, S.rho_im), mk<double>(tot[0], tot[1]));
    S.alpha_re = a.re;
    S.alpha_im = a.im;
    S.apend_re = a.re;
    S.apend_im = a.im;
}

// after the stencil with EPI_RESID: ||b − A x||² per (unmasked) RHS
static __global__ __launch_bounds__(BS) void k_fin_resid(const double *part, int nb, double *rn, const int *mask) {
    const int rhs = blockIdx.x;
    if (mask && !mask[rhs]) return;
    double tot[1];
    sum_partials<1>(part + (size_t)rhs * NPART * 4, nb, tot);
    if (threadIdx.x == 0) rn[rhs] = tot[0];
}

// ------------------------------------------------------------ the stencil

// y = A x (MODE_A) or y = P x (MODE_P) for the RHS blockIdx.y.
// EPI_STORE: y = op(x).  EPI_RESID: y = b − op(x), reduce ||y||² into rn.
// EPI_DOT: y = op(x), reduce xᵀy into the solver scalars (σ, α).
// EPI_BDOT, EPI_XDOT: y = op(x), partials of bᴴy, and of yᴴx and ‖y‖² (summed
// by the kernel that uses them).
// H value from the scratch of k_hpass at (i,j,k) with one index possibly −1
// or N: the Bloch image times the phase, or zero past a non-Bloch end
template <typename R>
__device__ inline cx<R> ldHb(const DGrid<R> &g, const cx<R> *__restrict__ hb, int c, int i, int j, int k) {
    cx<R> ph = cone<R>();
    bool wr = false;
    int id[3] = {i, j, k};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        if (id[a] < 0) {
            if (!g.bloch[a]) return czero<R>();
            id[a] += g.N[a]; ph = ph * g.phinv[a]; wr = true;
        } else if (id[a] >= g.N[a]) {
            if (!g.bloch[a]) return czero<R>();
            id[a] -= g.N[a]; ph = ph * g.ph[a]; wr = true;
        }
    }
    cx<R> v = hb[dofidx(g, c, id[0] + (int64_t)g.N[0] * (id[1] + (int64_t)g.N[1] * id[2]))];
    return wr ? v * ph : v;
}

// first pass of the two-pass direct kernel: H = μ⁻¹ Cₑ X at every cell, once
template <typename R, int MODE, bool MU>
__global__ __launch_bounds__(BS) void k_hpass(DGrid<R> g, OpData<R> od, const cx<R> *__restrict__ xall,
                                              cx<R> *__restrict__ hall, int64_t vs, const Scal *scal, int epi_dot) {
    const int rhs = blockIdx.y;
    if (epi_dot && (scal[rhs].done || scal[rhs].conv)) return;
    const cx<R> *x = xall + rhs * vs;
    cx<R> *hb = hall + rhs * vs;
    for (int64_t p = blockIdx.x * (int64_t)BS + threadIdx.x; p < g.M; p += (int64_t)gridDim.x * BS) {
        int i, j, k;
        cell3(g, p, i, j, k);
#pragma unroll
        for (int c = 0; c < 3; ++c) hb[dofidx(g, c, p)] = Hval<R, MODE, MU>(g, od, x, c, i, j, k);
    }
}

// HB: H comes from k_hpass's scratch (hall) instead of being recomputed at p
// and its six neighbours
template <typename R, int MODE, bool OFFD, bool MU, int EPI, bool HB = false>
__global__ __launch_bounds__(BS) void k_apply(DGrid<R> g, OpData<R> od, const cx<R> *__restrict__ xall,
                                              cx<R> *__restrict__ yall, const c64 *__restrict__ ball, int64_t vs,
                                              double *part, const Scal *scal,
                                              const int *__restrict__ mask = nullptr,
                                              const cx<R> *__restrict__ hall = nullptr) {
    const int rhs = blockIdx.y;
    const cx<R> *x = xall + rhs * vs;
    cx<R> *y = yall + rhs * vs;
    const cx<R> *hb = HB ? hall + rhs * vs : nullptr;
    bool skip = false;
    if (EPI == EPI_RESID && mask && !mask[rhs]) return;
    if (EPI == EPI_DOT) {
        if (scal[rhs].done) return;
        skip = scal[rhs].conv != 0;
    }
    if ((EPI == EPI_BDOT || EPI == EPI_XDOT) && (scal[rhs].done || scal[rhs].conv)) return;
    constexpr int NA = EPI == EPI_XDOT ? 3 : 2;
    double acc[NA] = {};
    if (!skip) {
        for (int64_t p = blockIdx.x * (int64_t)BS + threadIdx.x; p < g.M; p += (int64_t)gridDim.x * BS) {
            int i, j, k;
            cell3(g, p, i, j, k);
            // H_c(p) and Hm[c][a] = H_c(p ∓ â), the neighbour Cₘ's difference
            // along a takes (p − â along an EE axis, p + â along an HH axis)
            cx<R> H[3], Hm[3][3];
#pragma unroll
            for (int c = 0; c < 3; ++c) H[c] = HB ? hb[dofidx(g, c, p)] : Hval<R, MODE, MU>(g, od, x, c, i, j, k);
#pragma unroll
            for (int c = 0; c < 3; ++c)
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    if (a == c) continue;
                    int id[3] = {i, j, k};
                    id[a] += g.bft[a] == EE ? -1 : 1;
                    Hm[c][a] = HB ? ldHb(g, hb, c, id[0], id[1], id[2])
                                  : Hval<R, MODE, MU>(g, od, x, c, id[0], id[1], id[2]);
                }
            int id[3] = {i, j, k};
#pragma unroll
            for (int u = 0; u < 3; ++u) {
                int v = u == 0 ? 1 : (u == 1 ? 2 : 0), w = u == 0 ? 2 : (u == 1 ? 0 : 1);
                // E_u = ∂_v H_w − ∂_w H_v (backward along EE axes, forward along HH axes)
                cx<R> dv = g.bft[v] == EE ? H[w] - Hm[w][v] : Hm[w][v] - H[w];
                cx<R> dw = g.bft[w] == EE ? H[v] - Hm[v][w] : Hm[v][w] - H[v];
                cx<R> cc = g.sdlinv[g0type(g.bft, EE, v)][v][id[v]] * dv - g.sdlinv[g0type(g.bft, EE, w)][w][id[w]] * dw;
                int64_t e = dofidx(g, u, p);
                cx<R> xu = x[e];
                cx<R> out;
                cx<R> lf;
                if (MODE == MODE_A) {
                    out = cc - od.om2 * (od.epsd[3 * p + u] * xu);
                } else {
                    cx<R> qu = od.q[3 * p + u];
                    lf = qu * tfac(g, u, i, j, k, false);
                    cx<R> cd = ccdiag<R, MU>(g, od, u, i, j, k);
                    out = lf * cc + (cone<R>() - cd * (qu * qu)) * xu;
                }
                if (OFFD) {
                    cx<R> term = czero<R>();
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        int ww = t == 0 ? v : w;   // input component
                        int eix = (u + ww == 1) ? 0 : ((u + ww == 2) ? 1 : 2);   // (xy, xz, yz)
#pragma unroll
                        for (int oc = 0; oc < 2; ++oc) {
                            int cid[3] = {i, j, k};
                            cx<R> fo = mk<R>((R)0.5, (R)0);
                            if (oc == 1) {
                                cid[u] += 1;
                                if (cid[u] >= g.N[u]) {
                                    if (!g.bloch[u]) continue;
                                    cid[u] -= g.N[u];
                                    fo = (R)0.5 * g.ph[u];
                                }
                            }
                            int64_t cp = cid[0] + (int64_t)g.N[0] * (cid[1] + (int64_t)g.N[1] * cid[2]);
                            cx<R> ec = od.epso[3 * cp + eix];
                            int cw = cid[ww];
                            cx<R> ia = g.sdlinv[PRIM][ww][cw];
                            cx<R> wi0 = ((R)0.5 * g.sdl[DUAL][ww][cw]) * ia;
                            cx<R> s = wi0 * ldX<R, MODE>(g, od, x, ww, cid[0], cid[1], cid[2]);
                            int fid[3] = {cid[0], cid[1], cid[2]};
                            fid[ww] -= 1;
                            if (fid[ww] >= 0 || g.bloch[ww]) {
                                int fi = fid[ww] >= 0 ? fid[ww] : g.N[ww] - 1;
                                cx<R> wi1 = ((R)0.5 * g.sdl[DUAL][ww][fi]) * ia;
                                s = s + wi1 * ldX<R, MODE>(g, od, x, ww, fid[0], fid[1], fid[2]);
                            }
                            term = term + (fo * ec) * s;
                        }
                    }
                    if (MODE == MODE_A) out = out - od.om2 * term;
                    else out = out - od.om2 * (lf * term);
                }
                if (EPI == EPI_RESID) {
                    c64 bb = ball[rhs * vs + e];
                    cx<R> rr = mk<R>((R)bb.re - out.re, (R)bb.im - out.im);
                    if (yall) y[e] = rr;   // null output: the residual norm only
                    acc[0] += (double)rr.re * rr.re + (double)rr.im * rr.im;
                } else {
                    y[e] = out;
                    epi_add<EPI>(acc, cvt<double>(xu), cvt<double>(out), EPI == EPI_BDOT ? ball[rhs * vs + e] : czero<double>());
                }
            }
        }
    }
    if (EPI == EPI_STORE) return;
    block_partial<NA>(acc, part + (size_t)rhs * NPART * 4, (int)blockIdx.x);
}

// Sparse product for an operator built from a caller's CSC matrix A (stored
// row-major): MODE_A y = A x, MODE_P y = Q T A T⁻¹ Q x with qin = Q T⁻¹ and
// qout = Q T per DOF (Q = diag(A)^-1/2, T the symmetrizing scaling); the
// epilogues are those of k_apply.
// LPR lanes share a row (its entries are contiguous), summed by shuffles.
template <typename R, int MODE, int EPI>
__global__ __launch_bounds__(BS) void k_spmv(int64_t m, const int64_t *__restrict__ rowptr,
                                             const int32_t *__restrict__ colind, const c64 *__restrict__ val,
                                             const c64 *__restrict__ qin, const c64 *__restrict__ qout,
                                             const cx<R> *__restrict__ xall,
                                             cx<R> *__restrict__ yall, const c64 *__restrict__ ball, int64_t vs,
                                             double *part, const Scal *scal, const int *__restrict__ mask) {
    constexpr int LPR = 4;
    const int rhs = blockIdx.y;
    const cx<R> *x = xall + rhs * vs;
    cx<R> *y = yall + rhs * vs;
    bool skip = false;
    if (EPI == EPI_RESID && mask && !mask[rhs]) return;
    if (EPI == EPI_DOT) {
        if (scal[rhs].done) return;
        skip = scal[rhs].conv != 0;
    }
    if ((EPI == EPI_BDOT || EPI == EPI_XDOT) && (scal[rhs].done || scal[rhs].conv)) return;
    constexpr int NA = EPI == EPI_XDOT ? 3 : 2;
    double acc[NA] = {};
    const int lane = threadIdx.x % LPR;
    if (!skip) {
        for (int64_t i = (blockIdx.x * (int64_t)BS + threadIdx.x) / LPR; i < m; i += (int64_t)gridDim.x * (BS / LPR)) {
            c64 s = mk<double>(0, 0);
            for (int64_t k = rowptr[i] + lane; k < rowptr[i + 1]; k += LPR) {
                const int32_t j = colind[k];
                c64 xv = cvt<double>(x[j]);
                if (MODE == MODE_P) xv = xv * qin[j];
                s = s + val[k] * xv;
            }
#pragma unroll
            for (int o = 1; o < LPR; o <<= 1) {
                s.re += __shfl_xor(s.re, o, LPR);
                s.im += __shfl_xor(s.im, o, LPR);
            }
            if (lane) continue;
            const c64 xi = cvt<double>(x[i]);
            const c64 out = MODE == MODE_P ? qout[i] * s : s;
            if (EPI == EPI_RESID) {
                const c64 bb = ball[rhs * vs + i];
                const c64 rr = mk<double>(bb.re - out.re, bb.im - out.im);
                if (yall) y[i] = cvt<R>(rr);   // null output: the residual norm only
                acc[0] += rr.re * rr.re + rr.im * rr.im;
            } else {
                y[i] = cvt<R>(out);
                epi_add<EPI>(acc, xi, out, EPI == EPI_BDOT ? ball[rhs * vs + i] : czero<double>());
            }
        }
    }
    if (EPI == EPI_STORE) return;
    block_partial<NA>(acc, part + (size_t)rhs * NPART * 4, (int)blockIdx.x);
}

#include "stencil_tiled.hpp"
#include "stencil_plane.hpp"

// finish kernel of a stencil epilogue with a reduction (nb partials per RHS)
template <int EPI>
void launch_finish(hipStream_t s, int nb, int64_t nrhs, double *part, Scal *scal, double *rn, const int *mask) {
    if (EPI == EPI_DOT) k_fin_dot<<<(unsigned)nrhs, BS, 0, s>>>(part, nb, scal);
    else if (EPI == EPI_RESID) k_fin_resid<<<(unsigned)nrhs, BS, 0, s>>>(part, nb, rn, mask);
}

// launch one operator apply; returns the number of partial sums per RHS its
// reduction wrote (finish = false leaves them to the next kernel)
template <typename R, int MODE, int EPI>
int launch_apply(mfd_op *op, const cx<R> *x, cx<R> *y, const c64 *b, int64_t nrhs, double *part, Scal *scal, double *rn,
                 const int *mask, hipEvent_t after_main, bool finish) {
    const DGrid<R> &g = op->G.view<R>();
    const OpData<R> &od = opd<R>(op);
    int64_t vs = op->n;
    hipStream_t s = op->stream;
    if (op->csr) {   // an operator built from a caller's CSC matrix
        dim3 grid(ngrid(vs), (unsigned)nrhs);
        k_spmv<R, MODE, EPI><<<grid, BS, 0, s>>>(vs, op->csr_rowptr, op->csr_colind, op->csr_val, op->d64.qs,
                                                 op->csr_qo, x, y, b, vs, part, scal, mask);
        if (after_main) hipEventRecord(after_main, s);
        if (finish) launch_finish<EPI>(s, (int)grid.x, nrhs, part, scal, rn, mask);
        return (int)grid.x;
    }
    if (plane_ok(op, std::is_same<R, double>::value)) {
        const DGrid<double> &gp = op->G.d64;
        const int ntx = (gp.N[0] + PL_TX - 1) / PL_TX;
        const int64_t nt = ntx * (int64_t)((gp.N[1] + PL_TY - 1) / PL_TY);
        const dim3 grid((unsigned)std::min<int64_t>(nt, NPART), (unsigned)nrhs);
#define MFD_PLANE(OFF, TM) \
    k_apply_plane<R, MODE, EPI, OFF, TM><<<grid, PL_TX * PL_TY, 0, s>>>(gp, op->d64, op->d64.om2, x, y, b, vs, ntx, nt, part, scal, mask)
        if (gp.nc == 1) MFD_PLANE(false, true);   // corner ε couples Ex and Ey only
        else if (op->full) MFD_PLANE(true, false);
        else MFD_PLANE(false, false);
#undef MFD_PLANE
        if (after_main) hipEventRecord(after_main, s);
        if (finish) launch_finish<EPI>(s, (int)grid.x, nrhs, part, scal, rn, mask);
        return (int)grid.x;
    }
    const Tile tile = stencil_tile(op, std::is_same<R, double>::value, nrhs, MODE);
    int ty = tile.ty, kz = tile.kz, xr = tile.xr;
    const bool gd = MODE == MODE_P && op->gd;
    if (gd && ty == 8) ty = 4;   // the grad-div tile keeps two more LDS planes
    // order bit 1: 32-wide tiles of 2·TY rows (same threads per block);
    // the off-diagonal, grad-div, μ and reflected stencils are built 64-wide only
    const bool narrow = (xr & 2) && !op->full && !gd && !op->has_mu && !op->rev && !op->win;
    // μ ≠ 1 has a tiled form with diagonal ε (the grad-div form is never on with
    // μ); a grid too large for any tile goes to the direct kernel, which has no
    // grad-div form or window (ws_ensure refuses the reductions of those)
    bool tiled = (op->ee_all || op->rev) && ty > 0 && !(op->has_mu && op->full);
    if (tiled && !tile_fit(op->G.d64.N, nrhs, narrow, gd ? 4 : 8, EPI != EPI_STORE, NPART, ty, kz)) tiled = gd || op->win;
    if (tiled) {
        xr &= 1;
        const int tw = narrow ? 32 : 64, rows = narrow ? 2 * ty : ty;
        int nx = (g.N[0] + tw - 1) / tw, ny = (g.N[1] + rows - 1) / rows;
        int nch = (g.N[2] + kz - 1) / kz;
        dim3 grid(nx, ny, (unsigned)(nch * nrhs));
        const DGrid<double> &gr = op->G.r64;
        if (op->win && op->full) {   // a component window (2D and 1D models), μ = 1, boundft EE
            if (ty == 8) k_apply_tiled<R, MODE, EPI, 8, false, false, true, 64, false, false, true><<<grid, 512, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else if (ty == 2) k_apply_tiled<R, MODE, EPI, 2, false, false, true, 64, false, false, true><<<grid, 128, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else if (ty == 4) k_apply_tiled<R, MODE, EPI, 4, false, false, true, 64, false, false, true><<<grid, 256, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else k_apply_tiled<R, MODE, EPI, 1, false, false, true, 64, false, false, true><<<grid, 64, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
        } else if (op->win) {
            if (ty == 8) k_apply_tiled<R, MODE, EPI, 8, false, false, false, 64, false, false, true><<<grid, 512, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else if (ty == 2) k_apply_tiled<R, MODE, EPI, 2, false, false, false, 64, false, false, true><<<grid, 128, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else if (ty == 4) k_apply_tiled<R, MODE, EPI, 4, false, false, false, 64, false, false, true><<<grid, 256, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else k_apply_tiled<R, MODE, EPI, 1, false, false, false, 64, false, false, true><<<grid, 64, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
        } else if (op->rev && op->has_mu) {   // boundft HH on some axis: the grid reflected along those axes
            if (ty == 8) k_apply_tiled<R, MODE, EPI, 8, false, false, false, 64, true, true><<<grid, 512, 0, s>>>(gr, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else if (ty == 2) k_apply_tiled<R, MODE, EPI, 2, false, false, false, 64, true, true><<<grid, 128, 0, s>>>(gr, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else if (ty == 4) k_apply_tiled<R, MODE, EPI, 4, false, false, false, 64, true, true><<<grid, 256, 0, s>>>(gr, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else k_apply_tiled<R, MODE, EPI, 1, false, false, false, 64, true, true><<<grid, 64, 0, s>>>(gr, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
        } else if (op->rev) {
            if (ty == 8) k_apply_tiled<R, MODE, EPI, 8, false, false, false, 64, false, true><<<grid, 512, 0, s>>>(gr, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else if (ty == 2) k_apply_tiled<R, MODE, EPI, 2, false, false, false, 64, false, true><<<grid, 128, 0, s>>>(gr, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else if (ty == 4) k_apply_tiled<R, MODE, EPI, 4, false, false, false, 64, false, true><<<grid, 256, 0, s>>>(gr, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else k_apply_tiled<R, MODE, EPI, 1, false, false, false, 64, false, true><<<grid, 64, 0, s>>>(gr, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
        } else if (op->full) {   // off-diagonal ε (grad-div is never enabled with it)
            if (ty == 8) k_apply_tiled<R, MODE, EPI, 8, false, false, true><<<grid, 512, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else if (ty == 2) k_apply_tiled<R, MODE, EPI, 2, false, false, true><<<grid, 128, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else if (ty == 4) k_apply_tiled<R, MODE, EPI, 4, false, false, true><<<grid, 256, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else k_apply_tiled<R, MODE, EPI, 1, false, false, true><<<grid, 64, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
        } else if (gd) {
            if (ty == 2) k_apply_tiled<R, MODE, EPI, 2, true><<<grid, 128, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else if (ty == 4) k_apply_tiled<R, MODE, EPI, 4, true><<<grid, 256, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else k_apply_tiled<R, MODE, EPI, 1, true><<<grid, 64, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
        } else if (op->has_mu) {
            if (ty == 8) k_apply_tiled<R, MODE, EPI, 8, false, false, false, 64, true><<<grid, 512, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else if (ty == 2) k_apply_tiled<R, MODE, EPI, 2, false, false, false, 64, true><<<grid, 128, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else if (ty == 4) k_apply_tiled<R, MODE, EPI, 4, false, false, false, 64, true><<<grid, 256, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else k_apply_tiled<R, MODE, EPI, 1, false, false, false, 64, true><<<grid, 64, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
        } else if (narrow) {
            if (ty == 8) k_apply_tiled<R, MODE, EPI, 16, false, false, false, 32><<<grid, 512, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else if (ty == 2) k_apply_tiled<R, MODE, EPI, 4, false, false, false, 32><<<grid, 128, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else if (ty == 4) k_apply_tiled<R, MODE, EPI, 8, false, false, false, 32><<<grid, 256, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else k_apply_tiled<R, MODE, EPI, 2, false, false, false, 32><<<grid, 64, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
        } else {
            if (ty == 8) k_apply_tiled<R, MODE, EPI, 8, false><<<grid, 512, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else if (ty == 2) k_apply_tiled<R, MODE, EPI, 2, false><<<grid, 128, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else if (ty == 4) k_apply_tiled<R, MODE, EPI, 4, false><<<grid, 256, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
            else k_apply_tiled<R, MODE, EPI, 1, false><<<grid, 64, 0, s>>>(op->G.d64, op->d64, op->d64.om2, x, y, b, vs, kz, nch, part, scal, mask, xr);
        }
        if (after_main) hipEventRecord(after_main, s);
        if (finish) launch_finish<EPI>(s, nx * ny * nch, nrhs, part, scal, rn, mask);
        return nx * ny * nch;
    }
    dim3 grid(ngrid(g.M), (unsigned)nrhs);
    // two passes when the scratch is there: H = μ⁻¹ Cₑ X once per cell, then
    // E from H (instead of recomputing H at each cell and its six neighbours)
    const bool two = op->hbuf && op->hbuf_bytes >= sizeof(cx<R>) * (size_t)vs * (size_t)nrhs;
    cx<R> *hb = (cx<R> *)op->hbuf;
    if (two) {
        if (op->has_mu) k_hpass<R, MODE, true><<<grid, BS, 0, s>>>(g, od, x, hb, vs, scal, EPI >= EPI_DOT);
        else k_hpass<R, MODE, false><<<grid, BS, 0, s>>>(g, od, x, hb, vs, scal, EPI >= EPI_DOT);
    }
#define MFD_DIRECT(OFF, MU_)                                                                                   \
    do {                                                                                                       \
        if (two) k_apply<R, MODE, OFF, MU_, EPI, true><<<grid, BS, 0, s>>>(g, od, x, y, b, vs, part, scal, mask, hb); \
        else k_apply<R, MODE, OFF, MU_, EPI><<<grid, BS, 0, s>>>(g, od, x, y, b, vs, part, scal, mask);          \
    } while (0)
    if (op->full) {
        if (op->has_mu) MFD_DIRECT(true, true);
        else MFD_DIRECT(true, false);
    } else {
        if (op->has_mu) MFD_DIRECT(false, true);
        else MFD_DIRECT(false, false);
    }
#undef MFD_DIRECT
    if (after_main) hipEventRecord(after_main, s);
    if (finish) launch_finish<EPI>(s, (int)grid.x, nrhs, part, scal, rn, mask);
    return (int)grid.x;
}

template <typename R>
void launch_cocg_stencil(mfd_op *op, dim3 grid, int ty, int kz, int nch, int xr, const cx<R> *po, cx<R> *t,
                         const cx<R> *rr, cx<R> *pn, cx<R> *xi) {
    hipStream_t s = op->stream;
    if (ty == 8)
        k_apply_tiled<R, MODE_P, EPI_DOT, 8, false, true><<<grid, 512, 0, s>>>(op->G.d64, op->d64, op->d64.om2, po, t, nullptr, op->n, kz, nch, op->ws.part, op->ws.scal, nullptr, xr, rr, pn, xi);
    else if (ty == 2)
        k_apply_tiled<R, MODE_P, EPI_DOT, 2, false, true><<<grid, 128, 0, s>>>(op->G.d64, op->d64, op->d64.om2, po, t, nullptr, op->n, kz, nch, op->ws.part, op->ws.scal, nullptr, xr, rr, pn, xi);
    else if (ty == 4)
        k_apply_tiled<R, MODE_P, EPI_DOT, 4, false, true><<<grid, 256, 0, s>>>(op->G.d64, op->d64, op->d64.om2, po, t, nullptr, op->n, kz, nch, op->ws.part, op->ws.scal, nullptr, xr, rr, pn, xi);
    else
        k_apply_tiled<R, MODE_P, EPI_DOT, 1, false, true><<<grid, 64, 0, s>>>(op->G.d64, op->d64, op->d64.om2, po, t, nullptr, op->n, kz, nch, op->ws.part, op->ws.scal, nullptr, xr, rr, pn, xi);
}

}  // namespace mfd
