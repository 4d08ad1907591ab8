// The stencil of a 2D model: one plane of cells (a periodic one-cell z axis
// without a phase) and the unknowns (Ex, Ey) or Ez, whose curl-curl has one or
// two components of H and no z differences.
//
// The marching stencil serves such an operator as a plane of three components:
// its registers and LDS leave one 8-row block on a CU, which waits for its
// tables, its staging and its corner ε one after the other (640×522 cells of
// (Ex, Ey) with corner ε: 36 µs in three rounds of blocks).  Here a block
// asks for everything at once and three of 4 rows share a CU (13 KB of LDS,
// 154 registers): 18.9 µs for about 53 MB.  Four a CU need 26 spilled registers
// (23.0 µs; 8 rows 21.4), five more (38.6).  Every sum is formed from the same
// terms in the same order.
// FP64 data and arithmetic throughout, as in stencil_tiled.hpp.
constexpr int PL_TX = 64, PL_TY = 4;
template <typename R, int MODE, int EPI, bool OFFD, bool TM>
__global__ __launch_bounds__(PL_TX *PL_TY, 3) void k_apply_plane(DGrid<double> g, OpData<double> od, c64 om2,
                                                              const cx<R> *__restrict__ xall, cx<R> *__restrict__ yall,
                                                              const c64 *__restrict__ ball, int64_t vs, int ntx,
                                                              int64_t ntiles, double *part, const Scal *scal,
                                                              const int *__restrict__ mask) {
    constexpr int C0 = TM ? 2 : 0, NC = TM ? 1 : 2;   // the unknowns' components
    __shared__ c64 Xs[NC][PL_TY + 2][PL_TX + 2];
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
    const int tid = threadIdx.x, tx = tid % PL_TX, ty = tid / PL_TX;
    const int N0 = g.N[0], N1 = g.N[1];
    const c64 *aD0 = g.sdlinv[DUAL][0], *aP0 = g.sdlinv[PRIM][0], *aD1 = g.sdlinv[DUAL][1], *aP1 = g.sdlinv[PRIM][1];
    const c64 sdz = TM ? ldu(g.sdl[DUAL][2], 0) : ldu(g.sdl[PRIM][2], 0);
    for (int64_t tile = blockIdx.x; tile < (skip ? 0 : ntiles); tile += gridDim.x) {
        const int i0 = (int)(tile % ntx) * PL_TX, j0 = (int)(tile / ntx) * PL_TY;
        const int i = i0 + tx, j = j0 + ty;
        const bool own = i < N0 && j < N1;
        const int io = own ? i : 0, jo = j < N1 ? j : 0;
        const int im = io > 0 ? io - 1 : N0 - 1, jm = jo > 0 ? jo - 1 : N1 - 1;
        const int64_t p = io + (int64_t)N0 * jo;
        if (tile != (int64_t)blockIdx.x) __syncthreads();   // the last tile's reads of Xs are done
        // the owner's values, and this thread's point of the halo ring
        cx<R> xr[NC];
        c64 qc[NC], ec[NC], bv[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int64_t e = dofidx(g, C0 + c, p);
            xr[c] = x[e];
            qc[c] = MODE == MODE_P ? od.qs[3 * p + C0 + c] : cone<double>();
            ec[c] = MODE == MODE_A ? od.epsd[3 * p + C0 + c] : cone<double>();
            bv[c] = EPI == EPI_RESID || EPI == EPI_BDOT ? ball[rhs * vs + e] : czero<double>();
        }
        constexpr int NRING = 2 * (PL_TX + 2) + 2 * PL_TY;
        static_assert(NRING <= PL_TX * PL_TY, "");
        if (tid < NRING) {
            int ri, rj;
            if (tid < PL_TX + 2) { ri = tid; rj = 0; }
            else if (tid < 2 * (PL_TX + 2)) { ri = tid - (PL_TX + 2); rj = PL_TY + 1; }
            else { const int u = tid - 2 * (PL_TX + 2); ri = (u & 1) ? PL_TX + 1 : 0; rj = 1 + (u >> 1); }
            int gi = 0, gj = 0;
            c64 ph = cone<double>();
            const bool ok = wrap_ax(g, 0, i0 - 1 + ri, gi, ph) && wrap_ax(g, 1, j0 - 1 + rj, gj, ph);
            const int64_t pr = gi + (int64_t)N0 * gj;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                c64 v = czero<double>();
                if (ok) {
                    v = cvt<double>(x[dofidx(g, C0 + c, pr)]);
                    if (MODE == MODE_P) v = v * od.qs[3 * pr + C0 + c];
                    v = v * ph;
                }
                Xs[c][rj][ri] = v;
            }
        }
        const bool cpx = i + 1 < N0 || g.bloch[0], cpy = j + 1 < N1 || g.bloch[1];
        c64 e00 = czero<double>(), e10 = czero<double>(), e01 = czero<double>();
        if (OFFD && !TM) {
            const int ip = io + 1 < N0 ? io + 1 : 0, jp = jo + 1 < N1 ? jo + 1 : 0;
            e00 = od.epso[3 * p];
            if (cpx) e10 = od.epso[3 * (ip + (int64_t)N0 * jo)];
            if (cpy) e01 = od.epso[3 * (io + (int64_t)N0 * jp)];
        }
        // 1D factors: x per lane, y per wave (a wave is one row)
        const c64 ax = aD0[io], axm = aD0[im], exo = aP0[io], sx = g.sdl[TM ? PRIM : DUAL][0][io], sxo = g.sdl[TM ? DUAL : PRIM][0][io];
        const c64 ay = ldu(aD1, jo), aym = ldu(aD1, jm), eyo = ldu(aP1, jo), sy = ldu(g.sdl[PRIM][1], jo),
                  syo = ldu(g.sdl[DUAL][1], jo);
        c64 tmx = czero<double>(), tmy = czero<double>();
        if (MODE == MODE_P) {
            tmx = axis_term(g, 0, io);
            tmy = axis_term(g, 1, jo);
        }
        c64 xc[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            xc[c] = cvt<double>(xr[c]);
            // an unowned column or row next to the grid's end is the ghost of its
            // neighbour inside the tile
            c64 v = MODE == MODE_P ? xc[c] * qc[c] : xc[c];
            if (!own) {
                int gi = 0, gj = 0;
                c64 ph = cone<double>();
                v = czero<double>();
                if (wrap_ax(g, 0, i, gi, ph) && wrap_ax(g, 1, j, gj, ph)) {
                    const int64_t pg = gi + (int64_t)N0 * gj;
                    v = cvt<double>(x[dofidx(g, C0 + c, pg)]);
                    if (MODE == MODE_P) v = v * od.qs[3 * pg + C0 + c];
                    v = v * ph;
                }
            }
            Xs[c][ty + 1][tx + 1] = v;
        }
        __syncthreads();
        if (!own) continue;
        const int hi = tx + 1, hj = ty + 1;
        const bool xm = i > 0 || g.bloch[0], ym = j > 0 || g.bloch[1];   // H across the low ends
        c64 cc[NC], term[NC];
        if (TM) {
            const c64 z0 = Xs[0][hj][hi];
            const c64 hx = ay * (Xs[0][hj + 1][hi] - z0), hy = czero<double>() - ax * (Xs[0][hj][hi + 1] - z0);
            const c64 hxm = ym ? aym * (z0 - Xs[0][hj - 1][hi]) : czero<double>();
            const c64 hym = xm ? czero<double>() - axm * (z0 - Xs[0][hj][hi - 1]) : czero<double>();
            cc[0] = exo * (hy - hym) - eyo * (hx - hxm);
        } else {
            const c64 x0 = Xs[0][hj][hi], y0 = Xs[NC - 1][hj][hi];
            const c64 hz = ax * (Xs[NC - 1][hj][hi + 1] - y0) - ay * (Xs[0][hj + 1][hi] - x0);
            const c64 hzx = xm ? axm * (y0 - Xs[NC - 1][hj][hi - 1]) - ay * (Xs[0][hj + 1][hi - 1] - Xs[0][hj][hi - 1]) : czero<double>();
            const c64 hzy = ym ? ax * (Xs[NC - 1][hj - 1][hi + 1] - Xs[NC - 1][hj - 1][hi]) - aym * (x0 - Xs[0][hj - 1][hi]) : czero<double>();
            cc[0] = eyo * (hz - hzy);
            cc[NC - 1] = czero<double>() - exo * (hz - hzx);
            if (OFFD) {   // ε_xy: corner averages along y for Ex, along x for Ey
                const c64 h5 = mk<double>(0.5, 0);
                const c64 wx0 = (h5 * sx) * exo, wx1 = (h5 * g.sdl[DUAL][0][im]) * exo;
                const c64 wy0 = (h5 * syo) * eyo, wy1 = (h5 * ldu(g.sdl[DUAL][1], jm)) * eyo;
                term[0] = (h5 * e00) * (wy0 * y0 + wy1 * Xs[NC - 1][hj - 1][hi]);
                if (cpx) term[0] = term[0] + (h5 * e10) * (wy0 * Xs[NC - 1][hj][hi + 1] + wy1 * Xs[NC - 1][hj - 1][hi + 1]);
                term[NC - 1] = (h5 * e00) * (wx0 * x0 + wx1 * Xs[0][hj][hi - 1]);
                if (cpy) term[NC - 1] = term[NC - 1] + (h5 * e01) * (wx0 * Xs[0][hj + 1][hi] + wx1 * Xs[0][hj + 1][hi - 1]);
            }
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            c64 out;
            if (MODE == MODE_A) {
                out = cc[c] - om2 * (ec[c] * xc[c]);
                if (OFFD && !TM) out = out - om2 * term[c];
            } else {
                // w (cc − c qs x) + x, as in the marching stencil; T² is the
                // product of the stretched ∆l of the component's edge
                const c64 T2 = TM ? sx * sy : (c == 0 ? sx * sy : sxo * syo);
                const c64 w = qc[c] * (T2 * sdz);
                const c64 v = xc[c] * qc[c];
                const c64 cd = TM ? tmx + tmy : (c == 0 ? tmy : tmx);
                c64 in = cc[c] - cd * v;
                if (OFFD && !TM) in = in - om2 * term[c];
                out = w * in + xc[c];
            }
            const int64_t e = dofidx(g, C0 + c, p);
            if (EPI == EPI_RESID) {
                const c64 rr = mk<double>(bv[c].re - out.re, bv[c].im - out.im);
                if (yall) y[e] = cvt<R>(rr);   // null output: the residual norm only
                acc[0] += rr.re * rr.re + rr.im * rr.im;
            } else {
                y[e] = cvt<R>(out);
                epi_add<EPI>(acc, xc[c], out, bv[c]);
            }
        }
    }
    if (EPI == EPI_STORE) return;
    block_partial<NA>(acc, part + (size_t)rhs * NPART * 4, (int)blockIdx.x);
}
