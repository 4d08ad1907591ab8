// Device pieces shared by the stencil and solver kernels: launch constants,
// stencil modes and epilogues, and the fixed-order reductions.
#pragma once
#include "op.hpp"

namespace mfd {

constexpr int NPART = 16384;  // max blocks per reduction (per RHS)
constexpr int NGRID_MAX = 2048;   // grid cap of the grid-stride vector kernels
constexpr int BS = 256;
enum { MODE_A = 0, MODE_P = 1 };
enum { EPI_STORE = 0, EPI_RESID = 1, EPI_DOT = 2, EPI_BDOT = 3, EPI_XDOT = 4 };
// one value's share of a stencil's reduction: x the operand, y the result, b the
// other vector of EPI_BDOT
template <int EPI>
__device__ inline void epi_add(double *acc, c64 x, c64 y, c64 b) {
    if (EPI == EPI_DOT) {          // xᵀy
        acc[0] += x.re * y.re - x.im * y.im;
        acc[1] += x.re * y.im + x.im * y.re;
    } else if (EPI == EPI_BDOT) {  // bᴴy
        acc[0] += b.re * y.re + b.im * y.im;
        acc[1] += b.re * y.im - b.im * y.re;
    } else if (EPI == EPI_XDOT) {  // yᴴx, ‖y‖²
        acc[0] += y.re * x.re + y.im * x.im;
        acc[1] += y.re * x.im - y.im * x.re;
        acc[2] += y.re * y.re + y.im * y.im;
    }
}

template <typename R>
__device__ inline cx<R> czero() { return mk<R>((R)0, (R)0); }
template <typename R>
__device__ inline cx<R> cone() { return mk<R>((R)1, (R)0); }

// block reduction of NV doubles; result valid in thread 0
template <int NV>
__device__ inline void block_sum(double (&v)[NV]) {
    __shared__ double sh[8][NV];
#pragma unroll
    for (int a = 0; a < NV; ++a)
        for (int o = 32; o > 0; o >>= 1) v[a] += __shfl_down(v[a], o, 64);
    int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0)
        for (int a = 0; a < NV; ++a) sh[wv][a] = v[a];
    __syncthreads();
    if (threadIdx.x == 0)
        for (int a = 0; a < NV; ++a) {
            double s = 0;
            for (int b = 0; b < (int)(blockDim.x >> 6); ++b) s += sh[b][a];
            v[a] = s;
        }
    __syncthreads();
}

// Grid reductions on the solver's hot path: every block writes its partial
// sums with plain stores and a one-block finish kernel, launched next on the
// same stream, adds them in a fixed order (deterministic) and updates the
// solver scalars.  The kernel boundary orders the two, so no block needs a
// device-scope fence or a shared counter.
template <int NV>
__device__ inline void block_partial(double (&v)[NV], double *part, int bid) {
    block_sum<NV>(v);
    if (threadIdx.x == 0)
        for (int a = 0; a < NV; ++a) part[4 * bid + a] = v[a];
}
// fixed-order sum of nb partials by one block; result in thread 0
template <int NV>
__device__ inline void sum_partials(const double *part, int nb, double (&tot)[NV]) {
    for (int a = 0; a < NV; ++a) tot[a] = 0;
    for (int b = threadIdx.x; b < nb; b += blockDim.x)
        for (int a = 0; a < NV; ++a) tot[a] += part[4 * b + a];
    block_sum<NV>(tot);
}

// ‖r‖, θ, c, τ, β, ρ of an SQMR step from ‖r‖² and rᵀr
__device__ inline void sqmr_advance(Scal &S, const double (&tot)[3]) {
    const double rn = sqrt(tot[0]);
    const double th1 = rn / S.tau, c = 1.0 / sqrt(1.0 + th1 * th1);
    S.c2t2 = c * c * S.theta * S.theta;
    S.c2a_re = c * c * S.alpha_re;
    S.c2a_im = c * c * S.alpha_im;
    S.tau = S.tau * th1 * c;
    const c64 rho1 = mk<double>(tot[1], tot[2]);
    if (S.rho_re == 0.0 && S.rho_im == 0.0) { S.beta_re = S.beta_im = 0; S.breakdown = 1; S.conv = 1; }
    else {
        const c64 b = cdiv(rho1, mk<double>(S.rho_re, S.rho_im));
        S.beta_re = b.re;
        S.beta_im = b.im;
    }
    S.rho_re = rho1.re;
    S.rho_im = rho1.im;
    S.theta = th1;
    S.rnorm2 = tot[0];
    S.it += 1;
    if (S.tau <= S.target || S.it >= S.itmax || rn == 0.0) S.conv = 1;
}

// BiCGSTAB: α = ρ / (r̂ᴴv)
__device__ inline void bi_alpha(Scal &S, const double (&tot)[2]) {
    if (tot[0] == 0.0 && tot[1] == 0.0) { S.breakdown = 1; S.conv = 1; S.alpha_re = S.alpha_im = 0; return; }
    const c64 a = cdiv(mk<double>(S.rho_re, S.rho_im), mk<double>(tot[0], tot[1]));
    S.alpha_re = a.re;
    S.alpha_im = a.im;
}

// BiCGSTAB: β = (ρ_new/ρ)(α/ω), ρ, τ = ‖r‖ and convergence from r̂ᴴr and ‖r‖²
__device__ inline void bi_advance(Scal &S, const double (&tot)[3]) {
    const c64 rho1 = mk<double>(tot[0], tot[1]), om = mk<double>(S.om_re, S.om_im);
    S.tau = sqrt(tot[2]);
    S.it += 1;
    if ((S.rho_re == 0.0 && S.rho_im == 0.0) || (om.re == 0.0 && om.im == 0.0)) {
        S.breakdown = 1;
        S.conv = 1;
        S.beta_re = S.beta_im = 0;
    } else {
        const c64 b = cdiv(rho1, mk<double>(S.rho_re, S.rho_im)) * cdiv(mk<double>(S.alpha_re, S.alpha_im), om);
        S.beta_re = b.re;
        S.beta_im = b.im;
    }
    S.rho_re = rho1.re;
    S.rho_im = rho1.im;
    if (S.tau <= S.target || S.it >= S.itmax || S.tau == 0.0) S.conv = 1;
}

// --------------------------------------------------------------- the operator

template <typename R>
__device__ inline void cell3(const DGrid<R> &g, int64_t p, int &i, int &j, int &k) {
    if (g.M <= INT32_MAX) {   // a 64-bit division is a few hundred cycles, and there are up to four
        const uint32_t q = (uint32_t)p, t = q / (uint32_t)g.N[0];
        i = (int)(q - t * (uint32_t)g.N[0]);
        k = (int)(t / (uint32_t)g.N[1]);
        j = (int)(t - (uint32_t)k * (uint32_t)g.N[1]);
        return;
    }
    i = (int)(p % g.N[0]);
    int64_t t = p / g.N[0];
    j = (int)(t % g.N[1]);
    k = (int)(t / g.N[1]);
}
template <typename R>
__device__ inline void dof2cp(const DGrid<R> &g, int64_t e, int &c, int64_t &p) {
    if (g.M <= INT32_MAX / 3) {
        const uint32_t u = (uint32_t)e;
        if (g.cmpfirst) {
            p = u / 3;
            c = (int)(u - 3 * (uint32_t)p);
        } else {
            const uint32_t k = u / (uint32_t)g.M;
            c = g.c0 + (int)k;
            p = u - k * (uint32_t)g.M;
        }
        return;
    }
    if (g.cmpfirst) { c = (int)(e % 3); p = e / 3; }
    else { const int k = (int)(e / g.M); c = g.c0 + k; p = e - (int64_t)k * g.M; }
}
// T (or T⁻¹) for E_c at (i,j,k): product over axes of sqrt(s∆l) at E_c's grid
// type (which each axis's boundft sets)
template <typename R>
__device__ inline cx<R> tfac(const DGrid<R> &g, int c, int i, int j, int k, bool inv) {
    if (g.tdof) {
        const int64_t p = i + (int64_t)g.N[0] * (j + (int64_t)g.N[1] * k);
        return inv ? g.tdofinv[3 * p + c] : g.tdof[3 * p + c];
    }
    const cx<R> *const(*t)[3] = inv ? g.ssqinv : g.ssq;
    cx<R> a = t[gtype(g.bft, EE, c, 0)][0][i];
    cx<R> b = t[gtype(g.bft, EE, c, 1)][1][j];
    cx<R> d = t[gtype(g.bft, EE, c, 2)][2][k];
    return (a * b) * d;
}

// scaled iterate value at E_c(i,j,k); indices may be -1 or N on one or more
// axes (ghosts): Bloch wraps with the phase, non-Bloch gives zero
template <typename R, int MODE>
__device__ inline cx<R> ldX(const DGrid<R> &g, const OpData<R> &od, const cx<R> *__restrict__ x, int c, int i,
                            int j, int k) {
    cx<R> ph = cone<R>();
    bool wr = false;
    int id[3] = {i, j, k};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        if (id[a] >= g.N[a]) {
            if (!g.bloch[a]) return czero<R>();
            id[a] -= g.N[a]; ph = ph * g.ph[a]; wr = true;
        } else if (id[a] < 0) {
            if (!g.bloch[a]) return czero<R>();
            id[a] += g.N[a]; ph = ph * g.phinv[a]; wr = true;
        }
    }
    int64_t p = id[0] + (int64_t)g.N[0] * (id[1] + (int64_t)g.N[1] * id[2]);
    cx<R> v = x[dofidx(g, c, p)];
    if (MODE == MODE_P)   // the stored q·T⁻¹ where the operator has it (FP64 data)
        v = v * (od.qs ? od.qs[3 * p + c] : od.q[3 * p + c] * tfac(g, c, id[0], id[1], id[2], true));
    return wr ? v * ph : v;
}

// H_u at (i,j,k) = ∂_v X_w − ∂_w X_v (v = u+1, w = u+2), times 1/μ_u.  Cₑ
// differences run forward along an axis whose boundft is EE and backward where
// it is HH; Cₘ the other way (so one index may be -1 or N: the outer curl's
// ghost, wrapped with the Bloch phase or zero).
template <typename R, int MODE, bool MU>
__device__ inline cx<R> Hval(const DGrid<R> &g, const OpData<R> &od, const cx<R> *__restrict__ x, int u, int i,
                             int j, int k) {
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
    int v = u == 0 ? 1 : (u == 1 ? 2 : 0), w = u == 0 ? 2 : (u == 1 ? 0 : 1);
    // ∂_a X_c at id without the ∆l factor, in Cₑ's direction along a
    auto dif = [&](int a, int c) -> cx<R> {
        int i1[3] = {id[0], id[1], id[2]};
        if (g.bft[a] == EE) {
            i1[a] += 1;
            return ldX<R, MODE>(g, od, x, c, i1[0], i1[1], i1[2]) - ldX<R, MODE>(g, od, x, c, id[0], id[1], id[2]);
        }
        i1[a] -= 1;
        return ldX<R, MODE>(g, od, x, c, id[0], id[1], id[2]) - ldX<R, MODE>(g, od, x, c, i1[0], i1[1], i1[2]);
    };
    cx<R> h = g.sdlinv[g0type(g.bft, HH, v)][v][id[v]] * dif(v, w) - g.sdlinv[g0type(g.bft, HH, w)][w][id[w]] * dif(w, v);
    if (MU) {
        int64_t p = id[0] + (int64_t)g.N[0] * (id[1] + (int64_t)g.N[1] * id[2]);
        h = h * od.muinv[3 * p + u];
    }
    return wr ? h * ph : h;
}

// curl-curl diagonal for E_u at (i,j,k): Σ over the two derivative axes (Cₘ
// backward along an EE axis, taking H at p and p−1; forward along an HH axis,
// taking H at p and p+1; a non-Bloch ghost H is zero)
template <typename R, bool MU>
__device__ inline cx<R> ccdiag(const DGrid<R> &g, const OpData<R> &od, int u, int i, int j, int k) {
    int id[3] = {i, j, k};
    int64_t p = i + (int64_t)g.N[0] * (j + (int64_t)g.N[1] * k);
    cx<R> s = czero<R>();
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        int a = t == 0 ? (u == 0 ? 1 : (u == 1 ? 2 : 0)) : (u == 0 ? 2 : (u == 1 ? 0 : 1));
        int hc = t == 0 ? (u == 0 ? 2 : (u == 1 ? 0 : 1)) : (u == 0 ? 1 : (u == 1 ? 2 : 0));  // H component
        int ia = id[a], Na = g.N[a];
        const bool fwd = g.bft[a] == HH;   // Cₘ direction along a
        const int gh = g0type(g.bft, HH, a);
        int io = fwd ? (ia < Na - 1 ? ia + 1 : 0) : (ia > 0 ? ia - 1 : Na - 1);   // the other H index
        cx<R> m0 = cone<R>(), m1 = cone<R>();
        int64_t sta = a == 0 ? 1 : (a == 1 ? (int64_t)g.N[0] : (int64_t)g.N[0] * g.N[1]);
        if (MU) {
            m0 = od.muinv[3 * p + hc];
            m1 = od.muinv[3 * (p + (int64_t)(io - ia) * sta) + hc];
        }
        cx<R> ie = g.sdlinv[g0type(g.bft, EE, a)][a][ia];
        cx<R> term;
        if (Na == 1 && g.bloch[a]) {
            cx<R> f = mk<R>((R)2, (R)0) - g.ph[a] - g.phinv[a];
            term = (ie * (g.sdlinv[gh][a][0] * m0)) * f;
        } else if (!g.bloch[a] && (fwd ? ia == Na - 1 : ia == 0)) {
            term = ie * (g.sdlinv[gh][a][ia] * m0);
        } else {
            term = ie * (g.sdlinv[gh][a][ia] * m0 + g.sdlinv[gh][a][io] * m1);
        }
        s = s + term;
    }
    return s;
}

static inline unsigned nb(int64_t n, int bs = BS) { return (unsigned)((n + bs - 1) / bs); }
static inline unsigned ngrid(int64_t n) {
    int64_t b = (n + BS - 1) / BS;
    return (unsigned)(b < NGRID_MAX ? (b < 1 ? 1 : b) : NGRID_MAX);
}

template <typename R> inline const OpData<R> &opd(const mfd_op *op);
template <> inline const OpData<double> &opd<double>(const mfd_op *op) { return op->d64; }
template <> inline const OpData<float> &opd<float>(const mfd_op *op) { return op->d32; }

}  // namespace mfd
