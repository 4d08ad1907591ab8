// Device pieces shared by the stencil and solver kernels: launch constants,
// stencil modes and epilogues, and the fixed-order reductions.
#pragma once
#include "op.hpp"

namespace mfd {

constexpr int NPART = 16384;  // max blocks per reduction (per RHS)
constexpr int NGRID_MAX = 2048;   // grid cap of the grid-stride vector kernels
constexpr int BS = 256;
enum { MODE_A = 0, MODE_P = 1 };
enum { EPI_STORE = 0, EPI_RESID = 1, EPI_DOT = 2 };

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

}  // namespace mfd
