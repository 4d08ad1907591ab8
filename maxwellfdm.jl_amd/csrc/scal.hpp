// The solvers' scalars of a right-hand side (plain C++: host_checks.cpp).
#pragma once
#include <cstddef>

#ifndef MFD_HD
#ifdef __HIPCC__
#define MFD_HD __host__ __device__
#else
#define MFD_HD
#endif
#endif

namespace mfd {

// Per-RHS solver scalars, kept on the device.
struct Scal {
    double rho_re, rho_im;     // rᵀr (bilinear)
    double sig_re, sig_im;     // qᵀ P q
    double alpha_re, alpha_im;
    double beta_re, beta_im;
    double tau, theta, cn, target;
    double c2t2, c2a_re, c2a_im;
    double rnorm2;             // scratch: last reduced norm²
    int conv, done, breakdown, stag;
    long long it, itmax, it_ref;
    double tau_ref;
    double apend_re, apend_im;   // COCG: α of the step whose iterate update is still pending
    double om_re, om_im;         // BiCGSTAB: ω
};

// All of a right-hand side's scalars but stag, which other blocks of a resident
// launch may mark (RESIDENT_TIMEOUT) at any time
MFD_HD inline void scal_store(Scal &to, const Scal &s) {
    constexpr size_t at = offsetof(Scal, stag), next = at + sizeof(s.stag);
    __builtin_memcpy((void *)&to, (const void *)&s, at);
    __builtin_memcpy((char *)&to + next, (const char *)&s + next, sizeof(Scal) - next);
}

}  // namespace mfd
